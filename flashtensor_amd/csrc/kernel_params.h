// Launch-time parameter blocks shared by the host dispatcher and the kernels.
#pragma once
#include <stddef.h>
#include <stdint.h>

namespace ft {

struct Strides3 {
  int64_t b, s, h;
};

constexpr int kSplitMaxItems = 128, kSplitMaxBlocks = 64;  // of a (b, k/v head) pair

struct AttnKernelParams {
  const uint16_t* q;
  const uint16_t* k;
  const uint16_t* v;
  uint16_t* o;
  Strides3 sq, sk, sv, so;
  float* lse;     // [B,H,Sq] log2-domain normaliser of the plain softmax (may be null)
  float* lse_kf;  // [B,H,Sq] normaliser of the perturbed softmax (KeyFormer modes)
  const float* exp_rand;
  int64_t er_sb, er_sh, er_sr;
  uint64_t seed;
  int B, H, Sq, Skv;
  int off;          // Skv - Sq: query i sees keys j <= i + off when causal
  float logit_mul;  // reference rounding: f16(f16(acc) * logit_mul) == f16(f16(acc) / sqrt(D)); fast: log2e / sqrt(D)
  float inv_tau;
  // packed fp16 form of the same division for D = 128 (two packed ops on element pairs instead of one
  // mixed-precision multiply per element): t8 = fma(h, pk_hi, h * pk_lo) is 8 * f16(h / sqrt(D)) for every
  // fp16 h except where |h / sqrt(D)| < 7e-4, and there within 5e-7 of it; both halves hold the constant
  uint32_t pk_hi2, pk_lo2;
  float softcap;    // kKfSoftcap: logits become softcap * tanh(logit / softcap)
  int pair_order;   // block order of the causal attention kernel: heavy half descending, light half ascending
  int group;        // query heads per k/v head: query head h reads k/v head h / group
  int two_blocks;   // 256-row form: a workgroup takes query blocks nMB - 1 - slot and slot (set by the launcher)
  int head_major;   // workgroup order inside an XCD: all blocks of a (b, h) pair before the next pair's (launcher)
  // split form (attn_split.hpp): a row block's key tiles are shared out between workgroups, at most chunk_tiles each
  uint16_t* logits; // 16-bit logits of every row, kept for the column sums
  int logit_tiles;
  float* part;      // workspace of the shares' partial results (may be null where no block has more than one share)
  int chunk_tiles;
  int nitems;       // shares of all row blocks of a (b, k/v head) pair
  int part_waves;   // waves of a row block that have rows
  uint16_t items[kSplitMaxItems];       // row block << 8 | share; a block's shares are neighbours
  uint8_t first_item[kSplitMaxBlocks];  // where they begin
};

// How attention shares the key tiles of its row blocks out between workgroups; chunk_tiles 0: it does not.
struct SplitPlan {
  int chunk_tiles;   // tiles of a share, at most
  int items;         // shares of a (b, k/v head) pair
  int first_shared;  // row blocks from this one on have more than one share
  int nblocks, part_waves;
  int logit_tiles;   // logits are kept for the column sums: key tiles of a row, else 0
  bool one_per_cu;   // no more workgroups than CUs: keep them from sharing one
  size_t bytes;      // workspace of the shares' partial results and of the logits
  size_t logits_at;  // where in it the logits begin
  uint16_t list[kSplitMaxItems];
  uint8_t first_item[kSplitMaxBlocks];
};

// What the column sums of few rows are wanted for: sums [B, Hkv, Skv] (means over a group's heads), sums of squares (no
// groups) or null, and the odd width of SnapKV's window over the sums or 0.
struct SplitStats {
  float *colsum, *colsumsq;
  int pool;
};
constexpr int kSplitMaxPool = 65, kSplitStatRows = 64;

struct ColstatsKernelParams {
  const uint16_t* q;
  const uint16_t* k;
  Strides3 sq, sk;
  const float* lse;  // [B,H,Sq] normaliser of the distribution being summed
  float* colsum;     // [B,H,Skv]
  float* colsumsq;   // [B,H,Skv] or null
  uint8_t* keep;     // [B,H,Skv] CoRM modes: 1 where some row's probability reaches its threshold
  const float* exp_rand;  // KeyFormer noise [B,H,Sq,Skv]; CoRM tensor mode: thresholds [Sq,Skv] (er_sb = er_sh = 0)
  int64_t er_sb, er_sh, er_sr;
  uint64_t seed;
  int B, H, Sq, Skv;
  int off;
  float logit_mul;
  uint32_t pk_hi2, pk_lo2;  // as in AttnKernelParams
  float inv_tau;
  int group;  // query heads per k head
  int pool;        // kStatSumPool: half the odd width of SnapKV's window over the sums, whose means go to colsum
  int pair_order;  // key-block order for launches of two workgroups per CU: heavy half descending, light half ascending (launcher)
};

// what happens to a logit between the scaled QK^T and the softmax of the attention pass
// kKfSeededTau1 / kKfSeededFast: the seeded KeyFormer stream inside the packed fp16 path.  The perturbed
// weight exp((t + g) / tau) with g = -ln E equals exp(t / tau) E^(-1/tau); the in-kernel E lies in
// [6e-8, 16.7], so for tau >= 0.25 the plain softmax's running maximum also stabilises the perturbed sum
// (exponent <= (6 + 24) / tau <= 120) and no second maximum is tracked; tau == 1 needs 1 / E only.
// kKfTensor / kKfTensorLds: noise from a tensor, its tiles landing in LDS by direct-to-LDS loads a whole tile ahead, 4 or 16 bytes a
// lane (16: rows of whole aligned chunks, a (b, h) slice below 2 GiB)
enum KfMode { kKfNone = 0, kKfTensor = 1, kKfSeeded = 2, kKfSoftcap = 3, kKfSeededTau1 = 4, kKfSeededFast = 5, kKfTensorLds = 6 };
// kStatCormRule: thresholds 1 / (i + 1) per query row i; kStatCormTensor: thresholds read from a tensor
enum StatMode {
  kStatSum = 0, kStatSumSq = 1, kStatKfTensor = 2, kStatKfSeeded = 3, kStatCormRule = 4, kStatCormTensor = 5,
  kStatKfSeededTau1 = 6, kStatKfSeededFast = 7, // seeded KeyFormer inside the packed fp16 path (see KfMode)
  kStatSumPool = 8                              // kStatSum and SnapKV's window over the sums
};

}  // namespace ft
