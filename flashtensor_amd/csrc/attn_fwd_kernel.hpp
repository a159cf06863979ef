// Fused softmax attention forward for gfx950 (pass A of every softmax workload): the kernel template and its
// launch-shape selection.  Instantiated per element type and head size by attn_fwd_{f16,bf16}_{d64,d128}.hip (one
// translation unit each, so that they compile in parallel); attn_fwd.hip holds the dispatcher.
//
// Replaces the attention core the reference emits as a Triton kernel for cases/kernels/attn.py:18-34
// (and the identical prefix of h2o.py, kf.py, roco.py): O = softmax(QK^T / sqrt(D) + causal mask) V,
// never writing an S x S tensor.  Also emits the per-row log2-domain normaliser (max + log2 sum) that the
// column-statistics pass consumes, and in the KeyFormer modes the normaliser of the Gumbel-perturbed
// softmax of kf.py:36-39 instead.
//
// Mapping.  One workgroup = 32 WAVES query rows of one (b, h), one wave per 32 rows (4 waves and two
// workgroups per CU, or 8 waves and one: the same two waves per SIMD, but a staged K/V tile then serves
// twice as many rows); keys are streamed in tiles
// of 64 through double-buffered LDS (direct global->LDS loads).  Each wave computes the TRANSPOSED score
// block S^T = K Q^T with v_mfma_f32_32x32x16: a lane then owns one query (column l % 32) and 16 of the
// 32 keys of each block, so the online-softmax row max / row sum are in-lane reductions plus a single
// exchange with lane l ^ 32, and the accumulator registers are already the B operand (keys on the
// contraction axis) of O^T += V^T P^T.  V^T is fed by ds_read_b64_tr_b16 from the row-major V tile.
#pragma once
#include "device_common.hpp"
#include "kernel_params.h"
#include "noise.h"

#include <type_traits>

namespace ft {

constexpr int kAttnBN = 64;
constexpr bool kAttnTwoBlocks = true;

// Rescale threshold of the running maximum in log2 units: the stale maximum is kept (and O, l are not
// rescaled) while the new row maximum exceeds it by less than this, so unnormalised probabilities stay
// below 2^kRescaleSlack (exact in fp16/fp32; the final division uses the same maximum).
constexpr float kRescaleSlack = 6.f;
// Where the running maximum begins: the lowest finite value.  Visible logits may be -inf (a QK^T below the range of the
// tensor type); a tile that shows a row nothing else leaves the maximum here, and its exponentials are exp2(-inf - kNoMax) = 0,
// where a maximum of -inf would make them NaN.  A row that ends here has seen no finite logit: its sum is 0.
constexpr float kNoMax = -__FLT_MAX__;

// One share's partial result of a row block in the workspace (SPLIT): per wave of 32 rows the accumulator registers of
// its 64 lanes, row maxima and row sums.
struct SplitPartial {
  float *o, *m, *l;
};
__host__ __device__ constexpr int64_t split_wave_floats(int D) { return 32 * D + 64; }
__device__ __forceinline__ SplitPartial split_partial(float* base, int D, int64_t slot) {
  float* o = base + slot * split_wave_floats(D);
  return SplitPartial{o, o + 32 * D, o + 32 * D + 32};
}

// SPLIT: the form for few query rows over many keys (see attn_split.hpp).  A workgroup's rows are the (query, head)
// pairs of one k/v head, row r = query r / group of the group's head r % group, so that K and V are staged once for the
// whole group, and it walks only its share of the row block's key tiles; where a block has several shares, each leaves
// its accumulator, row maxima and row sums in the workspace and attn_combine_kernel folds them.  Built for the causal
// instantiation only: without a mask `off` is set to Skv, which hides nothing.
// STORE: the 16-bit logits of the rows go to the workspace as well, for the column sums (attn_split.hip).
// TEAMS = 2 (SPLIT): the two shares of a block of 64 rows are taken by two pairs of waves of one workgroup, each with LDS
// buffers of its own, and fold in LDS: each wave has its SIMD to itself, as in a launch of fewer 128-row blocks than CUs, which
// is bound by the chain of its longest block (0.9 us a tile at D128, whatever the other CUs do), and the chain is half as
// long.  B1 H8 S2048 D128 36 -> 29 us, soft-capped 58 -> 39; D64 25 -> 20 (when it is taken: attn_fwd.hip).  The KeyFormer modes
// have it too (B1 H16 S697, whole call, noise from a tensor 63 -> 50 us, from a seed 40 -> 33): their running sums of the perturbed
// softmax fold beside the plain ones.
template <typename T, int D, bool CAUSAL, bool EMU, int KF, int WAVES, bool SPLIT = false, bool STORE = false, int TEAMS = 1>
__global__ void __launch_bounds__(64 * WAVES * TEAMS, ((KF == kKfTensor || KF == kKfTensorLds) && D == 128 ? 1 : 8 / (WAVES * TEAMS))) attn_fwd_kernel(const AttnKernelParams p) {
  constexpr int BM = 32 * WAVES, BN = kAttnBN, NT = 64 * WAVES;
  constexpr int KSTEPS = D / 16;
  constexpr int DB = D / 32;
  typedef TileGeom<D> G;
  typedef typename T::vec8 vec8;
  constexpr int TILE_BYTES = BN * G::RB;
  constexpr bool kIsF16 = __is_same(typename T::elem, _Float16);
  constexpr bool kKfFast = KF == kKfSeededTau1 || KF == kKfSeededFast;           // seeded noise inside the packed path
  constexpr bool kSeeded = KF == kKfSeeded || kKfFast;
  // variants served by the pipelined fast path: the plain softmax in either type with either treatment of the
  // logits, and the packed seeded KeyFormer modes (fp16)
  constexpr bool kFastMasked = (kIsF16 && EMU && kKfFast) || KF == kKfNone || KF == kKfSoftcap;
  constexpr bool kCap = KF == kKfSoftcap;
  constexpr bool kTensor = KF == kKfTensor || KF == kKfTensorLds;  // noise tensor staged through LDS
  static_assert(!kKfFast || (kIsF16 && EMU), "the packed KeyFormer modes exist for fp16 with reference rounding only");
  // Software pipeline across tiles: the QK^T MFMAs of tile it+1 are issued in the same iteration as the
  // softmax (VALU) and PV MFMAs of tile it, so the matrix and vector pipes overlap inside one wave.
  // K therefore runs one tile ahead of V in LDS.
  // One LDS object per buffer: the compiler tracks outstanding direct-to-LDS loads per object, so reads
  // of one buffer do not wait for the loads in flight into the others.
  __shared__ __align__(16) char s_k0[TEAMS * TILE_BYTES];
  __shared__ __align__(16) char s_k1[TEAMS * TILE_BYTES];
  __shared__ __align__(16) char s_v0[TEAMS * TILE_BYTES];
  __shared__ __align__(16) char s_v1[TEAMS * TILE_BYTES];
  const int team = TEAMS > 1 ? wave_id() / WAVES : 0;
  char* const ldsK0 = s_k0 + team * TILE_BYTES;
  char* const ldsK1 = s_k1 + team * TILE_BYTES;
  char* const ldsV0 = s_v0 + team * TILE_BYTES;
  char* const ldsV1 = s_v1 + team * TILE_BYTES;
  __shared__ __align__(16) uint32_t s_col[TEAMS * 2 * BN];
  uint32_t* const ldsCol = s_col + team * 2 * BN;  // noise column terms of the current / next tile
  const int tid = TEAMS > 1 ? threadIdx.x % NT : threadIdx.x;
  // Noise from a tensor: every wave's slice of the next tile (32 rows x 64 keys fp32).  It is the wave's own, but a lane reads
  // its row's slots, which other lanes filled: the wave waits for all of its loads before it reads one.
  constexpr int kErWaveBytes = 32 * BN * 4;
  __shared__ __align__(16) char ldsEr[kTensor ? TEAMS * WAVES * kErWaveBytes : 16];

  static_assert(TEAMS == 1 || (SPLIT && !STORE && WAVES == 2 && TEAMS == 2), "the teams' instantiations");
  static_assert(!SPLIT || (CAUSAL && WAVES * TEAMS == 4 && (TEAMS > 1 || KF == kKfNone || KF == kKfSoftcap)), "the split form's instantiations");
  static_assert(!STORE || (SPLIT && EMU && KF == kKfNone), "logits are kept where they are 16-bit values");
  const int rows = SPLIT ? p.Sq * p.group : p.Sq;  // rows of a (b, h) pair; SPLIT: of a (b, k/v head) pair
  const int BH = SPLIT ? p.B * (p.H / p.group) : p.B * p.H;
  const int nMB = (rows + BM - 1) / BM;
  // (b, h) pair and rank among that pair's workgroups.  Workgroups are dealt round-robin to the 8 XCDs and, inside
  // an XCD, start in index order.  head_major: the workgroups of an XCD walk through that XCD's pairs one after
  // the other (all ranks of a pair are neighbours in the XCD's order), so that the workgroups resident on an XCD
  // at one time share the K/V of a few pairs in its L2; otherwise rank-major (every pair's rank 0 first).
  int bh = blockIdx.x % BH, rank = blockIdx.x / BH;
  if (p.head_major) {
    const int li = blockIdx.x >> 3, nrank = gridDim.x / BH;
    bh = (blockIdx.x & 7) + 8 * (li / nrank);
    rank = li % nrank;
  }
  // Heaviest (last) query blocks of every head first: longest-processing-time order keeps the causal
  // triangle balanced over the CUs.  Workgroups are dealt round-robin to the 8 XCDs, so with B*H a
  // multiple of 8 a head stays on one XCD and its K/V are shared through that XCD's L2.  (Walking an XCD
  // through its heads one at a time cuts the K/V re-reads from 1.6x to 1.1x of the operand size but
  // loses the balance: measured 15% slower.)
  int mb = nMB - 1 - rank;
  if (p.pair_order) {
    // Every workgroup is resident from the start (no more of them than slots), so nothing is left to hand out
    // as CUs free up: the heavy half is dealt first, descending, then the light half ascending, which tends to
    // put a heavy and a light block on the same CU (measured 50 -> 47 us at B1 H32 S2048; with more
    // workgroups than slots the descending order wins: 144 vs 164 us at S4096).
    const int half = (nMB + 1) / 2;
    mb = rank < half ? nMB - 1 - rank : rank - half;
  }
  int chunk = 0;
  if (TEAMS > 1) {
    chunk = team;
  } else if (SPLIT) {
    mb = p.items[rank] >> 8;
    chunk = p.items[rank] & 255;
  }
  const int b = SPLIT ? bh / (p.H / p.group) : bh / p.H;
  const int h = SPLIT ? (bh % (p.H / p.group)) * p.group : bh % p.H;  // SPLIT: the group's first head
  const int lane = lane_id(), wave = TEAMS > 1 ? wave_id() % WAVES : wave_id();
  const int g = lane >> 5, n = lane & 31;
  // two_blocks (causal, set by the launcher when the pairs fill the chip evenly): the workgroup takes query
  // block nMB - 1 - slot and then block slot, the heaviest with the lightest, so that every workgroup walks the
  // same number of key tiles and no workgroup is launched into a half-empty chip at the end
  // (compiled in only where the second pass costs no registers: with it the 4-wave form and the packed KeyFormer
  // modes spill, and a spilled register's reload waits for the tile loads in flight: both count in vmcnt)
  constexpr bool kTwoPass = WAVES == 8 && (KF == kKfNone || KF == kKfSoftcap);
  const int npass = (kTwoPass && p.two_blocks && 2 * rank != nMB - 1) ? 2 : 1;
  for (int pass = 0; pass < npass; ++pass) {
  if (kTwoPass && p.two_blocks) mb = pass == 0 ? nMB - 1 - rank : rank;
  if (pass) __syncthreads();  // every wave has left the first block's K/V tiles
  const int m0 = mb * BM;
  const int qrow = m0 + wave * 32 + n;
  const int qrow_c = qrow < rows ? qrow : rows - 1;
  const int qi = SPLIT ? qrow_c / p.group : qrow;      // query position of the row
  const int qi_c = SPLIT ? qi : qrow_c;
  const int hq = SPLIT ? h + qrow_c % p.group : h;     // its head
  const float NEG_INF = -__builtin_inff();

  const uint16_t* qptr = p.q + b * p.sq.b + (int64_t)qi_c * p.sq.s + hq * p.sq.h;
  vec8 qf[KSTEPS];
#pragma unroll
  for (int t = 0; t < KSTEPS; ++t) qf[t] = *reinterpret_cast<const vec8*>(qptr + 16 * t + 8 * g);

  const uint16_t* kbase = p.k + b * p.sk.b + (h / p.group) * p.sk.h;
  const uint16_t* vbase = p.v + b * p.sv.b + (h / p.group) * p.sv.h;

  // tiles of the workgroup, of this wave (not entirely above its diagonal), and of this wave's mask-free prefix
  const int wave_row0 = m0 + wave * 32;
  // STORE: logits [pair][row][key].  A lane has keys 16 b + 4 g + [0..3] and + 8 of its row; the halves of the wave swap
  // four keys each, so that a lane stores eight neighbours
  uint16_t* logit_row = STORE ? p.logits + ((int64_t)bh * rows + qrow_c) * (p.logit_tiles * BN) + 8 * g : nullptr;
  auto store_logits = [&](int b16, uint32_t a0, uint32_t a1, uint32_t b0, uint32_t b1) __attribute__((always_inline)) {
#if defined(__HIP_DEVICE_COMPILE__)
    const auto s0 = __builtin_amdgcn_permlane32_swap(a0, b0, false, false), s1 = __builtin_amdgcn_permlane32_swap(a1, b1, false, false);
    if (qrow < rows) *reinterpret_cast<uint4v*>(logit_row + 16 * b16) = uint4v{s0[0], s1[0], s0[1], s1[1]};
#endif
  };
  int Skv = p.Skv, off = p.off;  // SPLIT: counted from the first key of the workgroup's share,
  int tile0 = 0;                 // which is that of this tile of the row
  int n_end = Skv;
  if (CAUSAL) n_end = min(Skv, (SPLIT ? (min(m0 + BM, rows) - 1) / p.group + 1 : m0 + BM) + off);
  int ntiles = (n_end + BN - 1) / BN;
  int nch = 1;  // shares of this row block
  int ntrips = 0;  // TEAMS: barriers that every wave takes part in, whatever its own share
  if (SPLIT) {
    nch = TEAMS > 1 ? TEAMS : (ntiles + p.chunk_tiles - 1) / p.chunk_tiles;
    const int per = (ntiles + nch - 1) / nch, t0 = chunk * per, t1 = min(t0 + per, ntiles);
    ntrips = per;
    tile0 = t0;
    kbase += (int64_t)t0 * BN * p.sk.s;
    vbase += (int64_t)t0 * BN * p.sv.s;
    off -= t0 * BN;
    if (STORE) logit_row += t0 * BN;
    Skv = min(Skv, t1 * BN) - t0 * BN;
    ntiles = t1 - t0;  // >= 1: (nch - 1) per <= (nch - 1) chunk_tiles < tiles of the block (TEAMS: the second team may have none)
  }
  int nw = ntiles, n_fast = Skv / BN;
  if (CAUSAL && !SPLIT) {
    nw = min(ntiles, (wave_row0 + 31 + off) / BN + 1);
    n_fast = min(n_fast, (wave_row0 + off + 1) / BN);  // tiles with n0 + BN - 1 <= wave_row0 + off
  }
  if (SPLIT) {
    // the wave's first and last query position; a wave without rows, or whose rows see no key of the share, has no tiles
    const int pos0 = min(wave_row0, rows - 1) / p.group, pos1 = min(wave_row0 + 31, rows - 1) / p.group;
    nw = wave_row0 < rows ? min(ntiles, (max(pos1 + off, -BN) + BN) / BN) : 0;
    n_fast = min(n_fast, max(pos0 + off + 1, 0) / BN);
  }
  n_fast = min(n_fast, nw);
  const int n_free = n_fast;             // leading tiles of which this wave sees every key
  if (!kFastMasked) n_fast = 0;          // the pipelined loop (and its mask-free instance) is not used

  NoiseKeys nk = {0, 0};
  uint32_t a_i = 0;
  if (kSeeded) {
    nk = noise_keys(p.seed, (uint32_t)bh);
    a_i = noise_row(nk, (uint32_t)qi);
  }
  // Noise from a tensor: the wave's slice of a tile is 32 rows x 256 bytes.  kKfTensorLds: load r8 of a tile brings rows
  // 4 r8 + [0..3] whole (a load instruction then touches 8 cache lines; with a lane fetching its own row's chunks
  // it touched 32, and the address path, not HBM, bounded the pass): lane l fills slot l % 16 of row 4 r8 + l / 16
  // with global chunk (l % 16) ^ (row % 16), the XOR placement that lets 32 rows be read back one chunk column at
  // a time without bank conflicts.  Chunks past the end of a row re-read its last chunk (those keys are masked),
  // rows past Sq the last row.
  // kKfTensor, for rows that do not begin at multiples of 16 bytes or do not hold whole chunks (and slices of 2 GiB and
  // more): one row and 4 bytes a lane per load, into the same slots.  Four times the loads, but 16-byte ones at odd addresses
  // take the address path as long as four and do not coalesce (B1 H32 S3543 D128, whole call, noise read into registers
  // 618 us, by 16 bytes 615, by 4 bytes 480; rows of 3544 450).  Keys past the end of a row re-read its last one.
  // (kKfTensor: from the wave's first row on, so that one descriptor reaches its rows unless they are 64 MiB apart;
  // with a descriptor each S67 D64 takes 16.7 us for 14.3)
  constexpr int64_t kNearRow = kRsrcBytes / (32 * 4);  // the longest such row: of the 32nd every key is in reach
  const int er_row0 = KF == kKfTensor ? min(wave_row0, p.Sq - 1) : 0, er_rows = p.Sq - er_row0;
  const float* er_slice = kTensor ? p.exp_rand + b * p.er_sb + h * p.er_sh + er_row0 * p.er_sr : nullptr;
  rsrc_t er_rsrc = make_rsrc(er_slice);
  char* er_lds = ldsEr + (kTensor ? (team * WAVES + wave) * kErWaveBytes : 0);
  // per-lane state of those loads: two registers (the offsets of the eight loads are rebuilt from them for every
  // tile: kept in registers across the loop they would cost eight, and this path has none to spare)
  const int er_cs = (lane & 15) ^ (lane >> 4);  // slot ^ (row % 4); the row's bits 2..3 are those of r8
  const uint32_t er_row_bytes = (uint32_t)p.er_sr * 4u;
  const uint32_t er_off0 = kTensor ? (uint32_t)(m0 + wave * 32 + (lane >> 4)) * er_row_bytes : 0u;
  const uint32_t er_off_last = kTensor ? (uint32_t)(p.Sq - 1) * er_row_bytes : 0u;
  auto issue_er = [&](int t) __attribute__((always_inline)) {
    if constexpr (KF == kKfTensorLds) {
      const int last_chunk = p.Skv / 4 - 1;
      int cs = er_cs;
      uint32_t off0 = er_off0;
      asm volatile("" : "+v"(cs), "+v"(off0));  // not loop-invariant as far as the compiler can tell
#pragma unroll
      for (int r8 = 0; r8 < 8; ++r8) {
        const int c = min((tile0 + t) * (BN / 4) + (cs ^ (4 * (r8 & 3))), last_chunk);
        const uint32_t row_off = min(off0 + (uint32_t)(4 * r8) * er_row_bytes, er_off_last);
        load_lds16(er_rsrc, er_lds + r8 * 1024, row_off + (uint32_t)c * 16u, 0);
      }
    } else {
      const uint32_t last = (uint32_t)(p.Skv - 1) * 4u, tile_byte = (uint32_t)(tile0 + t) * (BN * 4u);
      uint32_t d0 = (uint32_t)lane * 4u;
      asm volatile("" : "+v"(d0));
      // (row offsets are wave-uniform)
      if (p.er_sr <= kNearRow) {
#pragma unroll
        for (int r = 0; r < 32; ++r)
          load_lds4(er_rsrc, er_lds + r * 256, min((d0 ^ (uint32_t)((r & 15) << 4)) + tile_byte, last), (uint32_t)min(r, er_rows - 1) * er_row_bytes);
      } else {
#pragma unroll 1
        for (int r = 0; r < 32; ++r) {
          const rsrc_t row = make_rsrc(er_slice + (int64_t)min(r, er_rows - 1) * p.er_sr);
          load_lds4(row, er_lds + r * 256, min((d0 ^ (uint32_t)((r & 15) << 4)) + tile_byte, last), 0);
        }
      }
    }
  };
  // the lane's query row n, chunks 2 k8 + g (keys 8 k8 + 4 g + [0..3] of the tile: score registers 4 (k8 % 4) + [0..3]
  // of half k8 / 4)
  // (slot (2 k8 + g) ^ (n % 16) of row n: byte offset ((g ^ n % 16) << 4) ^ (k8 << 5) inside the row, so one
  // register and one xor with a constant per read)
  const uint32_t er_rd0 = (uint32_t)(n * 256) | (uint32_t)((g ^ (n & 15)) << 4);
  auto read_er = [&](float (&dst)[2][16]) __attribute__((always_inline)) {
    uint32_t rd0 = er_rd0;
    asm volatile("" : "+v"(rd0));
#pragma unroll
    for (int k8 = 0; k8 < 8; ++k8) {
      const float4v e4 = *reinterpret_cast<const float4v*>(er_lds + (rd0 ^ (uint32_t)(k8 << 5)));
#pragma unroll
      for (int e = 0; e < 4; ++e) dst[k8 >> 2][4 * (k8 & 3) + e] = e4[e];
    }
  };

  TileStager<D, BN, NT, kRowSwizzle> stK;
  TileStager<D, BN, NT, kTrSwizzle> stV;
  stK.init(kbase, p.sk.s);
  stV.init(vbase, p.sv.s);
  auto stage_k = [&](int t, char* dst) __attribute__((always_inline)) {
    if (t < ntiles) stK.issue(t * BN, min(BN, Skv - t * BN), dst);
  };
  auto stage_v = [&](int t, char* dst) __attribute__((always_inline)) {
    if (t < ntiles) stV.issue(t * BN, min(BN, Skv - t * BN), dst);
    if (kSeeded && t < ntiles && tid < BN) ldsCol[(t & 1) * BN + tid] = noise_col(nk, (uint32_t)((tile0 + t) * BN + tid));
  };

  float16v o_acc[DB];
#pragma unroll
  for (int i = 0; i < DB; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) o_acc[i][r] = 0.f;
  float m_run = kNoMax, l_run = 0.f;  // running max (log2 domain) and this lane's share of the row sum
  float m_kf = kNoMax, l_kf = 0.f;
  float16v S0[2], S1[2];  // score accumulators of the current / next tile (they swap every tile)

  // Per-lane LDS byte offsets of the MFMA operand reads inside a tile (the XOR swizzles make them
  // lane-dependent, so they are computed once instead of per read).
  uint32_t koff[KSTEPS];  // K row n (and n + 32 via an immediate), chunk 2t + g
#pragma unroll
  for (int t = 0; t < KSTEPS; ++t) koff[t] = n * G::RB + (((2 * t + g) ^ G::row_swz(n)) << 4);
  uint32_t voff[DB];  // V^T operand: rows 4g + (l%16)/4 (+ 16 ks, + 8 via immediates), columns 32 db + ...
  {
    const int j16 = lane & 15, dhalf = (lane >> 4) & 1;
    const int r0 = 4 * g + (j16 >> 2);
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      const int d0 = 32 * db + 16 * dhalf + 4 * (j16 & 3);
      voff[db] = r0 * G::RB + (((d0 >> 3) ^ G::tr_swz(r0)) << 4) + (d0 & 7) * 2;
    }
  }

  // ---- S^T = K Q^T : [64 keys] x [32 queries] as two 32x32 blocks (16 LDS reads, 16 MFMAs), optionally
  // in two halves over the head dimension so that other work can sit between them
  auto qk_part = [&](float16v (&s)[2], const char* tk, auto t0_tag, auto t1_tag) __attribute__((always_inline)) {
    constexpr int T0 = decltype(t0_tag)::value, T1 = decltype(t1_tag)::value;
    if (T0 == 0) {
#pragma unroll
      for (int mbk = 0; mbk < 2; ++mbk)
#pragma unroll
        for (int r = 0; r < 16; ++r) s[mbk][r] = 0.f;
    }
    vec8 ka[KSTEPS][2];
#pragma unroll
    for (int t = T0; t < T1; ++t)
#pragma unroll
      for (int mbk = 0; mbk < 2; ++mbk) ka[t][mbk] = *reinterpret_cast<const vec8*>(tk + koff[t] + mbk * 32 * G::RB);
#pragma unroll
    for (int t = T0; t < T1; ++t)
#pragma unroll
      for (int mbk = 0; mbk < 2; ++mbk) s[mbk] = T::mfma(ka[t][mbk], qf[t], s[mbk]);
  };
  auto qk = [&](float16v (&s)[2], const char* tk) __attribute__((always_inline)) {
    qk_part(s, tk, std::integral_constant<int, 0>{}, std::integral_constant<int, KSTEPS>{});
  };
  // LDS latency is far longer than an MFMA, so operand reads must run several MFMAs ahead of their
  // consumers; sched_group_barrier sequences pin that order (the scheduler would otherwise sink each
  // read next to its use to save registers).  Masks: 0x008 MFMA, 0x100 LDS read, 0x002 VALU.
  auto sched_qk_alone = [&]() __attribute__((always_inline)) {
    __builtin_amdgcn_sched_group_barrier(0x100, 6, 0);
#pragma unroll
    for (int t = 0; t < KSTEPS - 3; ++t) {
      __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, 6, 0);
  };

  auto rescale = [&](float rowmax) __attribute__((always_inline)) {
    const bool grow = rowmax > m_run + kRescaleSlack;  // identical in both lanes of a row
    if (__any(grow)) {
      const float m_new = grow ? rowmax : m_run;
      const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
      if (KF == kKfSeededTau1) l_kf *= alpha;
      if (KF == kKfSeededFast) l_kf *= __builtin_amdgcn_exp2f((m_run - m_new) * p.inv_tau);
      m_run = m_new;
      l_run *= alpha;
#pragma unroll
      for (int i = 0; i < DB; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) o_acc[i][r] *= alpha;
    }
  };

  // ---- softmax of the pipelined path, in two parts so that the rescale branch sits between them.
  // Rounding is monotonic, so the row maximum of the rounded logits is the rounded maximum of the raw
  // accumulators.
  // MASKED (tiles that straddle the diagonal or the end of K): hidden keys are left out of the maximum, so
  // that a row whose largest visible logit defines the stabiliser gets exp2(0) = 1 for it exactly (row 0
  // of a causal problem then has the normaliser of the reference, bit for bit).
  const float rcp_cap = kCap ? 1.f / p.softcap : 0.f;
  // row maximum of one tile's logits in the log2 domain (what rescale() compares with the running maximum)
  auto tile_max = [&](auto masked_tag, const float16v (&s)[2], int n0) __attribute__((always_inline)) -> float {
    constexpr bool MASKED = decltype(masked_tag)::value;
    const int lim = (CAUSAL ? min(qi + off, Skv - 1) : Skv - 1) - n0 - 4 * g;
    auto at = [&](int mbk, int r) __attribute__((always_inline)) -> float {
      if (!MASKED) return s[mbk][r];
      const int jl = 32 * mbk + 8 * (r >> 2) + (r & 3);
      return jl > lim ? NEG_INF : s[mbk][r];
    };
    // four independent chains, then a short tree: the reduction is latency-, not throughput-bound.  Three-operand
    // maxima throughout (v_max3_f32; this translation unit is built without NaN honouring, so none of them is
    // preceded by quieting moves of the MFMA results).
    float m4[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int mbk = c >> 1, r0 = (c & 1) * 8;
      m4[c] = max3(at(mbk, r0), at(mbk, r0 + 1), at(mbk, r0 + 2));
      m4[c] = max3(m4[c], at(mbk, r0 + 3), at(mbk, r0 + 4));
      m4[c] = max3(m4[c], at(mbk, r0 + 5), at(mbk, r0 + 6));
    }
    const float t0 = max3(m4[0], at(0, 7), at(0, 15)), t1 = max3(m4[1], at(1, 7), at(1, 15));
    float amax = max3(max3(t0, t1, m4[2]), m4[3], m4[3]);
    const float other = xchg32(amax);
    amax = max3(amax, other, other);
    // soft-cap: the cap is monotonic as well (a product with a positive constant, tanh, roundings), so the
    // maximum of the capped logits is the capped maximum (fp16: to a unit in its last place, since the compiler rounds a product here
    // straight to a half; a stabiliser has no need to be the logit itself, and products rounded on their own, dependent on each other,
    // took two teams of D = 128 0.5 to 0.9 % longer)
    auto r16 = [](float x) { return T::to_float(T::from_float(x)); };
    if (EMU) {
      float t = r16(r16(amax) * p.logit_mul);
      if (kCap) t = r16(r16(tanh_exp_form(r16(t * rcp_cap))) * p.softcap);
      return t * kLog2e;
    } else if (kCap) {
      return p.softcap * tanh_exp_form(amax * (p.logit_mul * (1.f / kLog2e)) * rcp_cap) * kLog2e;
    }
    return amax * p.logit_mul;  // logit_mul = log2e / sqrt(D) when the logits stay in fp32
  };
  // MASKED: key j of the tile is hidden from this lane's query when j > qi + off or j >= Skv.
  auto fast_exp = [&](auto masked_tag, const float16v (&s)[2], vec8 (&pb)[4], int n0, int it) __attribute__((always_inline)) {
    constexpr bool MASKED = decltype(masked_tag)::value;
    const float neg_m = -m_run;
    const half2v pk_hi = __builtin_bit_cast(half2v, p.pk_hi2), pk_lo = __builtin_bit_cast(half2v, p.pk_lo2);
    // local key index of register r is 32 mbk + 8 (r / 4) + 4 g + r % 4; it is visible iff <= lim + 4 g
    const int lim = (CAUSAL ? min(qi + off, Skv - 1) : Skv - 1) - n0 - 4 * g;
    uint4v pw[4];
    // Eight elements (one MFMA operand) at a time, stage by stage, so that consecutive instructions are
    // independent: every stage's result is needed only four instructions later.
#pragma unroll
    for (int blk = 0; blk < 4; ++blk) {
      const int mbk = blk >> 1, rb = (blk & 1) * 8;
      float x[8];
      if constexpr (EMU && kIsF16) {
        half2v t2[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float2v a2 = {s[mbk][rb + 2 * i], s[mbk][rb + 2 * i + 1]};
          const half2v h2 = __builtin_convertvector(a2, half2v);  // QK^T is an fp16 tensor in the reference
          // ... divided by sqrt(D) in fp16: t2 = 8 * f16(h / sqrt(D)), exact for D = 64, two packed ops for D = 128
          t2[i] = D == 64 ? h2 : __builtin_elementwise_fma(h2, pk_hi, h2 * pk_lo);
        }
        if (STORE)
          store_logits(it * 4 + blk, __builtin_bit_cast(uint32_t, t2[0]), __builtin_bit_cast(uint32_t, t2[1]),
                       __builtin_bit_cast(uint32_t, t2[2]), __builtin_bit_cast(uint32_t, t2[3]));
        if constexpr (kCap) {
          // Gemma2's soft-cap (below), bound by the vector pipe: a product reads its half by itself (the sum with 0 makes it
          // v_fma_mix_f32), in place of a conversion and a product, and two products are rounded by one conversion.  A product is an
          // fp32 number first, as in the reference: rounded straight to a half (v_fma_mix{lo,hi}_f16) some logits are another half
          // where the cap has many bits (44.8: one in 50, 33.3: one in 500), and it is slower, since the two halves of a word wait for each
          // other.  450 vector instructions a mask-free tile; in turn with conversions of their own (546) and with the straight
          // rounding (418): B8 H32/8 S1885 D128 425 us, 460 and 436, B5 H16 S904 D64 34.2, 40.4 and 35.2, H32/8 Sq777 Skv3000 D128
          // 80.0, 84.3 and 81.4.
          auto mul = [](uint32_t w, float f) __attribute__((always_inline)) {
            const half2v h = __builtin_bit_cast(half2v, w);
            return float2v{__builtin_fmaf((float)h[0], f, 0.f), __builtin_fmaf((float)h[1], f, 0.f)};
          };
          auto round2 = [](float2v f) __attribute__((always_inline)) {
            uint32_t w = T::pack2(f[0], f[1]);
            asm("" : "+v"(w));  // one conversion of two, which the compiler would split (and join with the products) otherwise
            return w;
          };
          half2v c2[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            float2v z = mul(round2(mul(__builtin_bit_cast(uint32_t, t2[i]), rcp_cap * 0.125f)), 2.f * kLog2e);
#pragma unroll
            for (int e = 0; e < 2; ++e) z[e] = 1.f - __builtin_amdgcn_rcpf(__builtin_fmaf(__builtin_amdgcn_exp2f(z[e]), 0.5f, 0.5f));  // tanh_exp_form
            c2[i] = __builtin_bit_cast(half2v, round2(mul(round2(z), p.softcap)));
          }
#pragma unroll
          for (int i = 0; i < 8; ++i) x[i] = __builtin_fmaf((float)c2[i >> 1][i & 1], kLog2e, neg_m);
        } else {
#pragma unroll
          for (int i = 0; i < 8; ++i) x[i] = __builtin_fmaf((float)t2[i >> 1][i & 1], kLog2e / 8.f, neg_m);
        }
      } else if constexpr (EMU) {
        // bf16: round QK^T, multiply by the tuned constant (== dividing by sqrt(D) in bf16), round again; the
        // conversions handle two elements each, unpacking a half is a shift or a mask
        uint32_t tw[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const uint32_t h2 = T::pack2(s[mbk][rb + 2 * i], s[mbk][rb + 2 * i + 1]);
          const uint32_t t2 = T::pack2(T::lo(h2) * p.logit_mul, T::hi(h2) * p.logit_mul);
          tw[i] = t2;
          x[2 * i] = kCap ? T::lo(t2) * rcp_cap : __builtin_fmaf(T::lo(t2), kLog2e, neg_m);
          x[2 * i + 1] = kCap ? T::hi(t2) * rcp_cap : __builtin_fmaf(T::hi(t2), kLog2e, neg_m);
        }
        if (STORE) store_logits(it * 4 + blk, tw[0], tw[1], tw[2], tw[3]);
      } else {
#pragma unroll
        for (int i = 0; i < 8; ++i)
          x[i] = kCap ? s[mbk][rb + i] * (p.logit_mul * (1.f / kLog2e) * rcp_cap) : __builtin_fmaf(s[mbk][rb + i], p.logit_mul, neg_m);
      }
      if constexpr (kCap && !(EMU && kIsF16)) {
        // Gemma2's soft-cap, cap * tanh(logit / cap): three 16-bit tensor ops in the reference
        // (cases/kernels/gemma2.py:31-33), each rounded when the reference's rounding is reproduced
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float y0 = x[2 * i], y1 = x[2 * i + 1];
          if (EMU) {
            const uint32_t w = T::pack2(y0, y1);
            y0 = T::lo(w), y1 = T::hi(w);
          }
          float z0 = tanh_exp_form(y0), z1 = tanh_exp_form(y1);
          if (EMU) {
            const uint32_t w = T::pack2(z0, z1);
            const uint32_t c = T::pack2(T::lo(w) * p.softcap, T::hi(w) * p.softcap);
            x[2 * i] = __builtin_fmaf(T::lo(c), kLog2e, neg_m);
            x[2 * i + 1] = __builtin_fmaf(T::hi(c), kLog2e, neg_m);
          } else {
            x[2 * i] = __builtin_fmaf(z0 * p.softcap, kLog2e, neg_m);
            x[2 * i + 1] = __builtin_fmaf(z1 * p.softcap, kLog2e, neg_m);
          }
        }
      }
      if (MASKED) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int jl = 32 * mbk + 8 * ((rb + i) >> 2) + ((rb + i) & 3);
          x[i] = (jl > lim) ? NEG_INF : x[i];
        }
      }
      // KeyFormer, seeded: E = -ln u of the 8 (query, key) pairs; the column terms of keys
      // 32 mbk + 8 (rb / 4 [+ 1]) + 4 g + [0..3] are two aligned groups of four in LDS
      float ee[8];
      if constexpr (kKfFast) {
        const uint32_t* col = ldsCol + (it & 1) * BN + 32 * mbk + 2 * rb + 4 * g;
        const uint4v c0 = *reinterpret_cast<const uint4v*>(col), c1 = *reinterpret_cast<const uint4v*>(col + 8);
#pragma unroll
        for (int i = 0; i < 8; ++i)  // log2 u = -E / ln 2 (negative): the constant factor is applied once, at the end
          ee[i] = __builtin_amdgcn_logf(noise_uniform(a_i, i < 4 ? c0[i] : c1[i - 4]));
        if constexpr (KF == kKfSeededFast) {
          const float shift = -kLog2Ln2 * p.inv_tau;
#pragma unroll
          for (int i = 0; i < 8; ++i)  // exp2(((t - m) log2e - log2 E) / tau); hidden keys carry x = -inf
            l_kf += __builtin_amdgcn_exp2f(__builtin_fmaf(x[i] - __builtin_amdgcn_logf(-ee[i]), p.inv_tau, shift));
        }
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = __builtin_amdgcn_exp2f(x[i]);
      if constexpr (KF == kKfSeededTau1) {
#pragma unroll
        for (int i = 0; i < 8; ++i) l_kf = __builtin_fmaf(x[i], __builtin_amdgcn_rcpf(ee[i]), l_kf);  // -ln2 exp(t - m) / E
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        pw[blk][i] = T::pack2(x[2 * i], x[2 * i + 1]);  // whole 32-bit words: no 16-bit shuffles
        l_run = T::add2(pw[blk][i], l_run);             // row sum of the 16-bit P the MFMA consumes
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) pb[i] = __builtin_bit_cast(vec8, pw[i]);
  };

  // ---- generic path (tensor-noise KeyFormer, and the seeded modes outside the packed form): softmax of one
  // 32-key half of a tile, s (raw accumulators of one 32x32 block) -> pb (two MFMA operands of 16-bit
  // unnormalised probabilities).  Half a tile at a time keeps the live set small enough for the noise slice
  // of the next tile to be in flight beside the accumulators.
  // MASKED: some key of the half is hidden from some query of the wave (the diagonal, the end of K).
  auto softmax_half = [&](auto masked_tag, const float16v& s, vec8 (&pb)[2], int n0h, int buf, int mbk, const float (&er)[16]) __attribute__((always_inline)) {
    constexpr bool MASKED = decltype(masked_tag)::value;
    // ---- logits with the reference's rounding points when EMU (the same chains as the pipelined path: two elements per
    // conversion), and their row maximum in the log2 domain.  fp16 logits stay packed, times 8: the log2 domain's factor rides in the
    // v_fma_mix_f32 that subtract the noise and the maximum, and the maximum is taken two elements at a time: 11 registers and a
    // tenth of the vector instructions less (noise tensor, tau 1.5, whole call: H32 S4096 D128 516 -> 507 us, S3000 329 -> 324; D64 as before).
    constexpr bool kHalves = EMU && kIsF16;
    float x[kHalves ? 1 : 16];
    half2v x2[kHalves ? 8 : 1];
    // local key index of register r is 8 (r / 4) + 4 g + r % 4; it is visible iff <= lim + 4 g
    const int lim = (CAUSAL ? min(qi + off, Skv - 1) : Skv - 1) - n0h - 4 * g;
    float rowmax;
    if constexpr (kHalves) {
      const half2v pk_hi = __builtin_bit_cast(half2v, p.pk_hi2), pk_lo = __builtin_bit_cast(half2v, p.pk_lo2);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float2v a2 = {s[2 * i], s[2 * i + 1]};
        const half2v h2 = __builtin_convertvector(a2, half2v);  // QK^T is an fp16 tensor in the reference
        // ... divided by sqrt(D) in fp16: 8 * f16(h / sqrt(D)), exact for D = 64, two packed ops for D = 128
        x2[i] = D == 64 ? h2 : __builtin_elementwise_fma(h2, pk_hi, h2 * pk_lo);
        if (MASKED) {
#pragma unroll
          for (int e = 0; e < 2; ++e) x2[i][e] = (8 * (i >> 1) + 2 * (i & 1) + e > lim) ? (_Float16)NEG_INF : x2[i][e];
        }
      }
      half2v m2 = x2[0];
#pragma unroll
      for (int i = 1; i < 8; ++i) m2 = __builtin_elementwise_max(m2, x2[i]);
      rowmax = fmaxf((float)m2[0], (float)m2[1]);
      rowmax = fmaxf(rowmax, xchg32(rowmax)) * (kLog2e / 8.f);
    } else {
      if constexpr (EMU) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const uint32_t h2 = T::pack2(s[2 * i], s[2 * i + 1]);
          const uint32_t t2 = T::pack2(T::lo(h2) * p.logit_mul, T::hi(h2) * p.logit_mul);
          x[2 * i] = T::lo(t2) * kLog2e;
          x[2 * i + 1] = T::hi(t2) * kLog2e;
        }
      } else {
#pragma unroll
        for (int r = 0; r < 16; ++r) x[r] = s[r] * p.logit_mul;
      }
      if (MASKED) {
#pragma unroll
        for (int r = 0; r < 16; ++r) x[r] = (8 * (r >> 2) + (r & 3) > lim) ? NEG_INF : x[r];
      }
      rowmax = max3(x[0], x[1], x[2]);
#pragma unroll
      for (int r = 3; r < 15; r += 2) rowmax = max3(rowmax, x[r], x[r + 1]);
      rowmax = fmaxf(rowmax, x[15]);
      rowmax = fmaxf(rowmax, xchg32(rowmax));
    }
    auto less = [&](int r, float by) __attribute__((always_inline)) -> float {  // the logit in the log2 domain less `by`
      return kHalves ? __builtin_fmaf((float)x2[kHalves ? r >> 1 : 0][r & 1], kLog2e / 8.f, -by) : x[kHalves ? 0 : r] - by;
    };

    // ---- KeyFormer: running normaliser of softmax((logit + gumbel) / tau), gumbel = -ln(E)
    {
      float z[16];
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        float log2E;
        if (kTensor) {
          log2E = __builtin_amdgcn_logf(er[r]);
        } else {
          const int jl = 32 * mbk + 8 * (r >> 2) + 4 * g + (r & 3);
          const float u = noise_uniform(a_i, ldsCol[buf * BN + jl]);
          log2E = __builtin_amdgcn_logf(-kLn2 * __builtin_amdgcn_logf(u));
        }
        z[r] = less(r, log2E);  // times tau
      }
      float zmax = max3(z[0], z[1], z[2]);
#pragma unroll
      for (int r = 3; r < 15; r += 2) zmax = max3(zmax, z[r], z[r + 1]);
      zmax = fmaxf(zmax, z[15]);
      zmax = fmaxf(zmax, xchg32(zmax));
      // (finite: a half that is hidden entirely, zmax = -inf, adds exp2(-inf) = 0)
      const float mk_new = fmaxf(m_kf, zmax * p.inv_tau);
      float zs = 0.f;
#pragma unroll
      for (int r = 0; r < 16; ++r) zs += __builtin_amdgcn_exp2f(__builtin_fmaf(z[r], p.inv_tau, -mk_new));
      l_kf = l_kf * __builtin_amdgcn_exp2f(m_kf - mk_new) + zs;
      m_kf = mk_new;
    }

    rescale(rowmax);
    uint4v pw[2];
#pragma unroll
    for (int r = 0; r < 16; r += 2) {
      const uint32_t w = T::pack2(__builtin_amdgcn_exp2f(less(r, m_run)), __builtin_amdgcn_exp2f(less(r + 1, m_run)));
      l_run = T::add2(w, l_run);  // row sum of the 16-bit P the MFMA consumes
      pw[r >> 3][(r & 7) >> 1] = w;
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) pb[i] = __builtin_bit_cast(vec8, pw[i]);
  };

  // ---- O^T += V^T P^T (32 transposed LDS reads, 16 MFMAs)
  auto read_vt = [&](const char* tv, int ks, int db) __attribute__((always_inline)) -> vec8 {
    const char* p0 = tv + voff[db] + ks * 16 * G::RB;
    short4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(FT_LDS(short4v, p0));
    short4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(FT_LDS(short4v, p0 + 8 * G::RB));
    short8v both = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    return __builtin_bit_cast(vec8, both);
  };
  auto pv = [&](const vec8 (&pb)[4], const char* tv) __attribute__((always_inline)) {
    vec8 va[4][DB];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int db = 0; db < DB; ++db) va[ks][db] = read_vt(tv, ks, db);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int db = 0; db < DB; ++db) o_acc[db] = T::mfma(va[ks][db], pb[ks], o_acc[db]);
  };
  auto sched_pv_alone = [&]() __attribute__((always_inline)) {
    __builtin_amdgcn_sched_group_barrier(0x100, 8, 1);
#pragma unroll
    for (int i = 0; i < 4 * DB - 4; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 1);
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 1);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, 4, 1);
  };

  // One tile of the pipelined loop.  Three things overlap inside a wave: the QK^T MFMAs of the NEXT tile, the
  // softmax VALU chain of this tile (whose stabiliser was settled before the tile began) and this tile's PV
  // MFMAs; the row maximum of the next tile is taken at the end, under the PV MFMAs, so that its long dependent
  // chain (32 values -> 1, one lane exchange, the 16-bit roundings) never stands alone.  The only branch, the
  // rare rescale of the running maximum, sits at the very start of the tile.
  //   pend_max: log2-domain row maximum of the tile about to be processed (from the previous tile, or the prologue)
  float pend_max = NEG_INF;
  auto fast_tile = [&](auto masked_tag, auto next_masked_tag, auto stage_tag, float16v (&s_cur)[2], float16v (&s_next)[2],
                       const char* tk_next, const char* tv, int n0, int it, char* k_dst, char* v_dst) __attribute__((always_inline)) {
    constexpr bool STAGE = decltype(stage_tag)::value;
    constexpr int kValuGroup = kKfFast ? 12 : kCap ? 11 : 6;  // vector instructions placed after each MFMA
    vec8 pb[4];
    rescale(pend_max);
    // STAGE: the direct-to-LDS loads of K[it+2] and V[it+1] (both full tiles) are issued from inside this
    // block, one every few MFMAs.  Issued back to back they fill the texture-address queue (one 1 KB load
    // per 16 cycles per CU) and the wave stalls at issue for about a sixth of the tile time.
    if (STAGE) {  // after the rescale branch, so that the loads share a basic block with the MFMAs
      stK.issue_full((it + 2) * BN, k_dst);
      stV.issue_full((it + 1) * BN, v_dst);
    }
    qk(s_next, tk_next);
    if (kKfFast && STAGE && tid < BN)  // column terms of tile it + 1 (the other half of ldsCol)
      ldsCol[((it + 1) & 1) * BN + tid] = noise_col(nk, (uint32_t)((tile0 + it + 1) * BN + tid));
    fast_exp(masked_tag, s_cur, pb, n0, it);
    pv(pb, tv);
    pend_max = tile_max(next_masked_tag, s_next, n0 + BN);
    constexpr int kStageEvery = TEAMS > 1 ? 2 : 4;  // (the loads of a tile fall to fewer waves)
    __builtin_amdgcn_sched_group_barrier(0x100, 6, 2);
#pragma unroll
    for (int i = 0; i < 2 * KSTEPS; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 2);
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 2);
      if (STAGE && i % kStageEvery == 1) __builtin_amdgcn_sched_group_barrier(0x020, 1, 2);
      __builtin_amdgcn_sched_group_barrier(0x002, kValuGroup, 2);
    }
#pragma unroll
    for (int i = 0; i < 4 * DB; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 2);
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 2);
      if (STAGE && i % kStageEvery == 1) __builtin_amdgcn_sched_group_barrier(0x020, 1, 2);
      __builtin_amdgcn_sched_group_barrier(0x002, kValuGroup, 2);
    }
  };

  // One iteration = one barrier.  On entry K[it+1] and V[it] have been requested; K[it+2] and V[it+1] are
  // requested here, into the buffers every wave has finished reading.
  auto sync_and_stage = [&](int it, char* k_dst, char* v_dst) __attribute__((always_inline)) {
    wait_vmem();
    __syncthreads();
    stage_k(it + 2, k_dst);
    stage_v(it + 1, v_dst);
  };

  if constexpr (kFastMasked) {
  // ---- prologue: K[0], V[0], K[1] in flight; scores of tile 0
  stage_k(0, ldsK0);
  stage_v(0, ldsV0);
  stage_k(1, ldsK1);
  wait_vmem();
  __syncthreads();
  qk(S0, ldsK0);
  sched_qk_alone();

  int it = 0;
  // ---- mask-free tiles, two per trip so that the two score buffers swap roles without copies
  // pairs (it, it+1) of mask-free tiles whose staged tiles K[it+2], K[it+3], V[it+1], V[it+2] are whole tiles
  const int nf2 = max(0, min(n_fast, Skv / BN - 2)) & ~1;
  // tiles from nf2 on go through the masked instance (which is exact for a tile that needs no mask as well); so
  // does tile 0, which may be one of them.
  pend_max = tile_max(std::true_type{}, S0, 0);
  for (; it < nf2 - 2; it += 2) {
    wait_vmem();
    __syncthreads();
    fast_tile(std::false_type{}, std::false_type{}, std::true_type{}, S0, S1, ldsK1, ldsV0, 0, it, ldsK0, ldsV1);      // stages K[it+2], V[it+1]
    wait_vmem();
    __syncthreads();
    fast_tile(std::false_type{}, std::false_type{}, std::true_type{}, S1, S0, ldsK0, ldsV1, 0, it + 1, ldsK1, ldsV0);  // stages K[it+3], V[it+2]
  }
  if (it < nf2) {  // the last mask-free pair: the tile after it takes its maximum over visible keys
    wait_vmem();
    __syncthreads();
    fast_tile(std::false_type{}, std::false_type{}, std::true_type{}, S0, S1, ldsK1, ldsV0, 0, it, ldsK0, ldsV1);
    wait_vmem();
    __syncthreads();
    fast_tile(std::false_type{}, std::true_type{}, std::true_type{}, S1, S0, ldsK0, ldsV1, (it + 1) * BN, it + 1, ldsK1, ldsV0);
    it += 2;
  }
  // ---- tiles that straddle the diagonal or the end of K
  // Two per trip where the registers allow it (`it` is even here), so that the LDS buffers are named at compile
  // time: with a buffer chosen at run time the compiler cannot tell the tile being read from the tile being
  // loaded, and the first operand read of the tile waits for the K / V tiles requested a few instructions earlier.
  constexpr bool kTailPairs = KF == kKfNone || KF == kKfSoftcap;
  if constexpr (kTailPairs) {
    auto tail_tile = [&](int it, auto odd_tag) __attribute__((always_inline)) {
      constexpr bool odd = decltype(odd_tag)::value;
      // Behind all of the pair's first tile: nothing in the fp16 soft cap's chain keeps the compiler from raising this barrier to that
      // tile's last operand read, and waves with both tiles then stand in the middle of the first one until those whose last tile it is
      // have done theirs (H8 fp16, D64 S65 to S128 7.4 to 7.8 -> 6.7 to 7.1 us, D128 S128 9.2 -> 8.7, S200 10.9 -> 10.3; mask-free pairs,
      // which all waves walk together, are no faster for it).
      if constexpr (odd && kCap && EMU && kIsF16) __builtin_amdgcn_sched_barrier(0);
      sync_and_stage(it, odd ? ldsK1 : ldsK0, odd ? ldsV0 : ldsV1);
      fast_tile(std::true_type{}, std::true_type{}, std::false_type{}, S0, S1, odd ? ldsK0 : ldsK1, odd ? ldsV1 : ldsV0, it * BN, it, nullptr, nullptr);
#pragma unroll
      for (int mbk = 0; mbk < 2; ++mbk) S0[mbk] = S1[mbk];
    };
    for (; it + 1 < nw; it += 2) {
      tail_tile(it, std::false_type{});
      tail_tile(it + 1, std::true_type{});
    }
    if (it < nw) {
      tail_tile(it, std::false_type{});
      ++it;
    }
  }
  for (; it < nw; ++it) {
    const bool odd = it & 1;
    sync_and_stage(it, odd ? ldsK1 : ldsK0, odd ? ldsV0 : ldsV1);
    fast_tile(std::true_type{}, std::true_type{}, std::false_type{}, S0, S1, odd ? ldsK0 : ldsK1, odd ? ldsV1 : ldsV0, it * BN, it, nullptr, nullptr);
#pragma unroll
    for (int mbk = 0; mbk < 2; ++mbk) S0[mbk] = S1[mbk];
  }
  // ---- tiles entirely above this wave's diagonal: keep the workgroup's barriers and staging in step
  for (; it < (TEAMS > 1 ? ntrips : ntiles); ++it) sync_and_stage(it, (it & 1) ? ldsK1 : ldsK0, (it & 1) ? ldsV0 : ldsV1);
  } else {
  // ---- generic path: not pipelined across tiles.  K and V of tile it are read while those of tile it + 1 are
  // loaded; a tile is worked on as two halves of 32 keys (8 + 8 MFMAs each), every key masked by comparison.
  // Two tiles per trip, so that every LDS buffer is named at compile time: with a buffer chosen at run time
  // the compiler cannot tell the tile being read from the tile being loaded, and drains every load in flight
  // before the first LDS read of the tile.
  // Noise from a tensor: er[mbk] is this lane's slice of the noise tile (its query row, the 16 keys of its score registers
  // in half mbk), read from LDS at the top of the tile.  The S x S tensor is the one operand that comes from HBM every time.
  float er[2][16];
  auto qk_half = [&](float16v& s, const char* tk, int mbk) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = 0.f;
#pragma unroll
    for (int t = 0; t < KSTEPS; ++t)
      s = T::mfma(*reinterpret_cast<const vec8*>(tk + koff[t] + mbk * 32 * G::RB), qf[t], s);
  };
  auto pv_half = [&](const vec8 (&pb)[2], const char* tv, int mbk) __attribute__((always_inline)) {
#pragma unroll
    for (int ksl = 0; ksl < 2; ++ksl)
#pragma unroll
      for (int db = 0; db < DB; ++db) o_acc[db] = T::mfma(read_vt(tv, 2 * mbk + ksl, db), pb[ksl], o_acc[db]);
  };
  auto slow_tile = [&](int it, auto odd_tag) __attribute__((always_inline)) {
    constexpr bool odd = decltype(odd_tag)::value;
    wait_vmem();
    __syncthreads();
    if (kTensor && it < nw) {
      // this tile's slice from LDS to registers; the next tile's is requested into the same slots further down.  The
      // reads must have returned before those loads may overwrite their slots (nothing in the hardware orders an LDS
      // read against a later direct-to-LDS load).
      read_er(er);
      __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    }
    stage_k(it + 1, odd ? ldsK0 : ldsK1);
    stage_v(it + 1, odd ? ldsV0 : ldsV1);
    if (it < nw) {  // not entirely above this wave's diagonal
#pragma unroll
      for (int mbk = 0; mbk < 2; ++mbk) {
        float16v s;
        vec8 pb[2];
        qk_half(s, odd ? ldsK1 : ldsK0, mbk);
        if (it < n_free)
          softmax_half(std::false_type{}, s, pb, it * BN + 32 * mbk, odd ? 1 : 0, mbk, er[mbk]);
        else
          softmax_half(std::true_type{}, s, pb, it * BN + 32 * mbk, odd ? 1 : 0, mbk, er[mbk]);
        // The next tile's noise, in flight for the rest of the tile without holding a register.  Requested here, behind
        // the first half's contraction and softmax, rather than at the top of the tile in front of the K / V staging
        // loads: the eight loads no longer queue up with the staging at the moment every wave leaves the barrier
        // (B1 H32 S4096, same process: 538 -> 512 us per call; before the softmax 523, after the first half's PV 516,
        // four loads behind each half's softmax 524).
        if (kTensor && mbk == 0 && it + 1 < nw) issue_er(it + 1);
        pv_half(pb, odd ? ldsV1 : ldsV0, mbk);
      }
    }
  };
  if (kTensor && nw > 0) issue_er(0);
  stage_k(0, ldsK0);
  stage_v(0, ldsV0);
  int it = 0;
  const int trips = TEAMS > 1 ? ntrips : ntiles;
  for (; it + 1 < trips; it += 2) {
    slow_tile(it, std::false_type{});
    slow_tile(it + 1, std::true_type{});
  }
  if (it < trips) slow_tile(it, std::false_type{});
  }

  // ---- epilogue
  l_run += xchg32(l_run);
  if (kTensor || kSeeded) l_kf += xchg32(l_kf);
  if constexpr (TEAMS > 1) {
    // the second team's accumulators, row maxima and row sums through LDS (the tiles' buffers) to the first team
    float4v* fold_o = reinterpret_cast<float4v*>(s_k0) + wave * (DB * 4 * 64) + lane;
    float* fold_ml = reinterpret_cast<float*>(s_v0) + wave * 256 + lane;
    static_assert(WAVES * DB * 4 * 64 * 16 <= TEAMS * TILE_BYTES && WAVES * 256 * 4 <= TEAMS * TILE_BYTES, "room of the fold");
    wait_vmem();
    __syncthreads();
    if (team == 1) {
#pragma unroll
      for (int i = 0; i < DB * 4; ++i)
        fold_o[i * 64] = float4v{o_acc[i >> 2][4 * (i & 3)], o_acc[i >> 2][4 * (i & 3) + 1], o_acc[i >> 2][4 * (i & 3) + 2], o_acc[i >> 2][4 * (i & 3) + 3]};
      fold_ml[0] = m_run;
      fold_ml[64] = l_run;
      if (kTensor || kSeeded) {
        fold_ml[128] = m_kf;
        fold_ml[192] = l_kf;
      }
    }
    __syncthreads();
    if (team == 1) return;
    const float m1 = fold_ml[0], l1 = fold_ml[64];
    const float m_new = fmaxf(m_run, m1);
    const float w0 = __builtin_amdgcn_exp2f(m_run - m_new), w1 = __builtin_amdgcn_exp2f(m1 - m_new);
    if (kTensor || kSeeded) {
      const float lk1 = fold_ml[192];
      if constexpr (KF == kKfSeededTau1) {
        l_kf = __builtin_fmaf(lk1, w1, l_kf * w0);
      } else if constexpr (KF == kKfSeededFast) {
        l_kf = __builtin_fmaf(lk1, __builtin_amdgcn_exp2f((m1 - m_new) * p.inv_tau), l_kf * __builtin_amdgcn_exp2f((m_run - m_new) * p.inv_tau));
      } else {
        const float mk1 = fold_ml[128], mk = fmaxf(m_kf, mk1);
        l_kf = __builtin_fmaf(lk1, __builtin_amdgcn_exp2f(mk1 - mk), l_kf * __builtin_amdgcn_exp2f(m_kf - mk));
        m_kf = mk;
      }
    }
    m_run = m_new;
    l_run = __builtin_fmaf(l1, w1, l_run * w0);
#pragma unroll
    for (int i = 0; i < DB * 4; ++i) {
      const float4v o1 = fold_o[i * 64];
#pragma unroll
      for (int e = 0; e < 4; ++e) o_acc[i >> 2][4 * (i & 3) + e] = __builtin_fmaf(o1[e], w1, o_acc[i >> 2][4 * (i & 3) + e] * w0);
    }
  }
  if (SPLIT && TEAMS == 1 && nch > 1) {
    // unnormalised: accumulator registers as they are, one 16-byte piece per lane and store (coalesced), rows that exist
    const SplitPartial part = split_partial(p.part, D, ((int64_t)bh * p.nitems + rank) * p.part_waves + wave);
    if (qrow < rows) {
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4) {
          const float4v w = {o_acc[db][4 * q4], o_acc[db][4 * q4 + 1], o_acc[db][4 * q4 + 2], o_acc[db][4 * q4 + 3]};
          *reinterpret_cast<float4v*>(part.o + ((db * 4 + q4) * 64 + lane) * 4) = w;
        }
      if (g == 0) {
        part.m[n] = m_run;
        part.l[n] = l_run;
      }
    }
    return;
  }
  const float inv_l = 1.f / l_run;
  if (qrow < rows) {
    uint16_t* optr = p.o + b * p.so.b + (int64_t)qi * p.so.s + hq * p.so.h;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {
        const int d = 32 * db + 8 * q4 + 4 * g;
        uint16_t w[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) w[e] = T::from_float(o_acc[db][4 * q4 + e] * inv_l);
        uint2 pk;
        pk.x = (uint32_t)w[0] | ((uint32_t)w[1] << 16);
        pk.y = (uint32_t)w[2] | ((uint32_t)w[3] << 16);
        *reinterpret_cast<uint2*>(optr + d) = pk;
      }
    if (g == 0 && p.lse) p.lse[(SPLIT ? (int64_t)b * p.H + hq : (int64_t)bh) * p.Sq + qi] = m_run + __builtin_amdgcn_logf(l_run);
  }
  if (kTensor || kSeeded) {
    if (KF == kKfSeededTau1) l_kf *= -kLog2e;  // the sum was taken over 1 / log2 u = -ln2 / E
    // packed modes: the perturbed sum shares the plain softmax's stabiliser, scaled by 1 / tau
    const float base = KF == kKfSeededTau1 ? m_run : KF == kKfSeededFast ? m_run * p.inv_tau : m_kf;
    if (qrow < rows && g == 0) p.lse_kf[(int64_t)bh * p.Sq + qi] = base + __builtin_amdgcn_logf(l_kf);
  }
  }  // pass
}

// ---------------------------------------------------------------------------------------------------
// launch-shape selection (host)

int device_cu_count();     // attn_fwd.hip
int attn_split_override();  // attn_fwd.hip: 0, or -1: never split, n > 0: split into shares of n tiles
int attn_form_override();  // attn_fwd.hip: 0 or the AttnForm to take
int plain_form(int64_t BH, int group, int Sq, int Skv, int D, bool causal, bool cap);  // attn_fwd.hip
int kf_form(int64_t pairs, int Sq, int Skv, int D, bool causal, bool teams, int kf);  // attn_fwd.hip; teams: they are a choice

template <typename T, int D, bool CAUSAL, bool EMU, int KF>
hipError_t launch_one(const AttnKernelParams& p0, hipStream_t stream) {
  AttnKernelParams p = p0;
  p.pair_order = 0;
  p.two_blocks = 0;
  p.head_major = 0;
  const int forced = attn_form_override();
  const int64_t BH = (int64_t)p.B * p.H;
  const int64_t cus = device_cu_count();
  const int nMB = (p.Sq + 127) / 128, nMB8 = (p.Sq + 255) / 256;
  const int64_t n4 = nMB * BH, n8 = nMB8 * BH, pairs = (int64_t)((nMB8 + 1) / 2) * BH;
  constexpr bool kNoiseTensor = KF == kKfTensor || KF == kKfTensorLds, kPlain = KF == kKfNone || KF == kKfSoftcap;
  constexpr bool kHas8 = kPlain || KF == kKfSeededTau1 || KF == kKfSeededFast || kNoiseTensor;
  int form = forced;
  if (!(forced & 7)) {
    form = kPlain ? plain_form(BH, p.group, p.Sq, p.Skv, D, CAUSAL, KF == kKfSoftcap)
                  : kHas8 ? kf_form(BH, p.Sq, p.Skv, D, CAUSAL, EMU, KF) : kAttnFour;
  }
  if constexpr (kHas8) {
    if ((form & 7) >= kAttnEight) {
      p.two_blocks = kAttnTwoBlocks && kPlain && CAUSAL && nMB8 >= 2 && (form & 7) == kAttnEightPaired;
      p.head_major = BH % 8 == 0 && (form & kAttnHeadMajor) != 0;
      hipLaunchKernelGGL((attn_fwd_kernel<T, D, CAUSAL, EMU, KF, 8>), dim3((unsigned)(p.two_blocks ? pairs : n8)), dim3(512), 0, stream, p);
      return hipGetLastError();
    }
  }
  dim3 grid((unsigned)n4);
  p.pair_order = CAUSAL && (int64_t)grid.x <= 2 * cus;  // two workgroups of this form per CU
  p.head_major = BH % 8 == 0 && !p.pair_order && (form & kAttnHeadMajor) != 0;
  // no more workgroups than CUs: room for one in each (the dispatcher puts two on some otherwise, and leaves others idle)
  const unsigned pad = kPlain && n4 <= cus ? 88 * 1024 - 4 * kAttnBN * 2 * D : 0;
  hipLaunchKernelGGL((attn_fwd_kernel<T, D, CAUSAL, EMU, KF, 4>), grid, dim3(256), pad, stream, p);
  return hipGetLastError();
}

template <typename T, int D>
hipError_t launch_td(const AttnKernelParams& p, bool causal, bool emu, int kf, hipStream_t s) {
#define FT_CASE(C, E, K) \
  if (causal == C && emu == E && kf == K) return launch_one<T, D, C, E, K>(p, s);
  FT_CASE(true, true, kKfNone) FT_CASE(true, false, kKfNone) FT_CASE(false, true, kKfNone) FT_CASE(false, false, kKfNone)
  FT_CASE(true, true, kKfTensor) FT_CASE(true, false, kKfTensor) FT_CASE(false, true, kKfTensor) FT_CASE(false, false, kKfTensor)
  FT_CASE(true, true, kKfTensorLds) FT_CASE(true, false, kKfTensorLds) FT_CASE(false, true, kKfTensorLds) FT_CASE(false, false, kKfTensorLds)
  FT_CASE(true, true, kKfSeeded) FT_CASE(true, false, kKfSeeded) FT_CASE(false, true, kKfSeeded) FT_CASE(false, false, kKfSeeded)
  FT_CASE(true, true, kKfSoftcap) FT_CASE(true, false, kKfSoftcap) FT_CASE(false, true, kKfSoftcap) FT_CASE(false, false, kKfSoftcap)
  if constexpr (std::is_same<T, F16>::value) {  // packed KeyFormer modes: fp16 with reference rounding only
    if (emu) {
      FT_CASE(true, true, kKfSeededTau1) FT_CASE(false, true, kKfSeededTau1)
      FT_CASE(true, true, kKfSeededFast) FT_CASE(false, true, kKfSeededFast)
    }
  }
#undef FT_CASE
  return hipErrorInvalidValue;
}

}  // namespace ft
