// Dispatcher of the fused softmax attention forward: picks the instantiation of attn_fwd_kernel.hpp built by
// attn_fwd_{f16,bf16}_{d64,d128}.hip for the element type and head size of the call.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdlib>

#include "kernel_params.h"

namespace ft {

int device_cu_count() {
  static std::atomic<int> cus[16];  // zero-initialised; a racing first call stores the same value twice
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 16) return 256;
  int n = cus[dev].load(std::memory_order_relaxed);
  if (n == 0) {
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    cus[dev].store(n, std::memory_order_relaxed);
  }
  return n;
}

// Test hook: FT_ATTN_FORM in the environment overrides the launch shape the dispatcher would pick for the
// problem size ("4": 128-row workgroups; "8": 256-row workgroups, one query block each; "8x2": 256-row workgroups
// that take the heaviest and the lightest remaining block; an "h" appended: head-major workgroup order; "t": two teams of waves), so that
// every form can be checked on every shape whatever the CU count of the device.  Read on every launch.
int attn_form_override() {
  const char* e = getenv("FT_ATTN_FORM");
  if (!e || !*e) return 0;
  int form = 0;
  if (e[0] == '4') form = 1;
  else if (e[0] == '8') form = (e[1] == 'x' && e[2] == '2') ? 3 : 2;
  else if (e[0] == 't') form = 16;
  for (const char* c = e; *c; ++c)
    if (*c == 'h') form |= 8;
  return form;
}

// The same variable for the split form: "s<n>" shares out n tiles at a time, any other override keeps blocks whole.
int attn_split_override() {
  const char* e = getenv("FT_ATTN_FORM");
  if (!e || !*e) return 0;
  if (e[0] != 's') return -1;
  const int n = atoi(e + 1);
  return n > 0 ? n : -1;
}

hipError_t launch_attn_f16_d64(const AttnKernelParams& p, bool causal, bool emu, int kf, hipStream_t s);
hipError_t launch_attn_f16_d128(const AttnKernelParams& p, bool causal, bool emu, int kf, hipStream_t s);
hipError_t launch_attn_bf16_d64(const AttnKernelParams& p, bool causal, bool emu, int kf, hipStream_t s);
hipError_t launch_attn_bf16_d128(const AttnKernelParams& p, bool causal, bool emu, int kf, hipStream_t s);

hipError_t launch_attn_teams_f16(const AttnKernelParams& p, int D, bool emu, int kf, unsigned grid, hipStream_t s);
hipError_t launch_attn_teams_bf16(const AttnKernelParams& p, int D, bool emu, int kf, unsigned grid, hipStream_t s);
hipError_t launch_attn_teams_kf_f16(const AttnKernelParams& p, int D, int kf, unsigned grid, hipStream_t s);
hipError_t launch_attn_teams_kf_bf16(const AttnKernelParams& p, int D, int kf, unsigned grid, hipStream_t s);

// A form of the attention pass as launches are compared by: rows and teams of a workgroup, how many of them a CU holds, and the
// microseconds that one takes to begin and end and per key tile (of each team), alone on its CU and beside another.  Fitted to
// the differences between forms in 1900 random calls (some of them: tests/test_launch_forms.py).  Soft-capped ones by both types alike,
// since when fp16 has become shorter, two teams of D = 128 by 1 %, the other forms by 5 to 9, few tiles under the mask by up to 7 more:
// the form chosen is 0.6 % slower than the best one in the mean over the test's calls of either type (fp16 0.8 % before).
struct Form {
  int rows, teams, per_cu;
  double first, tile, shared;
};
constexpr Form kPlainTeams{64, 2, 1, 5.4, 0.94, 0.94}, kPlainFour{128, 1, 2, 6.2, 0.56, 0.82};  // D = 128
constexpr Form kCapTeams{64, 2, 1, 5.4, 1.68, 1.68}, kCapFour{128, 1, 2, 5.8, 1.3, 1.79};
constexpr Form kSeededTeams{64, 2, 1, 4.4, 1.84, 1.84}, kSeededFour{128, 1, 2, 4.8, 1.56, 1.79};
constexpr Form kTensorTeams{64, 2, 1, 3.2, 2.78, 2.78}, kTensorFour{128, 1, 1, 2.8, 2.54, 2.54}, kTensorEight{256, 1, 1, 2.6, 3.46, 3.46};
constexpr Form kTensorTeams64{64, 2, 1, 2.7, 1.58, 1.58}, kTensorFour64{128, 1, 2, 2.1, 1.62, 1.82};  // D = 64

// Workgroups are handed out longest first.  One round takes as long as its longest workgroup; of two, the second begins where the
// first one's shortest ends, with one as long; more take as long as all of the work spread evenly, and what the last round leaves
// empty is filled but for the shortest one's time.
static double form_us(const Form& f, int64_t pairs, int group, int Sq, int Skv, bool causal) {
  const int64_t rows = (int64_t)Sq * group, wgs = (rows + f.rows - 1) / f.rows * pairs, cus = device_cu_count();
  auto tiles = [&](int64_t upto) {  // of the block that ends with this row
    const int64_t keys = causal ? std::min<int64_t>(Skv, (upto - 1) / group + 1 + Skv - Sq) : Skv;
    return ((keys + 63) / 64 + f.teams - 1) / f.teams;
  };
  const double tile = wgs <= cus ? f.tile : f.shared, rounds = (double)wgs / (double)(f.per_cu * cus);
  const double most = f.first + tile * tiles(rows), least = f.first + tile * tiles(std::min<int64_t>(f.rows, rows));
  if (rounds <= 1) return most;
  return std::max(most, rounds <= 2 ? 2 * (most - (most - least) / rounds) : rounds * (most + least) / 2 + (std::ceil(rounds) - rounds) * least);
}

// Two teams of waves on blocks of 64 rows (attn_split.hpp) instead of four waves on 128: half the rows and half the chain of
// key tiles per workgroup.  Taken where the chain is the launch: with a workgroup of this form for every CU at most, from
// ten key tiles on (attention calls, same process: B1 H8 D128 S1000 21.1 -> 18.1 us, S2048 35.6 -> 29.3; D64, of whose
// workgroups a CU holds two, from five tiles on: H8 S1000 14.9 -> 12.0).  Shorter plain calls have 2 us at most to gain
// (S500 14.0 -> 12.3) and keep to the forms whose results agree bit for bit; soft-capped ones, whose waves are slow
// enough alone, take it from four tiles on (fp16 S300 13.1 -> 11.8, S500 18.8 -> 15.0, S130 9.2 either way).
// Under the causal mask with more of them too, where the blocks differ in length enough that the second round fills the gaps of the
// first.  D64: up to two for every CU (H8 S3000 33.5 -> 27.2, B2 H32 S500 10.7 -> 9.4) or, over more than 32 tiles, five for two (H16
// S2500 31.7 -> 26.9, S3000 36 -> 38), longer ones than 48 again keeping to the bit-equal forms; soft-capped up to thirteen for four
// CUs (fp16 H16 S3000 67 -> 55, H32 S1500 37.6 -> 33.0, B2 H32 S777 23.8 either way, S1000 26.8 -> 30.9).  D128: up to three for two CUs (H8 S3000
// 48 -> 40; H16 S2048, four for two, 36.6 -> 35.8, H32 S777 17.7 -> 20.8), soft-capped over twelve tiles or more four for two (bf16 H32 S777
// 29.4 -> 26.8, fp16 25.7 -> 24.7) and over more than 32 five (bf16 H16 S2500 89.7 -> 86.6, S3000 98 -> 112; fp16, of which four waves'
// tiles have become shorter since and two teams' have not, 73.5 -> 76.9), where the two launches' times say so too: chunks
// over many more keys than queries, whose blocks are nearly alike, take the second round in full (attention of H16/2 Sq1101 Skv12131
// 189 -> 265 us; over 200 random calls 7 % of the time, 53 % at most).
bool use_teams(int64_t pairs, int group, int Sq, int Skv, int D, bool causal, bool cap) {
  const int forced = attn_form_override();
  if (forced || attn_split_override()) return (forced & 16) != 0;
  const int64_t cus = device_cu_count(), grid = ((int64_t)Sq * group + 63) / 64 * pairs;
  const int tiles = (Skv + 63) / 64;
  if (tiles <= (cap ? 3 : D == 64 ? 5 : 10)) return false;
  if (grid <= cus) return true;
  if (!causal) return false;
  if (D == 64) return cap ? 4 * grid <= 13 * cus : tiles <= 48 && 2 * grid <= (tiles > 32 ? 5 : 4) * cus;
  if (2 * grid > (cap ? tiles > 32 ? 5 : 4 : 3) * cus || (cap && tiles <= 11)) return false;
  return form_us(cap ? kCapTeams : kPlainTeams, pairs, group, Sq, Skv, true) < form_us(cap ? kCapFour : kPlainFour, pairs * group, 1, Sq, Skv, true);
}

// 256-row workgroups (8 waves) stage K and V once for twice the rows, but round every prompt up to 256 rows and are half as many:
// under the causal mask the 128-row form is the faster one nearly everywhere (attention, B4 H32 D128 S777 53.5 -> 42.2 us, S1024
// 55.5 -> 51.3, S2600 321 -> 278, B2 S2600 151 -> 135; D64 B4 S1300 61 -> 51; soft-capped fp16 B4 S777 67 -> 51).
// - plain, soft-cap, causal: where hardly a row is padding and the blocks pair up, heaviest with lightest, into whole rounds of
//   the chip: one round (B1 H32 S4096 151.9 -> 148.5), or three and more, for which an XCD finishes a pair's blocks before it
//   starts the next pair's (B8 H32 S1536 229 -> 214, S2048 387 -> 373, B3 S4096 453 -> 443; two rounds B2 H32 S4096 292.5 and
//   293.7, B4 S2048 166 and 169).  D64 and soft-capped logits from four rounds on (B4 H32 S4096 360 -> 351, soft-capped fp16 860 ->
//   834, bf16 927 -> 896; three rounds 204 and 211, fp16 604 and 615), D64 at one round (89.5 -> 88.5; soft-capped bf16 218 and 221, fp16 199 either way).  Over half as many keys
//   again as queries the blocks are nearly alike, and D128 pairs them up at any whole number of rounds, soft-capped from four
//   blocks on (B8 H32 S1024 Skv2924 452 -> 364, B2 S2048 Skv5645 319 -> 311; soft-capped fp16 B8 H32/4 S1024 Skv10041 1893 -> 1752,
//   B4 H16 S2048 Skv4098 298 -> 293, B8 H32 S512 Skv1050 100 either way).
// - no mask: D128 up to 127 (b, h) pairs (B2 H32 S3600 477 -> 463; B4 S1024 86 -> 90; D64 B2 S2048 86 -> 98), where the last round, of
//   one workgroup a CU, is three quarters full or one of many (H24 B3 S2048 Skv5231, two rounds and a quarter, 436 against 486, soft-capped
//   fp16 B2 S2600 250 against 346).
// Head-major where the K and V of all pairs together are beyond every cache: with the mask from 256 pairs and nine rounds on (B8
// H32 S2304 475 -> 445 us, S2600 645 -> 570, soft-capped fp16 839 -> 762; S2048 374, paired 256-row blocks 373), without from 128 pairs
// (256 at D64) and two and a half rounds on (D128 B4 H32 S2600 518 -> 491, B8 S1024 193 -> 165, D64 99.5 -> 93; B4 D128 S513 38.6 -> 41.5).
// And where K and V outgrow the memory-side cache and blocks are alike in length: without the mask over 256 MB (B8 H32 S512 Skv6690
// D128 651 -> 492 us), over half as many keys again as queries over 400 (B8 H32 S1437 Skv3859 984 -> 710, S689 Skv7010 D64 509 ->
// 418; 256 to 400 MB 0.92 to 1.05 of the time).
int plain_form(int64_t BH, int group, int Sq, int Skv, int D, bool causal, bool cap) {
  const int64_t cus = device_cu_count(), nMB8 = ((int64_t)Sq + 255) / 256;
  const int64_t n4 = ((int64_t)Sq + 127) / 128 * BH, n8 = nMB8 * BH, pairs = (nMB8 + 1) / 2 * BH, rounds = pairs / cus;
  const bool long_keys = 2 * (int64_t)Skv >= 3 * (int64_t)Sq;
  if (causal) {
    const bool any = D == 128 && long_keys && (!cap || nMB8 >= 4);
    if (nMB8 >= 2 && pairs % cus == 0 && nMB8 * 256 * 100 <= (int64_t)Sq * 103 && (any || (rounds == 1 && !cap) || rounds >= (D == 128 && !cap ? 3 : 4)))
      return kAttnEightPaired | (rounds >= (any ? 2 : 3) ? kAttnHeadMajor : 0);
  } else if (D == 128 && BH < 128 && 4 * n8 >= 7 * cus && (n8 % cus == 0 || 4 * (n8 % cus) >= 3 * cus || n8 >= 5 * cus)) {
    return kAttnEight;
  }
  const double kv_bytes = (double)(BH / group) * Skv * D * 4;
  const bool far = (BH >= (causal || D == 64 ? 256 : 128) && n4 >= (causal ? 18 * cus : 5 * cus)) ||
                   (n4 > 2 * cus && (causal ? long_keys && kv_bytes > 400e6 : kv_bytes > 256e6));
  return kAttnFour | (far ? kAttnHeadMajor : 0);
}

// KeyFormer's passes do two to four times the vector work per tile, so the chain of a block's tiles bounds launches of more
// workgroups still, and half the chain pays from two key tiles on, always with a workgroup of teams for every CU at most (whole calls,
// same process, four waves on 128 rows against the teams: D128, noise from a tensor, B1 H8 S100 16.9 -> 15.5 us, S64 12.5 -> 14.0), and
// with more of them by the launches' times: under the mask noise from a tensor H8 S2091 165 -> 118, H32 S1500 148 -> 130, from a
// seed H8 S1003 51.8 -> 40.5; without it, or over many more keys than queries, not before a round is full (seeded B4 H16 S512
// 43.9 against 35.2 in one round of four waves).  Seeded noise at D64, two workgroups of teams a CU: up to nine for two CUs (H16 S3543
// 142 -> 127, H32 S2091 100 -> 95, S2527 128 -> 129), but where four waves fill just one round (B4 H32 S512 without the mask 46.1
// against 50.8, B2 H32 S1024 with it 50.7 against 56.6).
// 256-row workgroups: noise from a tensor at D128, whose slices leave a CU room for one workgroup of either form, by the launches' times as
// well (without the mask H32 S2048 311 -> 253, S2048 Skv4097 683 -> 563; H32 S2527 315 -> 297); at D64, where two of the 128-row form
// fit, from seven for four CUs on (H32 S3543 423 -> 408, S2527 226 -> 253) and, without the mask, for one full round (H32 S2048
// 235 -> 225).  Seeded noise, packed: D128 from two workgroups per CU on (B1 H32 S4096 345 -> 340 us whole; D64 260 -> 269).
// At most seven workgroups of teams for two CUs (noise from a tensor, D128), three for one (D64), five for two (seeded, D128): beyond,
// the blocks of one round of four waves share their CUs with shorter ones (H12 S4096, three for one, seeded 183 -> 206).
// Over 730 random calls of more teams than CUs the form so chosen is 0.3 % slower than the fastest on average (by counts of
// workgroups alone, as measured under the mask for prompts: 5.8 %, 36 % at most).
int kf_form(int64_t pairs, int Sq, int Skv, int D, bool causal, bool teams, int kf) {
  const bool tensor = kf == kKfTensor || kf == kKfTensorLds;
  const int64_t cus = device_cu_count(), grid = ((int64_t)Sq + 63) / 64 * pairs, n8 = ((int64_t)Sq + 255) / 256 * pairs;
  auto us = [&](const Form& f) { return form_us(f, pairs, 1, Sq, Skv, causal); };
  teams = teams && Skv > 64 && 2 * grid <= (tensor ? D == 128 ? 7 : 6 : D == 128 ? 5 : 9) * cus;
  if (teams && grid <= cus) return kAttnTeams;
  if (tensor && D == 128) {
    const double four = us(kTensorFour), eight = us(kTensorEight);
    if (teams && us(kTensorTeams) < std::min(four, eight)) return kAttnTeams;
    return eight < four ? kAttnEight : kAttnFour;
  }
  if (tensor) {
    if (teams && us(kTensorTeams64) < us(kTensorFour64)) return kAttnTeams;
    return 4 * n8 >= 7 * cus || (!causal && n8 <= cus && 10 * n8 >= 9 * cus) ? kAttnEight : kAttnFour;
  }
  if (D == 128) return teams && us(kSeededTeams) < us(kSeededFour) ? kAttnTeams : n8 >= 2 * cus ? kAttnEight : kAttnFour;
  // (four waves' one round under the mask: the generic path of long prompts is slow enough alone, S2048 bf16 teams 112, 121)
  const bool round = grid <= 4 * cus && (causal ? 10 * grid > 39 * cus && (kf != kKfSeeded || Sq <= 512) : 10 * grid > 35 * cus);
  return teams && !round ? kAttnTeams : kAttnFour;
}

hipError_t launch_attn_fwd(const AttnKernelParams& p, int D, bool bf16, bool causal, bool emu, int kf, hipStream_t s) {
  const int64_t rows = (int64_t)p.Sq * p.group, grid = (rows + 63) / 64 * p.B * (p.H / p.group);
  if ((kf == kKfNone || kf == kKfSoftcap) && rows < 0x7fffffff - 64 && grid < 0x7fffffff && use_teams((int64_t)p.B * (p.H / p.group), p.group, p.Sq, p.Skv, D, causal, kf == kKfSoftcap)) {
    AttnKernelParams pp = p;
    if (!causal) pp.off = p.Skv;
    // (D = 64: two workgroups per CU; see the kernel)
    pp.pair_order = causal && D == 64 && grid > device_cu_count() && grid <= 2 * device_cu_count();
    return bf16 ? launch_attn_teams_bf16(pp, D, emu, kf, (unsigned)grid, s) : launch_attn_teams_f16(pp, D, emu, kf, (unsigned)grid, s);
  }
  const bool tensor = kf == kKfTensor || kf == kKfTensorLds, seeded = kf == kKfSeeded || kf == kKfSeededTau1 || kf == kKfSeededFast;
  const int forced = attn_form_override();
  if (emu && (tensor || seeded) && grid < 0x7fffffff && (forced ? (forced & 16) != 0 : kf_form((int64_t)p.B * p.H, p.Sq, p.Skv, D, causal, true, kf) == kAttnTeams)) {
    AttnKernelParams pp = p;
    if (!causal) pp.off = p.Skv;
    pp.pair_order = pp.two_blocks = pp.head_major = 0;
    return bf16 ? launch_attn_teams_kf_bf16(pp, D, kf, (unsigned)grid, s) : launch_attn_teams_kf_f16(pp, D, kf, (unsigned)grid, s);
  }
  if (D == 128) return bf16 ? launch_attn_bf16_d128(p, causal, emu, kf, s) : launch_attn_f16_d128(p, causal, emu, kf, s);
  if (D == 64) return bf16 ? launch_attn_bf16_d64(p, causal, emu, kf, s) : launch_attn_f16_d64(p, causal, emu, kf, s);
  return hipErrorInvalidValue;
}

}  // namespace ft
