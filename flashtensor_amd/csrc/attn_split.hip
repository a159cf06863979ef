// When attention splits the keys of its row blocks (attn_split.hpp), and the kernel that folds the shares.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "attn_split.hpp"

namespace ft {

hipError_t launch_attn_split_f16(const AttnKernelParams& p, int D, bool emu, int kf, unsigned grid, unsigned lds, hipStream_t s);
hipError_t launch_attn_split_bf16(const AttnKernelParams& p, int D, bool emu, int kf, unsigned grid, unsigned lds, hipStream_t s);

bool use_teams(int64_t pairs, int group, int Sq, int Skv, int D, bool causal, bool cap);  // attn_fwd.hip

namespace {

struct SplitShape {
  int B, H, group, Sq, Skv, D, forced, cus;
  bool causal, cap, stats;
  bool operator==(const SplitShape& o) const {
    return B == o.B && H == o.H && group == o.group && Sq == o.Sq && Skv == o.Skv && D == o.D && forced == o.forced && cus == o.cus && causal == o.causal && cap == o.cap && stats == o.stats;
  }
};

// Microseconds by which launches are compared, fitted to 3700 calls of random shapes in every form, 1 to 96 shares a block, for the
// least regret of the choice, the least loss of any call against the plan before and the least error of the time (some of them,
// and what the choice has to reach: tests/test_split_plan_times.py).
//   A launch 4.4; K, V and kept logits come and go at 7.2 MB/us.
//   A tile 0.98 where a workgroup has its CU to itself and 1.74 where two share one, whose second one starts 0.6 late (soft-capped
//   logits 1.72 and 2.9); D = 64 takes 0.72 of that (soft-capped, whose chain is not shorter for it, 0.82); blocks of one wave, whose
//   other waves only load, feel 0.18 of the difference; a tile whose logits are kept takes a quarter more.
//   (Soft-capped logits by bf16; fp16's tiles, whose chain is shorter, take 0.93 to 0.97 of that in every form, and the choice is as
//   good for them: 0.9 % slower than the best form in the mean over the test's calls, of either type.  Figures a tenth lower change
//   the form of 227 of 3496 random calls, fp16 1.1 % faster in the mean, 0.81 to 1.16, but bf16 1.7 % slower, 0.92 to 1.17.)
//   A step of two teams 1.44 (2.1; D = 64 0.65 and 0.82 of it), and 1.45 times that where two workgroups share a CU (D = 64), unless
//   a team has one wave of rows.
//   Partial results are written and folded at 7.2 MB/us (0.55 of that time beside the column sums), by a kernel that takes 3.5 to
//   begin with and 0.75 for every further round of eight shares.
//   In a launch of more workgroups than fit at once each further one in a slot takes 2.3 until its first tile has landed (0.2 with
//   more waves than one, which hide it).
// Of 18800 calls the form so chosen is 0.8 % slower than the best one on average and 3 % in one of ten; without the terms for a shared
// CU, for soft-capped D = 64 and for kept logits 1.2 % and 4 %, and one call in 40 took over 5 % more than by the plan before those
// figures (H32 Sq540 Skv3350 D64 soft-capped 62 -> 82 us), now one in 135.
constexpr double kLaunch = 4.4, kCombine = 3.5, kFoldRound = 0.75, kSecond = 0.6, kPartBytes = 7.2e6, kKvBytes = 7.2e6, kMix = 0.22;

// `count` shares of `len` tiles.
struct ShareRun {
  int len, count;
};

// When the last workgroup of a launch ends that has more of them than slots: `copies` of every share, longest first, each
// to the slot that is free first.  Slots that come free together are one entry (there are few: a run adds at most one), so
// that a round of equal workgroups is one step, and a run on slots that are all free together none at all.
double rounds_us(const ShareRun* runs, int nruns, int64_t copies, int slots, double tile_us, double next_us) {
  struct Free {
    double at;
    int64_t n;
  } f[kSplitMaxBlocks + 2];
  int nf = 1;
  f[0] = {0.0, slots};
  for (int r = 0; r < nruns; ++r) {
    const double us = runs[r].len * tile_us + next_us;
    int64_t left = runs[r].count * copies;
    while (left > 0) {
      if (nf == 1 && left >= f[0].n) {
        f[0].at += us * (double)(left / f[0].n);
        left %= f[0].n;
        continue;
      }
      const int64_t n = std::min(left, f[0].n);
      const double at = f[0].at + us;
      left -= n;
      f[0].n -= n;
      if (f[0].n == 0) std::copy(f + 1, f + nf--, f);
      int i = nf;
      while (i > 0 && f[i - 1].at > at) --i;
      if (i > 0 && f[i - 1].at == at) {
        f[i - 1].n += n;
      } else {
        std::copy_backward(f + i, f + nf, f + nf + 1);
        f[i] = {at, n};
        ++nf;
      }
    }
  }
  return f[nf - 1].at;
}

SplitPlan make_plan(const SplitShape& a) {
  SplitPlan plan{};
  const int64_t pairs = (int64_t)a.B * (a.H / a.group);
  const int rows = a.Sq * a.group, nMB = (rows + 127) / 128, off = a.causal ? a.Skv - a.Sq : a.Skv;
  const int cus = a.cus;
  int tiles[kSplitMaxBlocks];
  int64_t total = 0;
  for (int mb = 0; mb < nMB; ++mb) {
    tiles[mb] = (std::min(a.Skv, (std::min(mb * 128 + 128, rows) - 1) / a.group + 1 + off) + 63) / 64;
    total += tiles[mb];
  }
  const int most = tiles[nMB - 1], part_waves = std::min(4, (rows + 31) / 32);
  // few rows: the column sums come from kept logits (2 bytes a pair each way against K once more and another launch)
  const bool keep = a.stats;
  const double size = a.D == 128 ? 1.0 : a.cap ? 0.82 : 0.72, alone = (a.cap ? 1.72 : 0.98) * size * (keep ? 1.26 : 1.0);
  const double full_cu = (a.cap ? 2.9 : 1.74) * size, shared_cu = part_waves == 1 ? alone + (full_cu - alone) * 0.18 : full_cu;
  const double next_us = part_waves == 1 ? 2.3 : 0.2;
  const double kv_us = pairs * (double)a.Skv * (a.D * 4 + (keep ? rows * 2 : 0)) / kKvBytes;
  auto launch_us = [&](double work) { return kLaunch + std::max(work, kv_us) + kMix * std::min(work, kv_us); };
  // second: tiles of the workgroup that shares a CU with the longest one, where all of them are resident at once
  auto resident_us = [&](int64_t wgs, int longest, int second, double shared_tile) {
    return wgs <= cus ? longest * alone : second * shared_tile + (longest - second) * alone + kSecond;
  };
  // more than that: handed out in order (longest first) to the slots of an XCD as they become free
  const int slots = std::max(1, 2 * cus / 8);
  const int64_t per_xcd = (pairs + 7) / 8;
  int lanes = 1;  // of a wave's 32 rows that have a share each to fold (combine_rows)
  while (lanes < std::min(rows, 32)) lanes *= 2;
  double best = 1e30;
  int best_chunk = 0;
  const int64_t teams = (rows + 63) / 64 * pairs;
  if (!keep && use_teams(pairs, a.group, a.Sq, a.Skv, a.D, a.causal, a.cap)) {  // undivided: two teams of waves per 64 rows
    const bool two_per_cu = a.D == 64 && teams > cus;
    const double step = (a.cap ? 2.1 : 1.44) * (a.D == 128 ? 1.0 : a.cap ? 0.82 : 0.65) * (two_per_cu && rows > 32 ? 1.45 : 1.0);
    int64_t sum = 0;
    int longest = 0;
    for (int r = 64; r < rows + 64; r += 64) {
      longest = ((std::min(a.Skv, (std::min(r, rows) - 1) / a.group + 1 + off) + 63) / 64 + 1) / 2;
      sum += longest;
    }
    // all at once, or as many rounds of the average, the last one of those that share a CU alone if there is one for every CU at most
    const int64_t nteams = (rows + 63) / 64, per_round = (two_per_cu ? 2 : 1) * cus, rest = teams % per_round;
    const double rounds = teams / per_round + (rest == 0 ? 0 : two_per_cu && rest <= cus && rows > 32 ? 1 / 1.45 : 1);
    best = launch_us(teams <= per_round ? longest * step : std::max((double)longest, (double)sum / nteams * rounds) * step);
  } else if (!keep) {  // a workgroup per 128 queries of a head, whose waves all work (part_waves is the split form's)
    const int nq = (a.Sq + 127) / 128;
    int64_t sum = 0;
    for (int i = 0; i < nq; ++i) sum += (std::min(a.Skv, std::min(i * 128 + 128, a.Sq) + off) + 63) / 64;
    const int64_t wgs = (int64_t)a.B * a.H * nq;
    // heavy and light blocks share a CU: the average makes up the longest block's company
    best = launch_us(wgs <= 2 * cus ? resident_us(wgs, most, (int)std::max<int64_t>(0, std::min<int64_t>(most, 2 * sum / nq - most)), full_cu)
                                    : std::max(most * alone, (double)sum * a.B * a.H * full_cu / (2.0 * cus) + 0.25 * most * alone));
  }
  if (nMB > 1) best *= 0.98;  // (a workspace of tens of megabytes and a second launch for less than the figures can tell apart)
  for (int parts = 1; parts <= kSplitMaxItems; ++parts) {
    const int chunk = a.forced > 0 ? a.forced : (most + parts - 1) / parts;
    if (parts > 1 && chunk == (most + parts - 2) / (parts - 1) && !a.forced) continue;
    int items = 0, shared = 0, nruns = 0;
    ShareRun runs[kSplitMaxBlocks];  // longest first
    for (int mb = nMB - 1; mb >= 0 && items <= kSplitMaxItems; --mb) {
      const int nch = (tiles[mb] + chunk - 1) / chunk, len = (tiles[mb] + nch - 1) / nch;
      items += nch;
      shared += nch > 1 ? nch : 0;
      int at = nruns;
      while (at > 0 && runs[at - 1].len < len) --at;
      if (at > 0 && runs[at - 1].len == len) {
        runs[at - 1].count += nch;
      } else {
        for (int j = nruns++; j > at; --j) runs[j] = runs[j - 1];
        runs[at] = {len, nch};
      }
    }
    if (items > kSplitMaxItems) break;
    const int64_t wgs = items * pairs;
    const int rounds = (((most + chunk - 1) / chunk + 7) / 8 * lanes + 31) / 32;
    // (where logits are kept the second launch is made anyway: H8 Sq2 Skv230 D128 13.2 -> 9.6 us, B4 H32 Sq1 Skv574 18.5 -> 15.9; not
    // where undivided blocks are a workgroup per CU: B8 H32 Sq1 Skv700 23.2 -> 27.0, B16 H16 Sq1 Skv133 12.1 -> 14.5)
    const double fold = shared ? (keep && pairs * nMB < cus ? 0 : kCombine) + kFoldRound * (rounds - 1) + (double)shared * pairs * std::min(rows, 128) * a.D * 4 * (keep ? 0.55 : 1.0) * 2 / kPartBytes : 0;
    // The search ends where no further cut can win: smaller shares mean more of them, so the folding, and in a launch of
    // several rounds the least that the slots' work adds up to, only grow.
    const double least = wgs > 2 * cus ? (total * shared_cu + items * next_us) * per_xcd / slots : 0;
    if (a.forced <= 0 && launch_us(least) + fold >= best) break;
    int second = 0;  // the share at place cus / pairs
    for (int64_t i = 0, left = std::min<int64_t>(items - 1, cus / pairs); i < nruns && left >= 0; left -= runs[i++].count) second = runs[i].len;
    const double us = launch_us(wgs <= 2 * cus ? resident_us(wgs, runs[0].len, second, shared_cu) : rounds_us(runs, nruns, per_xcd, slots, shared_cu, next_us)) + fold;
    if (a.forced > 0 || us < best) {
      best = us;
      best_chunk = chunk;
    }
    if (a.forced > 0 || chunk == 1) break;
  }
  if (!best_chunk) return plan;
  plan.chunk_tiles = best_chunk;
  plan.nblocks = plan.first_shared = nMB;
  plan.part_waves = part_waves;
  int order[kSplitMaxBlocks], len[kSplitMaxBlocks];
  for (int mb = 0; mb < nMB; ++mb) {
    const int nch = (tiles[mb] + best_chunk - 1) / best_chunk;
    order[mb] = mb;
    len[mb] = (tiles[mb] + nch - 1) / nch;
    if (nch > 1) plan.first_shared = std::min(plan.first_shared, mb);
  }
  std::stable_sort(order, order + nMB, [&](int x, int y) { return len[x] > len[y]; });
  for (int i = 0; i < nMB; ++i) {
    const int mb = order[i], nch = (tiles[mb] + best_chunk - 1) / best_chunk;
    plan.first_item[mb] = (uint8_t)plan.items;
    for (int c = 0; c < nch; ++c) plan.list[plan.items++] = (uint16_t)(mb << 8 | c);
  }
  plan.one_per_cu = plan.items * pairs <= cus;
  if (plan.first_shared < nMB) plan.bytes = (size_t)(pairs * plan.items * part_waves * split_wave_floats(a.D)) * sizeof(float);
  if (keep) {
    plan.logit_tiles = (a.Skv + 63) / 64;
    plan.logits_at = plan.bytes;
    plan.bytes += (size_t)(pairs * rows * plan.logit_tiles) * 64 * sizeof(uint16_t);
  }
  return plan;
}

// Whether the column sums of few rows come from kept logits.  Up to 32 rows always; up to kSplitStatRows where the column pass would
// read K once per query head of a group, and a launch take the mean (130 random calls of 33 to 64 rows: H32/8 Sq16 Skv8966 D128
// B4 92 -> 46 us, Sq12 Skv16000 52 -> 27, H16/2 Sq5 Skv10808 D64 25.9 -> 16.2), and for heads of their own where the logits'
// 4 bytes a pair, there and back, cost less than the 2 D bytes a key of K again and a launch (D128 H16 Sq40 Skv16372 46 -> 38,
// Sq48 Skv2524 22.8 -> 18.7, H8 Sq64 Skv10574 24.7 -> 24.3, but H32 Sq64 Skv8000 55.1 -> 57.7; D64 H8 Sq40 Skv5543 17.2 -> 15.1,
// H16 Sq48 Skv10507 25.6 -> 25.8, 64 rows -0.9 to 0.5 us either way).
// More than 32 rows never in more than 4 GiB of workspace: at 2 bytes a row and key they take a quarter of K and V for 64 rows of D = 128
// (half of them, D = 64), so only calls over 8 GiB of K and V reach that.  It is a bound on the scratch, not on the gain: over 4.3
// GiB of them, B128 H32/8 Sq16 Skv8192 D128, the kept logits take 1 GiB and the call 1440 us, the column pass none and 2450.  Up to 32
// rows, an eighth of K and V (a quarter), have no bound: B128 H32/8 Sq8 Skv66000 D128 with 4 GiB for 32 GiB of them 8630 us, the column
// pass 18960 (D64 5670 and 10530; heads of their own, B32 H32 Sq32 D64, 6130 and 5240).
constexpr double kMaxLogitBytes = 4.0 * (1 << 30);

bool keep_logits(int64_t pairs, int group, int64_t rows, int Skv, int D) {
  if (rows <= 32) return true;
  if (rows > kSplitStatRows || (double)pairs * rows * Skv * 2 > kMaxLogitBytes) return false;
  return group > 1 || (rows <= (D == 128 ? kSplitStatRows : 48) && (double)pairs * Skv * (rows - (D == 128 ? 44 : 30)) < 2.5e6);
}

}  // namespace

// stats: column sums of rounded logits are wanted too.  The reference holds until the thread's next call.
// A plan costs 0.1 to 2.4 us of host time (a whole search by simulated launches: 9 to 280) and is asked for several times per
// operator call: each thread keeps its last ones.
const SplitPlan& split_plan(int B, int H, int group, int Sq, int Skv, int D, bool causal, bool cap, bool stats) {
  struct Entry {
    SplitShape shape{};
    SplitPlan plan{};
  };
  constexpr int kEntries = 16;
  static const SplitPlan whole{};
  static thread_local Entry kept[kEntries];
  const int forced = attn_split_override(), cus = device_cu_count();
  const int64_t pairs = (int64_t)B * (H / group), rows = (int64_t)Sq * group;
  if (forced < 0 || rows > 128 * kSplitMaxBlocks || pairs * ((rows + 127) / 128) > 4 * cus) return whole;
  if (Skv > INT32_MAX - 64 || (causal && Skv < Sq)) return whole;  // refused by every entry point
  // A whole prompt (more than half as many queries as keys) keeps its blocks whole: at most a sixth is to be gained there (B1 H8 S2048:
  // 35 against 29 us), and its results are those of every launch form of the unsplit kernel, bit for bit.
  if (Skv < 2 * (int64_t)Sq && forced == 0) return whole;
  // One row block: Skv matters through its tiles only, and a generation loop, whose Skv grows with every step, makes a plan
  // once in 64 steps.
  if (rows <= 128) Skv = (Skv + 63) / 64 * 64;
  const SplitShape shape{B, H, group, Sq, Skv, D, forced, cus, causal, cap, stats && keep_logits(pairs, group, rows, Skv, D)};
  Entry& e = kept[(unsigned)(B * 31 + H * 7 + group * 3 + Sq * 5 + Skv / 64 + D + cap + 2 * shape.stats) % kEntries];
  if (!(e.shape == shape)) e = Entry{shape, make_plan(shape)};
  return e.plan;
}

namespace {

__device__ __forceinline__ int shares_of_block(const AttnKernelParams& p, int mb) {
  const int n_end = min(p.Skv, (min(mb * 128 + 128, p.Sq * p.group) - 1) / p.group + 1 + p.off);
  return ((n_end + kAttnBN - 1) / kAttnBN + p.chunk_tiles - 1) / p.chunk_tiles;
}

// Folds the shares of a row, U at a time: running maximum and sum, and Q pieces of four channels (Q = 0: none) of the shares'
// accumulators.  slot0: the row's wave in the first share, n: the row in the wave; every `step`-th share is taken, nch of them.
// A share that shows the row no finite logit has m = kNoMax, l = 0.
template <int U, int Q, typename L>
__device__ __forceinline__ void fold_shares(const AttnKernelParams& p, int D, int64_t slot0, int n, int nch, int step, float& M, float& sum, float4v (&acc)[Q ? Q : 1], L load) {
  M = kNoMax, sum = 0.f;
#pragma unroll
  for (int q = 0; q < Q; ++q) acc[q] = float4v{0.f, 0.f, 0.f, 0.f};
  for (int c0 = 0; c0 < nch; c0 += U) {
    float m[U], l[U];
    float4v o[U][Q ? Q : 1];
#pragma unroll
    for (int u = 0; u < U; ++u) {  // shares past the last one re-read it, with weight 0
      const SplitPartial s = split_partial(p.part, D, slot0 + (int64_t)min(c0 + u, nch - 1) * step * p.part_waves);
      m[u] = s.m[n];
      l[u] = s.l[n];
#pragma unroll
      for (int q = 0; q < Q; ++q) o[u][q] = load(s, q);
    }
    float M1 = M;
#pragma unroll
    for (int u = 0; u < U; ++u) M1 = fmaxf(M1, m[u]);
    const float move = __builtin_amdgcn_exp2f(M - M1);
    sum *= move;
#pragma unroll
    for (int q = 0; q < Q; ++q) acc[q] *= move;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const float w = c0 + u < nch ? __builtin_amdgcn_exp2f(m[u] - M1) : 0.f;
      sum = __builtin_fmaf(w, l[u], sum);
#pragma unroll
      for (int q = 0; q < Q; ++q)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[q][e] = __builtin_fmaf(w, o[u][q][e], acc[q][e]);
    }
    M = M1;
  }
}

// A wave takes Q of the four pieces of (32 rows of a shared block, 32 channels); every load is up to 1 KB contiguous, in the
// accumulators' own register layout.  Bound by the latency of its loads, over many rows by their bytes.
// FEW (up to 32 rows): up to 16 rows (a generation step's) the lanes that have no row take every SUB-th share of the
// others' and meet by lane exchanges, so that eighty shares of four rows are one round of loads and not ten (whole calls: B1 H16/4 Sq1
// Skv5195 16.6 -> 10.6 us, H32/8 Sq1 Skv4000 15.4 -> 11.7, soft-capped B2 H16/4 Sq1 Skv3058 18.6 -> 13.0); eight shares or fewer
// are one round anyway.
// More rows: Q = 2, four shares a round, or Q = 1, eight a round (as it was before); launch_attn_split says which.
template <typename T, int D, int Q, bool FEW>
__device__ __forceinline__ void combine_rows(const AttnKernelParams& p, int first_shared, int unit) {
  constexpr int DB = D / 32;
  const int rows = p.Sq * p.group, Hkv = p.H / p.group;
  const int nshared = (rows + 127) / 128 - first_shared;
  const int q0 = unit % (4 / Q) * Q;
  int i = unit / (4 / Q);
  const int db = i % DB;
  i /= DB;
  const int wv = i % p.part_waves;
  i /= p.part_waves;
  const int mb = first_shared + i % nshared, bh = i / nshared;
  if (bh >= p.B * Hkv) return;
  const int lane = lane_id(), g = lane >> 5;
  int n = lane & 31, sub = 0, rp = 32;  // row in the wave; which shares
  if (FEW) {
    rp = 1;
    while (rp < 32 && (rp < rows || 32 / rp >= 2 * ((shares_of_block(p, mb) + 7) / 8))) rp *= 2;
    sub = n / rp;
    n &= rp - 1;
  }
  const int row = mb * 128 + wv * 32 + n, slots = 32 / rp;
  const int64_t slot0 = ((int64_t)bh * p.nitems + p.first_item[mb]) * p.part_waves + wv;
  const int nch = shares_of_block(p, mb), rc = min(row, rows - 1) - (row - n);  // (lanes without a row repeat the last one)
  float M, L;
  float4v acc[Q];
  fold_shares<8 / Q, Q>(p, D, slot0 + (int64_t)sub * p.part_waves, max(rc, 0), (nch - sub + slots - 1) / slots, slots, M, L, acc,
                                 [&](const SplitPartial& s, int q) { return *reinterpret_cast<const float4v*>(s.o + ((db * 4 + q0 + q) * 64 + g * 32 + max(rc, 0)) * 4); });
  if (FEW) {
    for (int d = rp; d < 32; d *= 2) {
      const float M2 = __shfl_xor(M, d), L2 = __shfl_xor(L, d), M1 = fmaxf(M, M2);
      const float w = __builtin_amdgcn_exp2f(M - M1), w2 = __builtin_amdgcn_exp2f(M2 - M1);
      L = __builtin_fmaf(L2, w2, L * w);
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[0][e] = __builtin_fmaf(__shfl_xor(acc[0][e], d), w2, acc[0][e] * w);
      M = M1;
    }
  }
  if (row >= rows || sub > 0) return;
  const float inv = 1.f / L;
  const int b = bh / Hkv, h = (bh % Hkv) * p.group + row % p.group, qi = row / p.group;
  uint16_t* optr = p.o + b * p.so.b + (int64_t)qi * p.so.s + h * p.so.h;
#pragma unroll
  for (int q = 0; q < Q; ++q)
    *reinterpret_cast<uint2*>(optr + 32 * db + 8 * (q0 + q) + 4 * g) = make_uint2(T::pack2(acc[q][0] * inv, acc[q][1] * inv), T::pack2(acc[q][2] * inv, acc[q][3] * inv));
  if (db == 0 && q0 == 0 && g == 0 && p.lse) p.lse[((int64_t)b * p.H + h) * p.Sq + qi] = M + __builtin_amdgcn_logf(L);
}

template <typename T, int D, int Q, bool FEW>
__global__ void __launch_bounds__(256) attn_combine_kernel(const AttnKernelParams p, int first_shared) {
  combine_rows<T, D, Q, FEW>(p, first_shared, blockIdx.x * 4 + wave_id());
}

// The column sums of few rows from their kept logits, and (the last `gridDim.x - ncol` workgroups) the folding of the
// shares: one launch where the column pass would read K a second time, per query head, behind the launch that folds.
// B4 H32/8 Sq1 Skv4097: 31 + 5 us (column pass, group mean) and 4 for the folding -> 4.1 for all of it.
// A workgroup takes 512 keys of one (b, k/v head), eight of them per lane; its waves share out the rows and meet in LDS.
// A wave requests all of its rows (1 KB each) before the row normalisers are folded.
constexpr int kStatTiles = 8;
__host__ __device__ constexpr int stat_step(int pool) { return pool ? kStatTiles - 1 : kStatTiles; }  // half a tile on either side for the window

// WIDE: more than 32 rows.
template <typename T, int D, bool SQ, bool WIDE>
__global__ void __launch_bounds__(256) split_stats_kernel(const AttnKernelParams p, const SplitStats st, int ncol) {
  if ((int)blockIdx.x >= ncol) {
    combine_rows<T, D, 1, !WIDE>(p, 0, (blockIdx.x - ncol) * 4 + wave_id());
    return;
  }
  constexpr int KT = kStatTiles * kAttnBN;
  constexpr bool kF16 = __is_same(typename T::elem, _Float16);
  constexpr int kRows = WIDE ? kSplitStatRows : 32;
  __shared__ float s_nlse[kRows];
  __shared__ __align__(16) float s_sum[4][KT];
  __shared__ __align__(16) float s_sq[SQ ? 4 : 1][SQ ? KT : 4];
  const int rows = p.Sq * p.group, Hkv = p.H / p.group, pairs = p.B * Hkv;
  const int bh = blockIdx.x % pairs, tile = blockIdx.x / pairs;
  const int t = threadIdx.x, lane = lane_id(), wave = wave_id();
  const int tile0 = tile * stat_step(st.pool) - (st.pool ? 1 : 0);
  const int k0 = 8 * lane, j0 = tile0 * kAttnBN + k0;  // the lane's first key, of the workgroup's and of the row
  const int stride = p.logit_tiles * kAttnBN;
  const uint16_t* col = p.logits + (int64_t)bh * rows * stride + max(0, min(j0, stride - 8));
  const int per = (rows + 3) >> 2;  // rows of a wave, the last ones past the end
  float sum[8] = {}, sq[8] = {};
  auto rows_of_wave = [&](auto n_tag) __attribute__((always_inline)) {
    constexpr int N = decltype(n_tag)::value;
    uint4v w[N];
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int r = min(wave * per + min(i, per - 1), rows - 1);
      w[i] = *reinterpret_cast<const uint4v*>(col + (int64_t)r * stride);
    }
    // eight threads a row for its shares (WIDE: four): one round of loads up to 64 shares (32)
    constexpr int parts = 256 / kRows;
    const int row = t & (kRows - 1), part = t / kRows, rc = min(row, rows - 1);
    const int nch = shares_of_block(p, 0);
    if (nch > 1) {
      float M = kNoMax, L = 0.f;
      float4v none[1];
      if (part < nch)
        fold_shares<8, 0>(p, D, ((int64_t)bh * p.nitems + part) * p.part_waves + rc / 32, rc % 32, (nch - part + parts - 1) / parts, parts, M, L, none,
                          [](const SplitPartial&, int) { return float4v{}; });
      s_sum[0][t] = M;
      s_sum[1][t] = L;
      __syncthreads();
      if (t < kRows) {
#pragma unroll
        for (int u = 1; u < parts; ++u) M = fmaxf(M, s_sum[0][kRows * u + t]);
        L = 0.f;
#pragma unroll
        for (int u = 0; u < parts; ++u) L = __builtin_fmaf(__builtin_amdgcn_exp2f(s_sum[0][kRows * u + t] - M), s_sum[1][kRows * u + t], L);
        s_nlse[t] = -(M + __builtin_amdgcn_logf(L));
      }
    } else if (t < kRows) {
      s_nlse[t] = -p.lse[((int64_t)(bh / Hkv) * p.H + (bh % Hkv) * p.group + rc % p.group) * p.Sq + rc / p.group];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int r = wave * per + i;
      const float nlse = s_nlse[min(r, rows - 1)];
      const int last = i < per && r < rows ? min(r / p.group + p.off, p.Skv - 1) : -1;  // the row's last visible key
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float x = e & 1 ? T::hi(w[i][e >> 1]) : T::lo(w[i][e >> 1]);
        const float pr = __builtin_amdgcn_exp2f(__builtin_fmaf(x, kF16 ? kLog2e / 8.f : kLog2e, nlse));  // fp16 logits are kept times 8
        const int j = j0 + e;
        const float v = j >= 0 && j <= last ? pr : 0.f;  // hidden, or outside the row (what is kept there is not defined)
        sum[e] += v;
        if (SQ) sq[e] = __builtin_fmaf(v, v, sq[e]);
      }
    }
  };
  if constexpr (!WIDE) {
    if (per <= 1)
      rows_of_wave(std::integral_constant<int, 1>{});
    else if (per <= 3)
      rows_of_wave(std::integral_constant<int, 3>{});
    else
      rows_of_wave(std::integral_constant<int, 8>{});
  } else if (per <= 12) {
    rows_of_wave(std::integral_constant<int, 12>{});
  } else {
    rows_of_wave(std::integral_constant<int, kRows / 4>{});
  }
#pragma unroll
  for (int hf = 0; hf < 2; ++hf) {
    *reinterpret_cast<float4v*>(&s_sum[wave][k0 + 4 * hf]) = float4v{sum[4 * hf], sum[4 * hf + 1], sum[4 * hf + 2], sum[4 * hf + 3]};
    if constexpr (SQ) *reinterpret_cast<float4v*>(&s_sq[wave][k0 + 4 * hf]) = float4v{sq[4 * hf], sq[4 * hf + 1], sq[4 * hf + 2], sq[4 * hf + 3]};
  }
  __syncthreads();
  float tot[KT / 256];
#pragma unroll
  for (int i = 0; i < KT / 256; ++i) {
    const int k = t + 256 * i;
    tot[i] = ((s_sum[0][k] + s_sum[1][k]) + (s_sum[2][k] + s_sum[3][k])) / (float)p.group;
  }
  if (st.pool) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < KT / 256; ++i) s_sum[0][t + 256 * i] = tot[i];
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < KT / 256; ++i) {
    const int k = t + 256 * i, j = tile0 * kAttnBN + k;
    if (j < 0 || j >= p.Skv) continue;
    if (st.pool) {
      if (k < 32 || k >= KT - 32) continue;
      float s = 0.f;
      for (int u = -(st.pool / 2); u <= st.pool / 2; ++u) s += s_sum[0][k + u];
      tot[i] = s / (float)st.pool;
    }
    st.colsum[(int64_t)bh * p.Skv + j] = tot[i];
    if constexpr (SQ) st.colsumsq[(int64_t)bh * p.Skv + j] = (s_sq[0][k] + s_sq[1][k]) + (s_sq[2][k] + s_sq[3][k]);
  }
}

}  // namespace

// `stats`: column sums of the rows wanted (plan.logit_tiles > 0), else null
hipError_t launch_attn_split(const AttnKernelParams& p0, const SplitPlan& plan, char* ws, const SplitStats* stats, int D, bool bf16, bool causal,
                             bool emu, int kf, hipStream_t s) {
  AttnKernelParams p = p0;
  p.pair_order = p.two_blocks = p.head_major = 0;
  p.part = reinterpret_cast<float*>(ws);
  p.chunk_tiles = plan.chunk_tiles;
  p.nitems = plan.items;
  p.part_waves = plan.part_waves;
  if (stats) {
    p.logits = reinterpret_cast<uint16_t*>(ws + plan.logits_at);
    p.logit_tiles = plan.logit_tiles;
  }
  std::copy(plan.list, plan.list + plan.items, p.items);
  std::copy(plan.first_item, plan.first_item + plan.nblocks, p.first_item);
  if (!causal) p.off = p.Skv;
  const int64_t pairs = (int64_t)p.B * (p.H / p.group);
  const unsigned grid = (unsigned)(pairs * plan.items);
  // what a workgroup lacks to more than half of a CU's LDS
  const unsigned pad = plan.one_per_cu ? 88 * 1024 - 4 * kAttnBN * 2 * D : 0;
  hipError_t e = bf16 ? launch_attn_split_bf16(p, D, emu, kf, grid, pad, s) : launch_attn_split_f16(p, D, emu, kf, grid, pad, s);
  const int nshared = plan.nblocks - plan.first_shared;
  if (e != hipSuccess || (nshared == 0 && !stats)) return e;
  const int64_t ncomb = pairs * nshared * plan.part_waves * (D / 32);
  if (stats) {
    // (with a window the outputs of workgroup c end half a tile short of its keys)
    const int step = stat_step(stats->pool) * kAttnBN;
    const int64_t ncol = pairs * ((p.Skv + (stats->pool ? kAttnBN / 2 : 0) + step - 1) / step);
    const dim3 g((unsigned)(ncol + ncomb)), blk(256);
    const bool wide = (int64_t)p.Sq * p.group > 32;
#define FT_CASE(T, DD, SQ)                                                                                               \
  {                                                                                                                      \
    if (wide) hipLaunchKernelGGL((split_stats_kernel<T, DD, SQ, true>), g, blk, 0, s, p, *stats, (int)ncol);             \
    else hipLaunchKernelGGL((split_stats_kernel<T, DD, SQ, false>), g, blk, 0, s, p, *stats, (int)ncol);                 \
  }
    if (stats->colsumsq) {
      if (D == 128 && bf16) FT_CASE(BF16, 128, true)
      else if (D == 128) FT_CASE(F16, 128, true)
      else if (bf16) FT_CASE(BF16, 64, true)
      else FT_CASE(F16, 64, true)
    } else {
      if (D == 128 && bf16) FT_CASE(BF16, 128, false)
      else if (D == 128) FT_CASE(F16, 128, false)
      else if (bf16) FT_CASE(BF16, 64, false)
      else FT_CASE(F16, 64, false)
    }
#undef FT_CASE
    return hipGetLastError();
  }
  // Up to kSplitStatRows rows: as in the folds beside the column sums, whose rows are the same bit for bit.  More of them, up to five
  // shares of a block: two pieces a wave, four shares a round (B1 H32/8 Sq501 Skv5760, four shares, 7.9 -> 6.2 us; two pieces with
  // eight a round 7.1, four pieces 6.5; soft-capped Sq777 Skv3000, five shares, 12.5 -> 12.3; six to eight shares 4.35..4.9 against
  // 4.28..5.1, sixteen 4.7 against 5.4, thirty-one 5.8 against 7.7).
  const int64_t rows = (int64_t)p.Sq * p.group;
  const int most = (std::min<int64_t>(p.Skv, (rows - 1) / p.group + 1 + p.off) + kAttnBN - 1) / kAttnBN;
  const bool few = rows <= 32, two = rows > kSplitStatRows && most <= 5 * plan.chunk_tiles;
  const dim3 cgrid((unsigned)(two ? (ncomb + 1) / 2 : ncomb)), cblk(256);
#define FT_CASE(T, DD)                                                                                                       \
  {                                                                                                                          \
    if (few) hipLaunchKernelGGL((attn_combine_kernel<T, DD, 1, true>), cgrid, cblk, 0, s, p, plan.first_shared);             \
    else if (two) hipLaunchKernelGGL((attn_combine_kernel<T, DD, 2, false>), cgrid, cblk, 0, s, p, plan.first_shared);       \
    else hipLaunchKernelGGL((attn_combine_kernel<T, DD, 1, false>), cgrid, cblk, 0, s, p, plan.first_shared);                \
  }
  if (D == 128 && bf16) FT_CASE(BF16, 128)
  else if (D == 128) FT_CASE(F16, 128)
  else if (bf16) FT_CASE(BF16, 64)
  else FT_CASE(F16, 64)
#undef FT_CASE
  return hipGetLastError();
}

}  // namespace ft
