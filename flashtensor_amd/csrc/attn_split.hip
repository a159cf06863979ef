// When attention splits the keys of its row blocks (attn_split.hpp), and the kernel that folds the shares.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <functional>
#include <vector>

#include "attn_split.hpp"

namespace ft {

hipError_t launch_attn_split_f16(const AttnKernelParams& p, int D, bool emu, int kf, unsigned grid, unsigned lds, hipStream_t s);
hipError_t launch_attn_split_bf16(const AttnKernelParams& p, int D, bool emu, int kf, unsigned grid, unsigned lds, hipStream_t s);

namespace {

struct SplitShape {
  int B, H, group, Sq, Skv, D, forced, cus;
  bool causal, cap;
  bool operator==(const SplitShape& o) const {
    return B == o.B && H == o.H && group == o.group && Sq == o.Sq && Skv == o.Skv && D == o.D && forced == o.forced && cus == o.cus && causal == o.causal && cap == o.cap;
  }
};

// Microseconds by which launches are compared, from timings of this kernel and of the unsplit one at 1 to 48 tiles per
// workgroup, D = 128 (D = 64 takes 0.6 of a tile's time).  A workgroup takes 7 us for its first loads, its last stores
// and the launch, then 0.9 per tile where it has its CU to itself and 2.2 where two share one: the second wave of a
// SIMD hides little of the first one's work (soft-capped logits: 1.9 and 3.5; there it does).  Partial results are
// written at 10 MB/us and folded at 7, by a kernel that takes 5.5 us to begin with, its launch included; K and V come from HBM at 5.
constexpr double kLaunch = 7.0, kCombine = 5.5, kPartWrite = 10e6, kPartRead = 7e6, kKvBytes = 5e6;

SplitPlan make_plan(const SplitShape& a) {
  SplitPlan plan{};
  const int64_t pairs = (int64_t)a.B * (a.H / a.group), rows64 = (int64_t)a.Sq * a.group;
  if (rows64 > 128 * kSplitMaxBlocks || pairs * ((rows64 + 127) / 128) > 4 * a.cus || a.forced < 0) return plan;
  // A whole prompt (more than half as many queries as keys) keeps its blocks whole: at most a sixth is to be gained there (B1 H8 S2048:
  // 35 against 29 us), and its results are those of every launch form of the unsplit kernel, bit for bit.
  if (a.Skv < 2 * (int64_t)a.Sq && a.forced == 0) return plan;
  const int rows = (int)rows64, nMB = (rows + 127) / 128, off = a.causal ? a.Skv - a.Sq : a.Skv;
  const int cus = a.cus;
  int tiles[kSplitMaxBlocks];
  int64_t total = 0;
  for (int mb = 0; mb < nMB; ++mb) {
    tiles[mb] = (std::min(a.Skv, (std::min(mb * 128 + 128, rows) - 1) / a.group + 1 + off) + 63) / 64;
    total += tiles[mb];
  }
  const int most = tiles[nMB - 1], part_waves = std::min(4, (rows + 31) / 32);
  const double size = a.D == 128 ? 1.0 : 0.6, alone = (a.cap ? 1.9 : 0.9) * size, shared_cu = (a.cap ? 3.5 : 2.2) * size;
  const double kv_us = pairs * (double)a.Skv * a.D * 4 / kKvBytes;
  // second: tiles of the workgroup that shares a CU with the longest one, where all of them are resident at once
  // more than that: handed out in order (longest first) to the slots of an XCD as they become free
  auto rounds_us = [&](const int* len, int items) {
    const int slots = std::max(1, 2 * cus / 8);
    const int64_t per_xcd = (pairs + 7) / 8;
    std::vector<double> free_at(slots, 0.0);  // a heap whose front is the earliest
    double end = 0;
    for (int i = 0; i < items; ++i)
      for (int64_t j = 0; j < per_xcd; ++j) {
        std::pop_heap(free_at.begin(), free_at.end(), std::greater<double>());
        free_at.back() += len[i] * shared_cu;
        end = std::max(end, free_at.back());
        std::push_heap(free_at.begin(), free_at.end(), std::greater<double>());
      }
    return end;
  };
  auto kernel_us = [&](int64_t wgs, const int* len, int items, int longest, int second, double sum) {
    const double work = wgs <= cus       ? longest * alone
                        : wgs <= 2 * cus ? second * shared_cu + (longest - second) * alone
                        : len            ? rounds_us(len, items)
                                         : std::max(longest * alone, sum * shared_cu / (2.0 * cus) + 0.25 * longest * alone);
    return kLaunch + std::max(work, kv_us) + 0.25 * std::min(work, kv_us);
  };
  double best;
  int best_chunk = 0;
  {  // the unsplit form: a workgroup per 128 queries of a head
    const int nq = (a.Sq + 127) / 128;
    int64_t sum = 0;
    for (int i = 0; i < nq; ++i) sum += (std::min(a.Skv, std::min(i * 128 + 128, a.Sq) + off) + 63) / 64;
    const int64_t wgs = (int64_t)a.B * a.H * nq;
    // heavy and light blocks share a CU: the average makes up the longest block's company
    best = kernel_us(wgs, nullptr, 0, most, (int)std::max<int64_t>(0, std::min<int64_t>(most, 2 * sum / nq - most)), (double)sum * a.B * a.H);
  }
  for (int parts = 1; parts <= kSplitMaxItems; ++parts) {
    const int chunk = a.forced > 0 ? a.forced : (most + parts - 1) / parts;
    if (chunk < 1 || (parts > 1 && chunk == (most + parts - 2) / (parts - 1) && !a.forced)) continue;
    int items = 0, shared = 0, len[kSplitMaxItems];
    for (int mb = 0; mb < nMB && items <= kSplitMaxItems; ++mb) {
      const int nch = (tiles[mb] + chunk - 1) / chunk;
      for (int c = 0; c < nch && items + c < kSplitMaxItems; ++c) len[items + c] = (tiles[mb] + nch - 1) / nch;
      items += nch;
      shared += nch > 1 ? nch : 0;
    }
    if (items > kSplitMaxItems) break;
    std::sort(len, len + items, std::greater<int>());
    double us = kernel_us(items * pairs, len, items, len[0], len[std::min<int64_t>(items - 1, cus / pairs)], (double)total * pairs);
    if (shared) us += kCombine + (double)shared * pairs * std::min(rows, 128) * a.D * 4 * (1 / kPartWrite + 1 / kPartRead);
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
  return plan;
}

}  // namespace

// The plan of a shape costs some microseconds and a program calls with few shapes: each thread keeps its last ones.
const SplitPlan& split_plan(int B, int H, int group, int Sq, int Skv, int D, bool causal, bool cap) {
  struct Entry {
    SplitShape shape{};
    SplitPlan plan{};
  };
  constexpr int kEntries = 16;
  static thread_local Entry kept[kEntries];
  const SplitShape shape{B, H, group, Sq, Skv, D, attn_split_override(), device_cu_count(), causal, cap};
  Entry& e = kept[(unsigned)(B * 31 + H * 7 + group * 3 + Sq * 5 + Skv + D + cap) % kEntries];
  if (!(e.shape == shape)) e = Entry{shape, make_plan(shape)};
  return e.plan;
}

// One workgroup per (wave of 32 rows of a shared block, 32 channels), a wave per four of a lane's 16 channels: weights of
// the shares from their row maxima, then the shares' accumulators in their own register layout (every load is 1 KB
// contiguous).  Bound by the latency of its loads, so eight shares are requested at a time.
template <typename T, int D>
__global__ void __launch_bounds__(256) attn_combine_kernel(const AttnKernelParams p, int first_shared) {
  constexpr int DB = D / 32, U = 8;
  const int rows = p.Sq * p.group, Hkv = p.H / p.group;
  const int nMB = (rows + 127) / 128, nshared = nMB - first_shared;
  int i = blockIdx.x;
  const int db = i % DB;
  i /= DB;
  const int wv = i % p.part_waves;
  i /= p.part_waves;
  const int mb = first_shared + i % nshared, bh = i / nshared;
  const int lane = lane_id(), q4 = wave_id(), g = lane >> 5, n = lane & 31;
  const int row = mb * 128 + wv * 32 + n;
  if (row >= rows) return;
  const int n_end = min(p.Skv, (min(mb * 128 + 128, rows) - 1) / p.group + 1 + p.off);
  const int nch = ((n_end + kAttnBN - 1) / kAttnBN + p.chunk_tiles - 1) / p.chunk_tiles;
  const int64_t slot0 = ((int64_t)bh * p.nitems + p.first_item[mb]) * p.part_waves + wv;
  float M = -__builtin_inff(), L = 0.f;
  float4v acc = {0.f, 0.f, 0.f, 0.f};
  for (int c0 = 0; c0 < nch; c0 += U) {
    float m[U], l[U];
    float4v o[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {  // shares past the last one re-read it, with weight 0
      const SplitPartial s = split_partial(p.part, D, slot0 + (int64_t)min(c0 + u, nch - 1) * p.part_waves);
      m[u] = s.m[n];
      l[u] = s.l[n];
      o[u] = *reinterpret_cast<const float4v*>(s.o + ((db * 4 + q4) * 64 + lane) * 4);
    }
    float M1 = M;
#pragma unroll
    for (int u = 0; u < U; ++u) M1 = fmaxf(M1, m[u]);
    const float f = __builtin_amdgcn_exp2f(M - M1);  // share 0 sees every row's first key: M1 is finite
    L *= f;
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[e] *= f;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const float w = c0 + u < nch ? __builtin_amdgcn_exp2f(m[u] - M1) : 0.f;  // 0 too for a share that hides every key from the row
      L = __builtin_fmaf(w, l[u], L);
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[e] = __builtin_fmaf(w, o[u][e], acc[e]);
    }
    M = M1;
  }
  const float inv = 1.f / L;
  const int b = bh / Hkv, h = (bh % Hkv) * p.group + row % p.group, qi = row / p.group;
  uint16_t* optr = p.o + b * p.so.b + (int64_t)qi * p.so.s + h * p.so.h;
  *reinterpret_cast<uint2*>(optr + 32 * db + 8 * q4 + 4 * g) = make_uint2(T::pack2(acc[0] * inv, acc[1] * inv), T::pack2(acc[2] * inv, acc[3] * inv));
  if (db == 0 && q4 == 0 && g == 0 && p.lse) p.lse[((int64_t)b * p.H + h) * p.Sq + qi] = M + __builtin_amdgcn_logf(L);
}

hipError_t launch_attn_split(const AttnKernelParams& p0, const SplitPlan& plan, float* part, int D, bool bf16, bool causal, bool emu, int kf,
                             hipStream_t s) {
  AttnKernelParams p = p0;
  p.pair_order = p.two_blocks = p.head_major = 0;
  p.part = part;
  p.chunk_tiles = plan.chunk_tiles;
  p.nitems = plan.items;
  p.part_waves = plan.part_waves;
  std::copy(plan.list, plan.list + plan.items, p.items);
  std::copy(plan.first_item, plan.first_item + plan.nblocks, p.first_item);
  if (!causal) p.off = p.Skv;
  const int64_t pairs = (int64_t)p.B * (p.H / p.group);
  const unsigned grid = (unsigned)(pairs * plan.items);
  // what a workgroup lacks to more than half of a CU's LDS
  const unsigned pad = plan.one_per_cu ? 88 * 1024 - 4 * kAttnBN * 2 * D : 0;
  hipError_t e = bf16 ? launch_attn_split_bf16(p, D, emu, kf, grid, pad, s) : launch_attn_split_f16(p, D, emu, kf, grid, pad, s);
  if (e != hipSuccess || plan.first_shared == plan.nblocks) return e;
  const dim3 cgrid((unsigned)(pairs * (plan.nblocks - plan.first_shared) * plan.part_waves * (D / 32))), cblk(256);
  if (D == 128 && bf16) hipLaunchKernelGGL((attn_combine_kernel<BF16, 128>), cgrid, cblk, 0, s, p, plan.first_shared);
  else if (D == 128) hipLaunchKernelGGL((attn_combine_kernel<F16, 128>), cgrid, cblk, 0, s, p, plan.first_shared);
  else if (bf16) hipLaunchKernelGGL((attn_combine_kernel<BF16, 64>), cgrid, cblk, 0, s, p, plan.first_shared);
  else hipLaunchKernelGGL((attn_combine_kernel<F16, 64>), cgrid, cblk, 0, s, p, plan.first_shared);
  return hipGetLastError();
}

}  // namespace ft
