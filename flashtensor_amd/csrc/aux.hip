// Small epilogue kernels: heavy-hitter selection (top-k of a per-key score row) and materialisation of
// the seeded KeyFormer noise tensor.  Neither exists in the reference: its H2O case ends at the score
// (cases/kernels/h2o.py:34-38) and its KeyFormer case receives the noise as an input (kf.py:48).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "device_common.hpp"
#include "noise.h"

namespace ft {

// One workgroup of NT threads sorts one row: (score, index) pairs packed into 64-bit keys whose unsigned
// order is "score descending, index ascending", bitonic network over N = NT E keys, first k indices written
// out.  Thread t keeps keys t E .. t E + E - 1 in registers, so a compare-exchange at distance < E stays inside
// the thread, one at distance < 64 E is a lane exchange inside the wave (no barrier), and only the few
// steps at distance >= 64 E go through LDS (3 with 256 threads, 6 with 512) instead of one barrier per
// network step.  E <= 16 keeps the fully unrolled network's keys in registers.

__device__ __forceinline__ uint32_t float_order_desc(float x) {
  uint32_t u = __builtin_bit_cast(uint32_t, x);
  u = (u & 0x80000000u) ? ~u : (u | 0x80000000u);  // ascending unsigned order == ascending float order
  return ~u;                                       // flipped: larger scores first
}

// Value of lane l ^ M for a compile-time M < 64, without the LDS crossbar a generic shuffle goes through (the sort is
// a chain of ~60 dependent exchanges per row, so their latency is its run time): quad permutes for 1 and 2, half-row
// mirror + quad reversal for 4 ((l ^ 7) ^ 3), a rotation by half a row for 8, v_permlane16_swap / v_permlane32_swap
// for 16 and 32.
template <int M>
__device__ __forceinline__ uint32_t lane_xor_u32(uint32_t v) {
#if defined(__HIP_DEVICE_COMPILE__)
  static_assert(M == 1 || M == 2 || M == 4 || M == 8 || M == 16 || M == 32, "one bit of the lane index");
  const int x = (int)v;
  if constexpr (M == 1) return (uint32_t)__builtin_amdgcn_update_dpp(x, x, 0xB1, 0xF, 0xF, false);  // quad_perm [1,0,3,2]
  if constexpr (M == 2) return (uint32_t)__builtin_amdgcn_update_dpp(x, x, 0x4E, 0xF, 0xF, false);  // quad_perm [2,3,0,1]
  if constexpr (M == 4) {
    const int h = __builtin_amdgcn_update_dpp(x, x, 0x141, 0xF, 0xF, false);                         // row_half_mirror
    return (uint32_t)__builtin_amdgcn_update_dpp(h, h, 0x1B, 0xF, 0xF, false);                       // quad_perm [3,2,1,0]
  }
  if constexpr (M == 8) return (uint32_t)__builtin_amdgcn_update_dpp(x, x, 0x128, 0xF, 0xF, false);  // row_ror:8
  if constexpr (M == 16) {
    const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);  // {rows 0,0,2,2}, {rows 1,1,3,3}
    return (threadIdx.x & 16) ? (uint32_t)r[0] : (uint32_t)r[1];
  }
  if constexpr (M == 32) {
    const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);  // {lower half twice}, {upper half twice}
    return (threadIdx.x & 32) ? (uint32_t)r[0] : (uint32_t)r[1];
  }
#endif
  return v;
}

template <int M>
__device__ __forceinline__ uint64_t lane_xor_u64(uint64_t v) {
  const uint32_t lo = lane_xor_u32<M>((uint32_t)v), hi = lane_xor_u32<M>((uint32_t)(v >> 32));
  return ((uint64_t)hi << 32) | lo;
}

// one compare-exchange step of the bitonic network at distance STRIDE inside runs of SIZE keys
template <int E, int NT, int SIZE, int STRIDE>
__device__ __forceinline__ void bitonic_step(uint64_t (&key)[E], uint64_t* xch, int t) {
  if constexpr (STRIDE < E) {
#pragma unroll
    for (int e = 0; e < E; ++e) {
      if ((e & STRIDE) == 0) {
        const bool up = ((t * E + e) & SIZE) == 0;
        const uint64_t a = key[e], b = key[e | STRIDE];
        const bool swap = (a > b) == up;
        key[e] = swap ? b : a;
        key[e | STRIDE] = swap ? a : b;
      }
    }
  } else {
    constexpr int M = STRIDE / E;  // partner thread t ^ M holds the partner of every key of this thread
    const bool lower = (t & M) == 0;
    if constexpr (M >= 64) {
#pragma unroll
      for (int e = 0; e < E; ++e) xch[e * NT + t] = key[e];
      __syncthreads();
    }
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const uint64_t a = key[e];
      uint64_t b;
      if constexpr (M >= 64)
        b = xch[e * NT + (t ^ M)];
      else
        b = lane_xor_u64<M>(a);
      const bool up = ((t * E + e) & SIZE) == 0;
      const bool want_min = lower == up;
      key[e] = ((a < b) == want_min) ? a : b;
    }
    if constexpr (M >= 64) __syncthreads();
  }
}
template <int E, int NT, int SIZE, int STRIDE>
__device__ __forceinline__ void bitonic_merge(uint64_t (&key)[E], uint64_t* xch, int t) {
  bitonic_step<E, NT, SIZE, STRIDE>(key, xch, t);
  if constexpr (STRIDE > 1) bitonic_merge<E, NT, SIZE, STRIDE / 2>(key, xch, t);
}
template <int E, int NT, int SIZE>
__device__ __forceinline__ void bitonic_sort(uint64_t (&key)[E], uint64_t* xch, int t) {
  bitonic_merge<E, NT, SIZE, SIZE / 2>(key, xch, t);
  if constexpr (SIZE < E * NT) bitonic_sort<E, NT, SIZE * 2>(key, xch, t);
}

template <int E, int NT>
__global__ void __launch_bounds__(NT) topk_kernel(const float* __restrict__ score, int S, int k, int64_t* __restrict__ idx) {
  constexpr int N = NT * E;
  __shared__ uint64_t xch[N];  // slot-major: key e of thread t at [e * NT + t]
  const int t = threadIdx.x;
  const float* row = score + (int64_t)blockIdx.x * S;
  uint64_t key[E];
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int i = t * E + e;
    key[e] = i < S ? (((uint64_t)float_order_desc(row[i]) << 32) | (uint32_t)i) : ~0ull;  // padding sorts last
  }
  bitonic_sort<E, NT, 2>(key, xch, t);
  int64_t* out = idx + (int64_t)blockIdx.x * k;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int i = t * E + e;
    if (i < k) out[i] = (int64_t)(uint32_t)key[e];
  }
}

// Rows of which at most one of the NW equal runs is wanted (k <= 64 E; k = S / 8 is the usual one): every wave sorts a run
// of 64 E keys with lane exchanges alone, then pairs of runs are merged down to the 64 E first keys of both (the smaller of
// key i of one and key 64 E - 1 - i of the other, a bitonic sequence, and one merge pass), log2 NW levels through LDS with
// two barriers each, half of the waves dropping out at every level.  The network over the whole row has two barriers for
// every step across waves and works on all keys to the end (k = S / 8 of 32 rows, per call: S = 512 7.5 -> 4.6 us, 1024
// 7.3 -> 4.9: bound by the chain of compare-exchanges of one CU, which is why longer rows go to topk_select_kernel).
template <int E, int NW>
__global__ void __launch_bounds__(64 * NW) topk_runs_kernel(const float* __restrict__ score, int S, int k, int64_t* __restrict__ idx) {
  constexpr int R = 64 * E;
  __shared__ uint64_t run[NW / 2][R];
  const int lane = lane_id(), wave = wave_id();
  const float* row = score + (int64_t)blockIdx.x * S;
  uint64_t key[E];
#pragma unroll
  for (int e = 0; e < E; ++e) {  // any slot will do: the index is part of the key
    const int i = wave * R + e * 64 + lane;
    key[e] = i < S ? (((uint64_t)float_order_desc(row[i]) << 32) | (uint32_t)i) : ~0ull;  // padding sorts last
  }
  bitonic_sort<E, 64, 2>(key, nullptr, lane);
#pragma unroll
  for (int half = NW / 2; half > 0; half >>= 1) {
    if (wave >= half && wave < 2 * half) {
#pragma unroll
      for (int e = 0; e < E; ++e) run[wave - half][lane * E + e] = key[e];
    }
    __syncthreads();
    if (wave < half) {
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const uint64_t other = run[wave][R - 1 - (lane * E + e)];
        key[e] = other < key[e] ? other : key[e];
      }
      bitonic_merge<E, 64, R, R / 2>(key, nullptr, lane);
    }
    if (half > 1) __syncthreads();  // this level's runs have been read
  }
  if (wave != 0) return;
  int64_t* out = idx + (int64_t)blockIdx.x * k;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int i = lane * E + e;
    if (i < k) out[i] = (int64_t)(uint32_t)key[e];
  }
}

// The k first entries of a row by selection, then a sort of those alone: one workgroup per row, whose (score, index) words it
// holds in registers, E per thread (E = 0: reads the row again in every pass, in its own order).
//   1. The word of rank k, by its digits from the top, 11 bits at a time: a histogram in LDS of the entries that have the
//      digits found so far, a prefix sum over its bins, and the bin in which rank k lies.  It ends as soon as that bin is wanted
//      whole, after two or three passes for distinct scores; ties go on into the index, whose smallest values make the cut.
//   2. The entries up to that word go to LDS in any order, and a bitonic network over NT W >= k keys ranks them.
// The same answers as the register sort, ties and NaNs included (a NaN of positive sign has the largest order key and sorts
// first, as in torch.topk).
// Bound by latency: some ten barriers, the counting (64 lanes that hit one bin take 64 turns) and the sort's chain.  k = S / 8 of 32
// rows, per call, scores with and without noise, against sorted runs and (S > 8192) a selection by bytes whose bins one thread
// walked: S = 2048 8.3 -> 6.7, 4096 16.3 -> 8.9, 8192 34.9 -> 14, 16384 75..89 -> 25, 65536 212..251 -> 86..95.  Scores in
// their own order instead of 0.618 of the row apart: falling ones 8.7, 11.6, 19.3.  First the leading bits that all keys share, to
// begin below them, saved less than that extra barrier.
__device__ __forceinline__ uint32_t wave_prefix_sum(uint32_t v) {
  int x = (int)v;
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xF, 0xF, true);   // row_shr:1, 2, 4, 8
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xF, 0xF, true);
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xF, 0xF, true);
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xF, 0xF, true);
  x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xA, 0xF, false);  // the last lane of a row to the next one: rows 1 and 3
  x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xC, 0xF, false);  // lane 31 to the upper half
  return (uint32_t)x;
}

constexpr int kTopkSelectMax = 16384;  // 128 KB of LDS for the winners: k = S / 8 up to S = 131072

template <int NT, int E, int W>
__global__ void __launch_bounds__(NT) topk_select_kernel(const float* __restrict__ score, int S, int k, int64_t* __restrict__ idx) {
  constexpr int NW = NT / 64, kBins = 2048, kPer = kBins / NT, kAhead = E ? E : 8, kN = NT * kAhead;
  __shared__ uint64_t win[E > 2 * W ? NT * E / 2 : NT * W];
  __shared__ __align__(16) uint32_t hist[kBins];
  __shared__ uint32_t wave_sum[NW];
  __shared__ uint32_t s_digit, s_before, s_count, s_slot;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const float* row = score + (int64_t)blockIdx.x * S;
  uint32_t key[kAhead];
  auto load = [&](uint32_t i0) __attribute__((always_inline)) {
#pragma unroll
    for (int e = 0; e < kAhead; ++e) key[e] = float_order_desc(row[min(i0 + e * NT + t, S - 1u)]);
  };
  // E > 0: neighbouring scores are often alike, and 64 lanes that count in one bin wait for each other: the lanes of a wave
  // take entries 0.618 of the row apart (an odd step: each one once, no two lanes in a bank).
  constexpr uint32_t kStep = (uint32_t)(kN * 0.618) | 1;
  auto index = [&](uint32_t i0, int e) __attribute__((always_inline)) { return E ? (e * NT + t) * kStep % kN : i0 + e * NT + t; };
  if (E) {
    load(0);
    uint32_t* all = reinterpret_cast<uint32_t*>(win);
#pragma unroll
    for (int e = 0; e < kAhead; ++e) all[e * NT + t] = key[e];
    __syncthreads();
#pragma unroll
    for (int e = 0; e < kAhead; ++e) key[e] = all[index(0, e)];
  }
#pragma unroll
  for (int b = 0; b < kPer; ++b) hist[t * kPer + b] = 0;
  if (t == 0) s_slot = 0;
  __syncthreads();

  // ---- 1. the word of rank k
  int ks = 32;  // bits of the key that are open still, and of the index
  int is = S <= 1 << 21 ? 21 : 32;
  uint32_t T = 0, I = 0;        // the others
  uint32_t want = (uint32_t)k;  // rank among the entries that have these
  while (true) {
    const bool by_key = ks > 0;
    const int bits = by_key ? min(11, ks) : is == 10 ? 10 : 11, next = (by_key ? ks : is) - bits;
    const uint32_t mask = (1u << bits) - 1;
    for (int64_t i0 = 0; i0 < S; i0 += kAhead * NT) {
      if (!E) load((uint32_t)i0);
#pragma unroll
      for (int e = 0; e < kAhead; ++e) {
        const uint32_t i = index((uint32_t)i0, e);
        const bool open = by_key ? ks == 32 || key[e] >> ks == T : key[e] == T && (is == 32 || i >> is == I);
        const bool on = open && i < (uint32_t)S;
        const uint32_t digit = (by_key ? key[e] : i) >> next & mask;
        if (E == 0) {  // the wave's first digit at once, the others one by one (k = S / 8, falling scores: 16384 32.5 -> 24.6 us)
          const uint64_t m = __ballot(on);
          if (m == 0) continue;
          const int lead = __builtin_ctzll(m);
          const uint32_t d0 = __builtin_amdgcn_readlane(digit, lead);
          const uint64_t same = __ballot(on && digit == d0);
          if (lane == lead) atomicAdd(&hist[d0], (uint32_t)__popcll(same));
          if (on && digit != d0) atomicAdd(&hist[digit], 1u);
        } else if (on) {
          atomicAdd(&hist[digit], 1u);
        }
      }
    }
    __syncthreads();
    uint32_t h[kPer], sum = 0;
#pragma unroll
    for (int b = 0; b < kPer; ++b) {
      h[b] = hist[t * kPer + b];
      hist[t * kPer + b] = 0;
      sum += h[b];
    }
    const uint32_t upto = wave_prefix_sum(sum);
    if (lane == 63) wave_sum[wave] = upto;
    __syncthreads();
    uint32_t cum = upto - sum;
#pragma unroll
    for (int w = 0; w < NW; ++w) cum += w < wave ? wave_sum[w] : 0;
    if (cum < want && want <= cum + sum) {
#pragma unroll
      for (int b = 0; b < kPer; ++b) {
        if (cum < want && want <= cum + h[b]) {
          s_digit = t * kPer + b;
          s_before = cum;
          s_count = h[b];
        }
        cum += h[b];
      }
    }
    __syncthreads();
    want -= s_before;
    if (by_key) {
      T = T << bits | s_digit;
      ks = next;
    } else {
      I = I << bits | s_digit;
      is = next;
    }
    if (s_count == want || is == 0) break;  // (at the index's last digit the count is 1)
  }

  // ---- 2. the winners, and their order
  if (ks > 0 || is == (S <= 1 << 21 ? 21 : 32)) {  // (the key decided)
    is = 0;
    I = ~0u;
  }
  for (int64_t i0 = 0; i0 < S; i0 += kAhead * NT) {
    if (!E) load((uint32_t)i0);
    uint64_t in[kAhead];
    uint32_t total = 0, slot = 0;
#pragma unroll
    for (int e = 0; e < kAhead; ++e) {
      const uint32_t i = index((uint32_t)i0, e), top = key[e] >> ks;
      in[e] = __ballot(i < (uint32_t)S && (top < T || (top == T && i >> is <= I)));
      total += (uint32_t)__popcll(in[e]);
    }
    if (lane == 0 && total) slot = atomicAdd(&s_slot, total);
    slot = __builtin_amdgcn_readfirstlane(slot);
#pragma unroll
    for (int e = 0; e < kAhead; ++e) {
      if (in[e] >> lane & 1) win[slot + (uint32_t)__popcll(in[e] & ((1ull << lane) - 1ull))] = (uint64_t)key[e] << 32 | index((uint32_t)i0, e);
      slot += (uint32_t)__popcll(in[e]);
    }
  }
  for (int i = k + t; i < NT * W; i += NT) win[i] = ~0ull;  // padding sorts last
  __syncthreads();
  uint64_t best[W];
#pragma unroll
  for (int e = 0; e < W; ++e) best[e] = win[e * NT + t];  // (the slots that this thread's keys take in the network's exchanges)
  bitonic_sort<W, NT, 2>(best, win, t);
  int64_t* out = idx + (int64_t)blockIdx.x * k;
#pragma unroll
  for (int e = 0; e < W; ++e) {
    const int i = t * W + e;
    if (i < k) out[i] = (int64_t)(uint32_t)best[e];
  }
}

hipError_t launch_topk(const float* score, int64_t rows, int S, int k, int64_t* idx, hipStream_t s) {
  const dim3 grid((unsigned)rows);
  // Runs where they are two barriers a level and little else (k = S / 8 of 32 rows, S = 1024: 4.8 us, selection 5.7).  Selection with
  // S / 8 threads above (figures at the kernel).  The network over the whole row where most of it is wanted (k = 3 S / 4: 2048 9.8,
  // 4096 20, 8192 40; selection at k = S / 2 takes 10.4..11, 15 and 26, so it has S <= 2048 up to a quarter only), or it is short.
#define FT_RUNS(MAX_S, E, NW)                                                                                    \
  if (S <= MAX_S && k <= 64 * E) {                                                                               \
    hipLaunchKernelGGL((topk_runs_kernel<E, NW>), grid, dim3(64 * NW), 0, s, score, S, k, idx);                  \
    return hipGetLastError();                                                                                    \
  }
#define FT_SELECT(MAX_S, NT, E, W)                                                                               \
  if (S <= MAX_S && k <= NT * W) {                                                                               \
    hipLaunchKernelGGL((topk_select_kernel<NT, E, W>), grid, dim3(NT), 0, s, score, S, k, idx);                  \
    return hipGetLastError();                                                                                    \
  }
  FT_RUNS(512, 1, 8) FT_RUNS(1024, 2, 8)
  if (S > 8192) {
    if (k > kTopkSelectMax) return hipErrorInvalidValue;
    FT_SELECT(INT32_MAX, 1024, 0, 1) FT_SELECT(INT32_MAX, 1024, 0, 2) FT_SELECT(INT32_MAX, 1024, 0, 4)
    FT_SELECT(INT32_MAX, 1024, 0, 8) FT_SELECT(INT32_MAX, 1024, 0, 16)
  } else if (S > 4096) {
    FT_SELECT(8192, 1024, 8, 1) FT_SELECT(8192, 1024, 8, 2) FT_SELECT(8192, 1024, 8, 4)
  } else if (S > 2048) {
    FT_SELECT(4096, 512, 8, 1) FT_SELECT(4096, 512, 8, 2) FT_SELECT(4096, 512, 8, 4)
  } else if (S > 1024) {
    FT_SELECT(2048, 256, 8, 1) FT_SELECT(2048, 256, 8, 2)
  } else if (S > 512) {
    FT_SELECT(1024, 256, 4, 1)
  }
#undef FT_RUNS
#undef FT_SELECT
  if (S <= 512)
    hipLaunchKernelGGL((topk_kernel<2, 256>), grid, dim3(256), 0, s, score, S, k, idx);
  else if (S <= 1024)
    hipLaunchKernelGGL((topk_kernel<4, 256>), grid, dim3(256), 0, s, score, S, k, idx);
  else if (S <= 2048)  // more threads with fewer keys each beat fewer, fuller ones: 10.9 vs 12.9 us (8 keys x 256)
    hipLaunchKernelGGL((topk_kernel<4, 512>), grid, dim3(512), 0, s, score, S, k, idx);
  else if (S <= 4096)  // 21.3 vs 25.8 us (16 keys x 256)
    hipLaunchKernelGGL((topk_kernel<8, 512>), grid, dim3(512), 0, s, score, S, k, idx);
  else
    hipLaunchKernelGGL((topk_kernel<16, 512>), grid, dim3(512), 0, s, score, S, k, idx);
  return hipGetLastError();
}

__global__ void __launch_bounds__(256) noise_fill_kernel(float* __restrict__ dst, int Sq, int Skv, uint64_t seed) {
  const int bh = blockIdx.z;
  const int i = blockIdx.y;
  const NoiseKeys nk = noise_keys(seed, (uint32_t)bh);
  const uint32_t a_i = noise_row(nk, (uint32_t)i);
  float* row = dst + ((int64_t)bh * Sq + i) * Skv;
  for (int j = blockIdx.x * blockDim.x + threadIdx.x; j < Skv; j += gridDim.x * blockDim.x) {
    const float u = noise_uniform(a_i, noise_col(nk, (uint32_t)j));
    row[j] = -0.6931471805599453f * __builtin_amdgcn_logf(u);
  }
}

hipError_t launch_noise_fill(float* dst, int B, int H, int Sq, int Skv, uint64_t seed, hipStream_t s) {
  if ((int64_t)B * H > 65535 || Sq > 65535) return hipErrorInvalidValue;
  dim3 grid((unsigned)((Skv + 1023) / 1024 < 1 ? 1 : (Skv + 1023) / 1024), (unsigned)Sq, (unsigned)(B * H));
  hipLaunchKernelGGL(noise_fill_kernel, grid, dim3(256), 0, s, dst, Sq, Skv, seed);
  return hipGetLastError();
}

// Stride-1 window mean along rows of length S with kernel / 2 zeros on both sides, divisor = kernel: the
// SnapKV smoothing of the per-key scores, F.avg_pool1d(score, kernel, padding = kernel // 2, stride = 1)
// (cases/kernels/snapkv.py:39).  The window is summed left to right like the library routine.
__global__ void __launch_bounds__(256) avgpool1d_kernel(const float* __restrict__ src, float* __restrict__ dst, int S, int kernel) {
  const int64_t row = blockIdx.y;
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= S) return;
  const float* r = src + row * S;
  const int pad = kernel / 2;
  float acc = 0.f;
  for (int t = -pad; t <= pad; ++t) {
    const int jj = j + t;
    if (jj >= 0 && jj < S) acc += r[jj];
  }
  dst[row * S + j] = acc / (float)kernel;
}

hipError_t launch_avgpool1d(const float* src, int64_t rows, int S, int kernel, float* dst, hipStream_t s) {
  if (rows > 65535) return hipErrorInvalidValue;
  dim3 grid((unsigned)((S + 255) / 256), (unsigned)rows);
  hipLaunchKernelGGL(avgpool1d_kernel, grid, dim3(256), 0, s, src, dst, S, kernel);
  return hipGetLastError();
}

// Mean over the `group` consecutive rows of each group: src [groups, group, S] -> dst [groups, S]
// (grouped-query H2O score, cases/attn_h2o.py:42-47; the mean over heads commutes with the sum over rows).
__global__ void __launch_bounds__(256) group_mean_kernel(const float* __restrict__ src, float* __restrict__ dst, int S, int group) {
  const int64_t grp = blockIdx.y;
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= S) return;
  const float* r = src + grp * group * S + j;
  float acc = 0.f;
  for (int t = 0; t < group; ++t) acc += r[(int64_t)t * S];
  dst[grp * S + j] = acc / (float)group;
}

hipError_t launch_group_mean(const float* src, int64_t groups, int group, int S, float* dst, hipStream_t s) {
  if (groups > 65535) return hipErrorInvalidValue;
  dim3 grid((unsigned)((S + 255) / 256), (unsigned)groups);
  hipLaunchKernelGGL(group_mean_kernel, grid, dim3(256), 0, s, src, dst, S, group);
  return hipGetLastError();
}

}  // namespace ft
