// Attention over few query rows and many keys (generation steps, a window of last queries, a chunk of a prompt): attn_fwd_kernel's SPLIT form, whose row blocks share their key tiles out between workgroups, and the
// plan that says when.  Instantiated by attn_split_{f16,bf16}.hip; attn_split.hip holds the plan, the dispatcher and the
// kernel that folds the shares.
//
// What bounds the unsplit form there: a row block is one workgroup that walks all of its tiles (0.9 us each where it has a CU to
// itself, D = 128), however few blocks there are.  B4 Sq1 Skv4097 with 32 query heads on 8 k/v heads: 128 workgroups of which one wave of four has
// one row, 65 tiles each, K and V staged four times over: 69 us for 67 MB.
#pragma once
#include "attn_fwd_kernel.hpp"

namespace ft {

template <typename T, int D>
hipError_t launch_split_td(const AttnKernelParams& p, bool emu, int kf, unsigned grid, unsigned lds, hipStream_t s) {
#define FT_CASE(E, K)                                                                                        \
  if (emu == E && kf == K) {                                                                                 \
    hipLaunchKernelGGL((attn_fwd_kernel<T, D, true, E, K, 4, true>), dim3(grid), dim3(256), lds, s, p);      \
    return hipGetLastError();                                                                                \
  }
  if (p.logits && emu && kf == kKfNone) {
    hipLaunchKernelGGL((attn_fwd_kernel<T, D, true, true, kKfNone, 4, true, true>), dim3(grid), dim3(256), lds, s, p);
    return hipGetLastError();
  }
  FT_CASE(true, kKfNone) FT_CASE(false, kKfNone) FT_CASE(true, kKfSoftcap) FT_CASE(false, kKfSoftcap)
#undef FT_CASE
  return hipErrorInvalidValue;
}

// Blocks of 64 rows, a workgroup of two teams for each (heaviest first).
template <typename T, int D>
hipError_t launch_teams_td(const AttnKernelParams& p, bool emu, int kf, unsigned grid, hipStream_t s) {
#define FT_CASE(E, K)                                                                                                    \
  if (emu == E && kf == K) {                                                                                             \
    hipLaunchKernelGGL((attn_fwd_kernel<T, D, true, E, K, 2, true, false, 2>), dim3(grid), dim3(256), 0, s, p);          \
    return hipGetLastError();                                                                                            \
  }
  FT_CASE(true, kKfNone) FT_CASE(false, kKfNone) FT_CASE(true, kKfSoftcap) FT_CASE(false, kKfSoftcap)
#undef FT_CASE
  return hipErrorInvalidValue;
}

// The same for KeyFormer with the reference's rounding of the logits (attn_teams_kf_{f16,bf16}.hip).
template <typename T, int D>
hipError_t launch_teams_kf_td(const AttnKernelParams& p, int kf, unsigned grid, hipStream_t s) {
#define FT_CASE(K)                                                                                                       \
  if (kf == K) {                                                                                                         \
    hipLaunchKernelGGL((attn_fwd_kernel<T, D, true, true, K, 2, true, false, 2>), dim3(grid), dim3(256), 0, s, p);       \
    return hipGetLastError();                                                                                            \
  }
  FT_CASE(kKfTensor) FT_CASE(kKfTensorLds) FT_CASE(kKfSeeded)
  if constexpr (std::is_same<T, F16>::value) {
    FT_CASE(kKfSeededTau1) FT_CASE(kKfSeededFast)
  }
#undef FT_CASE
  return hipErrorInvalidValue;
}

}  // namespace ft
