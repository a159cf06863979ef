// colstats_kernel.hpp with 64 keys per workgroup: the modes with the reference's rounding of the logits.
#include "colstats_kernel.hpp"

namespace ft {

template <typename T, int D>
static hipError_t launch_narrow_td(const ColstatsKernelParams& p, bool causal, int mode, hipStream_t s) {
#define FT_CASE(M) \
  if (mode == M) return causal ? launch_colstats_one<T, D, true, true, M, 1>(p, s) : launch_colstats_one<T, D, false, true, M, 1>(p, s);
  FT_CASE(kStatSum) FT_CASE(kStatSumPool) FT_CASE(kStatSumSq) FT_CASE(kStatKfSeeded) FT_CASE(kStatCormRule)
  if constexpr (std::is_same<T, F16>::value) {
    FT_CASE(kStatKfSeededTau1) FT_CASE(kStatKfSeededFast)
  }
#undef FT_CASE
  return hipErrorInvalidValue;
}

hipError_t launch_colstats_narrow(const ColstatsKernelParams& p, int D, bool bf16, bool causal, int mode, hipStream_t s) {
  if (D == 128) return bf16 ? launch_narrow_td<BF16, 128>(p, causal, mode, s) : launch_narrow_td<F16, 128>(p, causal, mode, s);
  if (D == 64) return bf16 ? launch_narrow_td<BF16, 64>(p, causal, mode, s) : launch_narrow_td<F16, 64>(p, causal, mode, s);
  return hipErrorInvalidValue;
}

}  // namespace ft
