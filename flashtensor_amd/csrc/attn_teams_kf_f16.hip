// attn_split.hpp's KeyFormer form with two teams of waves, instantiated for f16, head sizes 64 and 128.
#include "attn_split.hpp"

namespace ft {
hipError_t launch_attn_teams_kf_f16(const AttnKernelParams& p, int D, int kf, unsigned grid, hipStream_t s) {
  return D == 128 ? launch_teams_kf_td<F16, 128>(p, kf, grid, s) : launch_teams_kf_td<F16, 64>(p, kf, grid, s);
}
}  // namespace ft
