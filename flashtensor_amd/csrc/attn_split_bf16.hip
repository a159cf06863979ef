// attn_split.hpp instantiated for bf16, head sizes 64 and 128.
#include "attn_split.hpp"

namespace ft {
hipError_t launch_attn_split_bf16(const AttnKernelParams& p, int D, bool emu, int kf, unsigned grid, unsigned lds, hipStream_t s) {
  return D == 128 ? launch_split_td<BF16, 128>(p, emu, kf, grid, lds, s) : launch_split_td<BF16, 64>(p, emu, kf, grid, lds, s);
}
hipError_t launch_attn_teams_bf16(const AttnKernelParams& p, int D, bool emu, int kf, unsigned grid, hipStream_t s) {
  return D == 128 ? launch_teams_td<BF16, 128>(p, emu, kf, grid, s) : launch_teams_td<BF16, 64>(p, emu, kf, grid, s);
}

}  // namespace ft
