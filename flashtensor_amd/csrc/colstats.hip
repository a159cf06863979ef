// Dispatcher of the column-statistics pass (colstats_kernel.hpp) and its 128-key instantiations; colstats_{narrow,teams}.hip hold
// the 64-key ones.
#include <cstdlib>

#include "colstats_kernel.hpp"

namespace ft {

hipError_t launch_colstats_narrow(const ColstatsKernelParams& p, int D, bool bf16, bool causal, int mode, hipStream_t s);
hipError_t launch_colstats_teams(const ColstatsKernelParams& p, int D, bool bf16, bool causal, int mode, hipStream_t s);

// Test hook: FT_COLSTATS_KEYS=1 or 2 in the environment forces 64 or 128 keys per workgroup, 1t 64 and two teams of waves.
enum { kFormAuto = 0, kFormNarrow = 1, kFormWide = 2, kFormTeams = 3 };
static int form_override() {
  const char* e = getenv("FT_COLSTATS_KEYS");
  if (!e || (e[0] != '1' && e[0] != '2')) return kFormAuto;
  return e[0] == '2' ? kFormWide : e[1] == 't' ? kFormTeams : kFormNarrow;
}

template <typename T, int D>
static hipError_t launch_td(const ColstatsKernelParams& p, bool causal, bool emu, int mode, hipStream_t s) {
#define FT_CASE(C, E, M) \
  if (causal == C && emu == E && mode == M) return launch_colstats_one<T, D, C, E, M, 2>(p, s);
#define FT_MODES(C, E)                                                                                       \
  FT_CASE(C, E, kStatSum) FT_CASE(C, E, kStatSumPool) FT_CASE(C, E, kStatSumSq) FT_CASE(C, E, kStatKfTensor) FT_CASE(C, E, kStatKfSeeded) \
  FT_CASE(C, E, kStatCormRule) FT_CASE(C, E, kStatCormTensor)
  FT_MODES(true, true) FT_MODES(true, false) FT_MODES(false, true) FT_MODES(false, false)
  if constexpr (std::is_same<T, F16>::value) {  // packed KeyFormer modes: fp16 with reference rounding only
    if (emu) {
      FT_CASE(true, true, kStatKfSeededTau1) FT_CASE(false, true, kStatKfSeededTau1)
      FT_CASE(true, true, kStatKfSeededFast) FT_CASE(false, true, kStatKfSeededFast)
    }
  }
#undef FT_MODES
#undef FT_CASE
  return hipErrorInvalidValue;
}

hipError_t launch_colstats(const ColstatsKernelParams& p, int D, bool bf16, bool causal, bool emu, int mode, hipStream_t s) {
  const bool tensor = mode == kStatKfTensor || mode == kStatCormTensor;
  const int64_t wgs = (int64_t)p.B * p.H * ((p.Skv + 127) / 128), cus = device_cu_count();
  if (tensor && emu) {
    // Two teams of waves on 128 keys where a lane's loads of the tensor, one tile ahead, are what a tile waits for: twice the
    // loads in flight (keyformer calls, same process: B1 H8 S1003 83 -> 80 us, S2091 177 -> 169, H16 S2527 247 -> 227, H32 S1501
    // 166 -> 154; D64 H32 S2091 237 -> 226; even at two and a half workgroups per CU, 368 and 370 at H32 S2527)
    const int forced = form_override();
    if (forced ? forced == kFormTeams : wgs <= 9 * cus / 4) return launch_colstats_teams(p, D, bf16, causal, mode, s);
  }
  if (!tensor && emu) {
    int form = form_override();
    // 64 keys per workgroup where there are fewer than two workgroups of 128 per CU (h2o calls, same process: B1 H8 S1500
    // 49.6 -> 43.7 us, B1 H32 S1000 38.0 -> 34.7, keyformer B1 H16 S2048 101.7 -> 86.6; at two per CU the same or slower,
    // 77.4 and 78.7 at B1 H32 S2048, and at eight 62.0 and 66.7); and two teams of waves below one per CU, where a
    // workgroup of 64 keys often has its CU to itself (B1 H8 S1500 43.7 -> 41.0, S3000 76.4 -> 70.4, roco B1 H8 S2048 D64 39.4 ->
    // 37.1; at one per CU 56.3 and 56.1 at B1 H16 S2048, 34.7 and 35.3 at B1 H32 S1000, above it slower: 52.3 and 57.6 at B1 H32 S1500)
    if (!form) form = wgs < cus ? kFormTeams : wgs < 2 * cus ? kFormNarrow : kFormWide;
    if (form == kFormTeams) return launch_colstats_teams(p, D, bf16, causal, mode, s);
    if (form == kFormNarrow) return launch_colstats_narrow(p, D, bf16, causal, mode, s);
  }
  if (D == 128) return bf16 ? launch_td<BF16, 128>(p, causal, emu, mode, s) : launch_td<F16, 128>(p, causal, emu, mode, s);
  if (D == 64) return bf16 ? launch_td<BF16, 64>(p, causal, emu, mode, s) : launch_td<F16, 64>(p, causal, emu, mode, s);
  return hipErrorInvalidValue;
}

}  // namespace ft
