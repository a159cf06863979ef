// Dispatcher of the fused softmax attention forward: picks the instantiation of attn_fwd_kernel.hpp built by
// attn_fwd_{f16,bf16}_{d64,d128}.hip for the element type and head size of the call.
#include <hip/hip_runtime.h>

#include <atomic>
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

// Two teams of waves on blocks of 64 rows (attn_split.hpp) instead of four waves on 128: half the rows and half the chain of
// key tiles per workgroup.  Taken where the chain is the launch: with a workgroup of this form for every CU at most, from
// ten key tiles on (attention calls, same process: B1 H8 D128 S1000 21.1 -> 18.1 us, S2048 35.6 -> 29.3; D64, of whose
// workgroups a CU holds two, from five tiles on: H8 S1000 14.9 -> 12.0).  Shorter plain calls have 2 us at most to gain
// (S500 14.0 -> 12.3) and keep to the forms whose results agree bit for bit; soft-capped ones, whose waves are slow
// enough alone, take it from four tiles on (S300 13.4 -> 12.2, S500 19.4 -> 14.9, S130 9.6 -> 9.8).
// Under the causal mask, whose blocks differ in length, with more of them: D128 up to three for two CUs (H8 S3000 48 -> 40, H16 S1500
// 28.5 -> 25.8; H16 S2048, four for two, 36.6 -> 35.8 and H32 S777 17.7 -> 20.8), D64 up to two for every CU (H8 S3000 33.5 -> 27.2, B2
// H32 S500 10.7 -> 9.4) or, over more than 32 tiles, five for two (H16 S2500 31.7 -> 26.9, S3000 36 -> 38), longer ones than 48 again keeping to the bit-equal
// forms; soft-capped D128 over twelve tiles or more up to
// two for every CU (H32 S777 28.7 -> 26.0, B2 H32 S500 21.8 -> 23.4), over more than 32 five for two (H16 S2500 89 -> 81, S3000
// 97 -> 107), D64 up to thirteen for four CUs (H16 S3000 85 -> 66, H32 S1500 47 -> 37, B2 H32 S777 28.6 -> 27.4, S1000 32 -> 36).
bool use_teams(int Skv, int D, bool causal, bool cap, int64_t grid) {
  const int forced = attn_form_override();
  if (forced || attn_split_override()) return (forced & 16) != 0;
  const int64_t cus = device_cu_count();
  const int tiles = (Skv + 63) / 64;
  if (tiles <= (cap ? 3 : D == 64 ? 5 : 10)) return false;
  if (grid <= cus) return true;
  if (!causal) return false;
  if (D == 128 && !cap) return 2 * grid <= 3 * cus;
  if (D == 64 && cap) return 4 * grid <= 13 * cus;
  if (D == 64 && tiles > 48) return false;
  return (D == 64 || tiles > 11) && 2 * grid <= (tiles > 32 ? 5 : 4) * cus;
}

// KeyFormer's passes do two to four times the vector work per tile, so the chain of a block's tiles bounds launches of more
// workgroups still, and half the chain pays from two key tiles on (whole calls, same process, four waves on 128 rows against the
// teams).  Noise from a tensor, D128: B1 H8 S100 16.9 -> 15.5 us (S64 12.5 -> 14.0), S2091 165 -> 118, H16 S3543 328 -> 297, and at
// more than 3.5 workgroups for every CU slower, H32 S2091 214 -> 224; D64 H16 S2527 169 -> 146, H32 S1501 107 -> 107, S2091 166 -> 182.
// From a seed, D128: H8 S391 28.5 -> 25.0, S1003 51.8 -> 40.5, H16 S2091 109 -> 96, S2527 (2.5 for every CU) 146 -> 146 or, bf16,
// 176 -> 168, H32 S1501 92 -> 105; D64 H16 S3543 142 -> 127, H32 S2091 100 -> 95, S2527 128 -> 129.
static bool use_kf_teams(const AttnKernelParams& p, int D, int kf, int64_t grid) {
  const int forced = attn_form_override();
  if (forced) return (forced & 16) != 0;
  const int64_t cus = device_cu_count();
  if (p.Skv <= 64) return false;
  if (kf == kKfTensor || kf == kKfTensorLds) return grid <= (D == 128 ? 7 * cus / 2 : 3 * cus);
  return grid <= (D == 128 ? 5 * cus / 2 : 9 * cus / 2);
}

hipError_t launch_attn_fwd(const AttnKernelParams& p, int D, bool bf16, bool causal, bool emu, int kf, hipStream_t s) {
  const int64_t rows = (int64_t)p.Sq * p.group, grid = (rows + 63) / 64 * p.B * (p.H / p.group);
  if ((kf == kKfNone || kf == kKfSoftcap) && rows < 0x7fffffff - 64 && grid < 0x7fffffff && use_teams(p.Skv, D, causal, kf == kKfSoftcap, grid)) {
    AttnKernelParams pp = p;
    if (!causal) pp.off = p.Skv;
    // (D = 64: two workgroups per CU; see the kernel)
    pp.pair_order = causal && D == 64 && grid > device_cu_count() && grid <= 2 * device_cu_count();
    return bf16 ? launch_attn_teams_bf16(pp, D, emu, kf, (unsigned)grid, s) : launch_attn_teams_f16(pp, D, emu, kf, (unsigned)grid, s);
  }
  if (emu && (kf == kKfTensor || kf == kKfTensorLds || kf == kKfSeeded || kf == kKfSeededTau1 || kf == kKfSeededFast) && grid < 0x7fffffff && use_kf_teams(p, D, kf, grid)) {
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
