// What the forward scan kernels (ssm_scan.hip, ssm_scan_group.hip) share.
#pragma once

#include "common.h"

namespace hclsm {

// Internal mode of hclsm_ssm_block_scan_fwd: the MODEL clamps, dt = softplus(dt input) before
// its clamp, and the output multiplied by silu(gate) -- the SimplifiedSSMBlock epilogues
// (level0_ssm.py:73, :76, :103) fused into the scan.
constexpr int SCAN_BLOCK = HCLSM_SCAN_BLOCK;
struct ScanEpi {
  const void* gate;   // [batch][T][d_inner], I/O type; required in SCAN_BLOCK
  void* y_pre;        // optional: the scan output before gating (kept for the backward)
  float* ck;          // checkpointing launches only: [batch][ceil(T / 8)][16][d_inner] fp32, the state
                      // before steps 8, 16, ... (the backward's checkpoint slab; entry 0, the zero initial
                      // state, is not stored)
};

template <int MODE>
__device__ __forceinline__ float scan_dt(float v) {
  if constexpr (MODE == SCAN_BLOCK) v = softplus_f(v);
  if constexpr (MODE != HCLSM_SCAN_RAW) v = fminf(fmaxf(v, 1e-3f), 1.0f);
  return v;
}

// Forward scan with a channel's states split over the waves of a workgroup (ssm_scan_group.hip): fp32 or bf16,
// d_state a multiple of 8 from 24 to 128.  HCLSM_ERR_UNSUPPORTED where it does not apply (the caller runs the generic
// kernel).
int scan_fwd_group(int mode, const void* x, const void* dt, const float* A_log, const void* B, const void* C,
                   const float* Dskip, void* y, float* h_final, int64_t batch, int64_t T, int64_t Dn, int64_t S,
                   int dtype, hipStream_t st, ScanEpi epi);

}  // namespace hclsm
