// What the backward scan kernels (ssm_scan_bwd.hip, ssm_scan_bwd_group.hip) share: sums across the lanes of a wave.
#pragma once

#include "common.h"

namespace hclsm {

// Value of the partner lane across bit M for the reduce-scatter steps below 16 lanes.  The partner only
// has to differ in bit M and agree in the bits above it; when every bit below M is reduced later too
// (MASK_LO == 1) the DPP mirrors are used (lane ^ 15, lane ^ 7 inside a row), else exact xor partners.
template <int M, int MASK_LO>
__device__ __forceinline__ float rs_partner(float v) {
  const int b = __float_as_int(v);
  if constexpr (M == 8) {
    return __int_as_float(MASK_LO == 1 ? __builtin_amdgcn_update_dpp(0, b, 0x140, 0xf, 0xf, true)     // row_mirror
                                       : __builtin_amdgcn_update_dpp(0, b, 0x128, 0xf, 0xf, true));   // row_ror:8
  } else if constexpr (M == 4) {
    if constexpr (MASK_LO == 1)
      return __int_as_float(__builtin_amdgcn_update_dpp(0, b, 0x141, 0xf, 0xf, true));   // row_half_mirror
    else
      return __shfl_xor(v, 4, 64);
  } else if constexpr (M == 2) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, b, 0x4e, 0xf, 0xf, true));      // quad_perm 2,3,0,1
  } else {
    static_assert(M == 1, "rs_partner: M in {1, 2, 4, 8}");
    return __int_as_float(__builtin_amdgcn_update_dpp(0, b, 0xb1, 0xf, 0xf, true));      // quad_perm 1,0,3,2
  }
}

// (lo, hi) -> lo summed over the lane pair for the lower lane, hi summed for the upper lane, where the
// pair differs in bit 5 (M == 32) or bit 4 (M == 16): one gfx950 permlane swap exchanges the halves.
template <int M>
__device__ __forceinline__ float rs_swap_sum(float lo, float hi) {
  if constexpr (M == 32) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(lo), __float_as_uint(hi), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
  } else {
    static_assert(M == 16, "rs_swap_sum: M in {16, 32}");
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(lo), __float_as_uint(hi), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
  }
}

template <int V, int MASK_LO>
struct RS {
  // Reduce-scatter V values across the lanes that differ in bits [MASK_LO, 32] of the lane id.
  // On return v[0 .. V/2^h) holds sums for value indices starting at `off` (h = halving steps).
  template <int CNT, int M>
  static __device__ __forceinline__ void step(float* v, int lane, int& off) {
    if constexpr (M >= MASK_LO) {
      if constexpr (CNT > 1) {
        const bool upper = (lane & M) != 0;
#pragma unroll
        for (int i = 0; i < CNT / 2; ++i) {
          if constexpr (M >= 16) {
            v[i] = rs_swap_sum<M>(v[i], v[i + CNT / 2]);
          } else {
            const float keep = upper ? v[i + CNT / 2] : v[i];
            const float send = upper ? v[i] : v[i + CNT / 2];
            v[i] = keep + rs_partner<M, MASK_LO>(send);
          }
        }
        if (upper) off += CNT / 2;
        step<CNT / 2, M / 2>(v, lane, off);
      } else {
        if constexpr (M >= 16) v[0] = rs_swap_sum<M>(v[0], v[0]);
        else v[0] += rs_partner<M, MASK_LO>(v[0]);
        step<1, M / 2>(v, lane, off);
      }
    }
  }
  static __device__ __forceinline__ int run(float* v, int lane) {
    int off = 0;
    step<V, 32>(v, lane, off);
    return off;
  }
};

template <int N_, int MASK_LO> struct RSCount {  // values left per lane after RS
  static constexpr int h(int cnt, int m) { return (m < MASK_LO || cnt <= 1) ? cnt : h(cnt / 2, m / 2); }
  static constexpr int value = h(N_, 32);
};

}  // namespace hclsm
