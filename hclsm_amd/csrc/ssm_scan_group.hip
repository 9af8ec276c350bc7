// Selective SSM scan forward for wide states: the states of a channel are split over the waves of a workgroup.
//
// A workgroup owns 64 channels of one sequence; wave g of it keeps states g * SG .. g * SG + SG - 1 of those channels
// in registers for the whole sequence, so every lane runs the same loop as the d_state-16 kernels of ssm_scan.hip
// however wide the state is: B_t / C_t of the wave's states are uniform (scalar loads), no state is padding, and the
// grid has d_state / SG times the waves.  Each wave leaves its part of y_t = sum_s C_s h_s in LDS; once per TC steps
// the workgroup meets at a barrier, and wave w then adds the parts of steps w, w + NG, ... in group order, applies the
// epilogue and stores them.  Two LDS buffers: one barrier per TC steps.
//
// SG = 16, bf16 I/O: the input term u B_t and its add into h run on the matrix core (v_mfma_f32_32x32x8_bf16; see
// ssm_scan_fwd_mfma_kernel for the layout).  u = dt x is split exactly into three bf16 pieces (two hold a product of
// two bf16 values; the clamped dt of the model and block modes has 24 bits), so the products are exact in fp32.  That
// holds for finite values only: a lane's column also meets the other half's channel with zero weights, and a zero piece
// of u meets B.  So in a chunk with a u or a B of the wave's states that is not finite, the products with such a value
// are formed on the VALU and the operands have 0 there; what is finite comes out the same.  (One test per chunk and a
// scalar branch per step, 89 registers, five waves per SIMD; clamping u in every step took 96 to 101 registers, 1024 x 64
// x 384, S 32, model 167 against 153 us.  A second loop for such chunks took 108 to 128 registers: 161 to 200.)
// SG = 8: multiply and FMA on the VALU (an fp32 MFMA shares the VALU's multipliers: measured 6.5 ns per 4x4x1 product
// next to a stream of FMAs, against 1.75 ns per FMA).
//
// Bound by VALU issue: 5 issue slots per state update on the matrix core (exponent multiply, exp = 2, decay multiply,
// readout FMA), 6 on the VALU.  Measured on MI355X (us per launch; before: one to four lanes per channel, states
// padded to a power of two, B / C through LDS; last: the slots at 1.75 ns each):
//   128 x 16 x 256, S 32, fp32          15.6 ->   8.7   2.7     512 x 16 x 512, S 64, fp32   80.0 -> 61.9  43.0
//   1024 x 16 x 384, S 48, bf16 block  246.3 ->  80.8  40.3     512 x 16 x 512, S 64, bf16   79.3 -> 53.9  35.9
//   1024 x 64 x 384, S 32, bf16        183.7 -> 147.5 107.5     20 x 95 x 768, S 24, bf16    59.0 -> 34.1
// Not kept: two channels per lane (1024 x 16 x 384 block 109 against 81, others equal or slower), 8-step chunks (equal),
// B / C rows by vector loads a chunk ahead (172 registers: 10.7 against 8.6 at the first shape).
#include "internal.h"
#include "scan_common.h"

namespace hclsm {

typedef short s16x4_t __attribute__((ext_vector_type(4)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));

constexpr int GRP_MAX_WAVES = 16;

// exp(v) to about an ulp: 2^p with p = v log2(e) rounded, times 1 + the rounding error of p (and of log2(e)) in
// units of ln 2.  Infinities give 0 and inf.
__device__ __forceinline__ float exp_comp(float v) {
  const float p = v * HCLSM_LOG2E;
  float lo = fmaf(v, HCLSM_LOG2E, -p);
  lo = fmaf(v, 1.925963033500e-8f, lo);          // log2(e) - (float)log2(e)
  const float e = fast_exp2(p);
  const float r = fmaf(e, lo * HCLSM_LN2, e);
  return lo == lo && e < __FLT_MAX__ ? r : e;    // v = +-inf, or overflow: e itself (0 or inf)
}

template <int DT, int MODE, int SG, int TC>
__global__ void __launch_bounds__(64 * GRP_MAX_WAVES) __attribute__((amdgpu_waves_per_eu(SG == 16 ? 5 : 4)))
ssm_scan_fwd_group_kernel(const typename Elem<DT>::T* __restrict__ x, const typename Elem<DT>::T* __restrict__ dt,
                          const float* __restrict__ A_log, const typename Elem<DT>::T* __restrict__ Bm,
                          const typename Elem<DT>::T* __restrict__ Cm, const float* __restrict__ Dskip,
                          typename Elem<DT>::T* __restrict__ y, float* __restrict__ h_final, int T, int Dn, int S,
                          ScanEpi epi) {
  using TT = typename Elem<DT>::T;
  constexpr bool MM = DT == HCLSM_BF16 && SG == 16;   // input term on the matrix core
  constexpr int ES = (int)sizeof(TT);
  constexpr int NW = SG * ES / 4;                // 32-bit words of the wave's part of a B / C row
  static_assert(SG == 8 || MM, "8 states per lane, or 16 in the matrix-core form");
  extern __shared__ float red[];                 // [2][TC][NG][64] parts of y
  const int l = threadIdx.x & 63;
  const int g = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int NG = blockDim.x >> 6;
  const int n = blockIdx.x;
  const int s0 = g * SG;
  const int d = blockIdx.y * 64 + l;             // this lane's channel
  const bool act = d < Dn;
  const int dd = act ? d : Dn - 1;

  float a2[SG];
  {
    const float4* ap = reinterpret_cast<const float4*>(A_log + (size_t)dd * S + s0);
#pragma unroll
    for (int q = 0; q < SG / 4; ++q) {
      const float4 v = ap[q];
      const float e4[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float e = exp_comp(e4[r]);
        if (MODE != HCLSM_SCAN_RAW) e = fminf(fmaxf(e, 1e-6f), 1.0f);
        a2[4 * q + r] = -e * HCLSM_LOG2E;
      }
    }
  }
  const float dsk = (Dskip != nullptr && g == 0) ? Dskip[dd] : 0.f;   // the skip term goes with group 0's part
  const bool skip = Dskip != nullptr && g == 0;

  const size_t row0 = (size_t)n * T;
  const int slab = T * Dn * ES;                  // < 2^31 (checked by the dispatcher)
  const auto rx = __builtin_amdgcn_make_buffer_rsrc((void*)(x + row0 * Dn), 0, slab, kRawBufferWord3);
  const auto rd = __builtin_amdgcn_make_buffer_rsrc((void*)(dt + row0 * Dn), 0, slab, kRawBufferWord3);
  const auto ry = __builtin_amdgcn_make_buffer_rsrc((void*)(y + row0 * Dn), 0, slab, kRawBufferWord3);
  const auto rb = __builtin_amdgcn_make_buffer_rsrc((void*)(Bm + row0 * S), 0, T * S * ES, kRawBufferWord3);
  const auto rg = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(MODE == SCAN_BLOCK ? reinterpret_cast<const TT*>(epi.gate) + row0 * Dn : x + row0 * Dn), 0, slab,
      kRawBufferWord3);
  const auto rp = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(epi.y_pre ? reinterpret_cast<TT*>(epi.y_pre) + row0 * Dn : y + row0 * Dn), 0, epi.y_pre ? slab : 0,
      kRawBufferWord3);
  const int vo = dd * ES;
  const int vo_st = act ? vo : 0x7ffffff0;       // past num_records: the store is dropped
  const int pitch = Dn * ES;
  const int ii = l & 31;                         // matrix-core operand row of this lane: state s_row of half a_on
  const bool a_on = (((ii >> 2) & 1) == (l >> 5));
  const int vo_b = a_on ? (s0 + (ii & 3) + 4 * (ii >> 3)) * ES : 0x7ffffff0;
  const uint32_t* bw0 = reinterpret_cast<const uint32_t*>(Bm + row0 * S + s0);
  const uint32_t* cw0 = reinterpret_cast<const uint32_t*>(Cm + row0 * S + s0);
  const int rw = S * ES / 4;                     // words per B / C row

  float xv[TC], dv[TC];
  uint16_t bv[MM ? TC : 1];
  auto load = [&](int t0, float* xo, float* dO, uint16_t* bO) {
#pragma unroll
    for (int j = 0; j < TC; ++j) {
      const int t = t0 + j < T ? t0 + j : T - 1;   // clamped: always a valid row
      xo[j] = buf_ld<DT>(rx, vo, t * pitch);
      dO[j] = buf_ld<DT>(rd, vo, t * pitch);
      if constexpr (MM) bO[j] = __builtin_amdgcn_raw_buffer_load_b16(rb, vo_b, t * S * ES, 0);
    }
  };

  f32x16_t h;
#pragma unroll
  for (int s = 0; s < 16; ++s) h[s] = 0.f;

  // the gates of step t + 1 are formed between the state update of step t and its readout (the exponentials cover
  // the matrix-core latency)
  float gt[SG], dtc;
  auto gates = [&](float dw) {
    dtc = scan_dt<MODE>(dw);
#pragma unroll
    for (int s = 0; s < SG; ++s) gt[s] = dtc * a2[s];
#pragma unroll
    for (int s = 0; s < SG; ++s) gt[s] = fast_exp2(gt[s]);
  };

  uint32_t cw[NW], bw[NW];                       // this step's rows (uniform)
#pragma unroll
  for (int i = 0; i < NW; ++i) { cw[i] = cw0[i]; bw[i] = MM ? 0u : bw0[i]; }
  s16x4_t aop = {0, 0, 0, 0}, bop = {0, 0, 0, 0};
  auto word = [&](const uint32_t* w, int s) -> float {
    if constexpr (DT == HCLSM_BF16) return __uint_as_float(s & 1 ? w[s >> 1] & 0xffff0000u : w[s >> 1] << 16);
    else return __uint_as_float(w[s]);
  };
  auto step = [&](bool odd, int t, int slot, float xs, float dnext, uint16_t bb) {
    const int tn = t + 1 < T ? t + 1 : T - 1;
    uint32_t cwn[NW], bwn[NW];
#pragma unroll
    for (int i = 0; i < NW; ++i) {               // the next step's rows: uniform addresses, scalar loads
      cwn[i] = cw0[(size_t)tn * rw + i];
      if constexpr (!MM) bwn[i] = bw0[(size_t)tn * rw + i];
    }
    float u = dtc * xs;
    if constexpr (MM) {
#pragma unroll
      for (int s = 0; s < SG; ++s) h[s] *= gt[s];
      if (__builtin_expect(odd, 0)) {            // products with a value that is not finite
        const bool uf = fabsf(u) <= __FLT_MAX__;
#pragma unroll
        for (int i = 0; i < NW; ++i) bw[i] = bw0[(size_t)t * rw + i];
#pragma unroll
        for (int s = 0; s < SG; ++s)
          if (!(uf && fabsf(word(bw, s)) <= __FLT_MAX__)) h[s] = fmaf(u, word(bw, s), h[s]);
        u = uf ? u : 0.f;
        bb = (bb & 0x7f80) == 0x7f80 ? 0 : bb;
      }
      const uint32_t u1 = __float_as_uint(u) & 0xffff0000u;
      const float r1 = u - __uint_as_float(u1);
      const uint32_t u2 = __float_as_uint(r1) & 0xffff0000u;
      bop.x = (short)(u1 >> 16);
      bop.y = (short)(u2 >> 16);
      aop.x = aop.y = (short)bb;
      if constexpr (MODE != HCLSM_SCAN_RAW) {    // a clamped dt leaves more than 16 bits in u
        const float r2 = r1 - __uint_as_float(u2);
        bop.z = (short)(__float_as_uint(r2) >> 16);
        aop.z = (short)bb;
      }
      h = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(aop, bop, h, 0, 0, 0);
    } else {
#pragma unroll
      for (int s = 0; s < SG; ++s) h[s] = fmaf(gt[s], h[s], u * word(bw, s));
    }
    if constexpr (MM) __builtin_amdgcn_sched_barrier(0);
    gates(dnext);
    if constexpr (MM) __builtin_amdgcn_sched_barrier(0);
    float y0 = 0.f, y1 = 0.f;
#pragma unroll
    for (int s = 0; s < SG; s += 2) {
      y0 = fmaf(h[s], word(cw, s), y0);
      y1 = fmaf(h[s + 1], word(cw, s + 1), y1);
    }
    y0 += y1;
    if (skip) y0 = fmaf(dsk, xs, y0);
    red[(slot * NG + g) * 64 + l] = y0;
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      cw[i] = cwn[i];
      if constexpr (!MM) bw[i] = bwn[i];
    }
  };
  // step t's output: the parts of the groups in group order
  auto finish = [&](int t, int slot, float gw) {
    float yo = 0.f;
    for (int q = 0; q < NG; ++q) yo += red[(slot * NG + q) * 64 + l];
    if constexpr (MODE == SCAN_BLOCK) {
      buf_st<DT>(yo, rp, vo_st, t * pitch);
      yo *= silu_f(gw);
    }
    buf_st<DT>(yo, ry, vo_st, t * pitch);
  };

  load(0, xv, dv, bv);
  gates(dv[0]);
  int buf = 0;
  for (int t0 = 0; t0 < T; t0 += TC) {
    bool odd = false;                            // the chunk has a u or a B that is not finite
    if constexpr (MM) {                          // (past T: the last step's values again)
      float z = 0.f;                             // NaN if any u is not finite (a clamped dt always is)
      uint32_t b = 0;
#pragma unroll
      for (int j = 0; j < TC; ++j) {
        z = fmaf(MODE == HCLSM_SCAN_RAW ? dv[j] * xv[j] : xv[j], 0.f, z);
        const uint32_t m = bv[j] & 0x7fffu;
        b = b > m ? b : m;
      }
      odd = __any(z != z || b >= 0x7f80u);
    }
    float xn[TC], dn[TC];
    uint16_t bn[MM ? TC : 1];
    load(t0 + TC, xn, dn, bn);
    constexpr int NJ = TC / 2;                   // most steps of a chunk that one wave finishes (NG >= 2)
    float gv[MODE == SCAN_BLOCK ? NJ : 1];
    if constexpr (MODE == SCAN_BLOCK) {
#pragma unroll
      for (int i = 0; i < NJ; ++i) {
        const int t = t0 + g + i * NG;
        gv[i] = buf_ld<DT>(rg, vo, (t < T ? t : T - 1) * pitch);
      }
    }
#pragma unroll
    for (int j = 0; j < TC; ++j)
      if (t0 + j < T) step(odd, t0 + j, buf * TC + j, xv[j], j + 1 < TC ? dv[j + 1 < TC ? j + 1 : 0] : dn[0],
                           bv[MM ? j : 0]);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NJ; ++i) {
      const int j = g + i * NG;
      if (j < TC && t0 + j < T) finish(t0 + j, buf * TC + j, gv[MODE == SCAN_BLOCK ? i : 0]);
    }
#pragma unroll
    for (int j = 0; j < TC; ++j) { xv[j] = xn[j]; dv[j] = dn[j]; if constexpr (MM) bv[j] = bn[j]; }
    buf ^= 1;
  }

  if (h_final != nullptr && act) {
    float* hp = h_final + ((size_t)n * Dn + d) * S + s0;
#pragma unroll
    for (int s = 0; s < SG; ++s) hp[s] = h[s];
  }
}

template <int DT, int MODE, int SG>
static int launch_group(const void* x, const void* dt, const float* A_log, const void* B, const void* C,
                        const float* Dskip, void* y, float* h_final, int64_t batch, int64_t T, int64_t Dn, int64_t S,
                        hipStream_t st, ScanEpi epi) {
  using TT = typename Elem<DT>::T;
  constexpr int TC = 4;
  const int NG = (int)(S / SG);
  dim3 grid((unsigned)batch, (unsigned)((Dn + 63) / 64));
  const size_t lds = (size_t)2 * TC * NG * 64 * sizeof(float);
  hipLaunchKernelGGL((ssm_scan_fwd_group_kernel<DT, MODE, SG, TC>), grid, dim3(64 * NG), lds, st, (const TT*)x,
                     (const TT*)dt, A_log, (const TT*)B, (const TT*)C, Dskip, (TT*)y, h_final, (int)T, (int)Dn, (int)S,
                     epi);
  HCLSM_LAUNCH_CHECK();
  return 0;
}

static inline bool al(const void* p, uintptr_t a) { return (((uintptr_t)p) & (a - 1)) == 0; }

template <int DT, int SG>
static int group_mode(int mode, const void* x, const void* dt, const float* A_log, const void* B, const void* C,
                      const float* Dskip, void* y, float* h_final, int64_t batch, int64_t T, int64_t Dn, int64_t S,
                      hipStream_t st, ScanEpi epi) {
  if (mode == HCLSM_SCAN_RAW)
    return launch_group<DT, HCLSM_SCAN_RAW, SG>(x, dt, A_log, B, C, Dskip, y, h_final, batch, T, Dn, S, st, epi);
  if (mode == HCLSM_SCAN_MODEL)
    return launch_group<DT, HCLSM_SCAN_MODEL, SG>(x, dt, A_log, B, C, Dskip, y, h_final, batch, T, Dn, S, st, epi);
  return launch_group<DT, SCAN_BLOCK, SG>(x, dt, A_log, B, C, Dskip, y, h_final, batch, T, Dn, S, st, epi);
}

int scan_fwd_group(int mode, const void* x, const void* dt, const float* A_log, const void* B, const void* C,
                   const float* Dskip, void* y, float* h_final, int64_t batch, int64_t T, int64_t Dn, int64_t S,
                   int dtype, hipStream_t st, ScanEpi epi) {
  if (S % 8 != 0 || S < 24 || S > 8 * GRP_MAX_WAVES) return HCLSM_ERR_UNSUPPORTED;
  if (dtype != HCLSM_BF16 && dtype != HCLSM_F32) return HCLSM_ERR_UNSUPPORTED;
  const int64_t es = dtype == HCLSM_F32 ? 4 : 2;
  if (T * Dn * es >= 0x7fffffffLL || T * S * es >= 0x7fffffffLL) return HCLSM_ERR_UNSUPPORTED;
  if (!al(A_log, 16) || !al(B, 4) || !al(C, 4)) return HCLSM_ERR_UNSUPPORTED;
  int cus = 0;
  const int rc = device_cus(&cus);
  if (rc) return rc;
  const int64_t w16 = batch * ((Dn + 63) / 64) * S / 16;   // waves at 16 states a lane
  // 16 states a lane on the matrix core from four waves a CU on; below, 8 a lane double the waves (us, 16 | 8):
  // 128 x 16 x 256, S 32 (1024 waves) 10.8 | 8.7; 64 x 1024 x 384, S 32 (768) 537 | 440; 256 x 16 x 256, S 64 (4096)
  // 17.6 | 19.1; 1024 x 64 x 384, S 32 (12288) 149 | 174.  In fp32 both are within 3% of each other past that, so 8
  // is used throughout.  d_state 16 stays on one lane per channel (ssm_scan.hip): in bf16 so that the forward with and
  // without the backward's checkpoints is the same kernel; in fp32 a forward on a small grid is faster here (869 x 77 x
  // 64: 48.7 | 42.9) but a training step with the backward after it is not (213 | 233).
  const bool few = w16 <= 4 * (int64_t)cus;
  if (dtype == HCLSM_F32)
    return group_mode<HCLSM_F32, 8>(mode, x, dt, A_log, B, C, Dskip, y, h_final, batch, T, Dn, S, st, epi);
  if (S % 16 != 0 || few)
    return group_mode<HCLSM_BF16, 8>(mode, x, dt, A_log, B, C, Dskip, y, h_final, batch, T, Dn, S, st, epi);
  return group_mode<HCLSM_BF16, 16>(mode, x, dt, A_log, B, C, Dskip, y, h_final, batch, T, Dn, S, st, epi);
}

}  // namespace hclsm
