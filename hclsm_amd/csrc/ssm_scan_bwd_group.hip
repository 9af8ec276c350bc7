// Selective SSM scan backward (see ssm_scan_bwd.hip for the recurrences) for wide states: the states of a channel are
// split over the waves of a workgroup.
//
// A workgroup owns 64 channels; wave g keeps states g * SG .. of them, one lane a channel, so no state is padding and
// the step loop is the same however wide the state is.  It walks sequences blockIdx.x, + gridDim.x, ... (one gA / gD
// partial per workgroup instead of per sequence), and each sequence backwards in windows of 16 steps:
//   - B / C rows and, per step and channel, dt (after softplus / clamps), dt x and the output's gradient go to LDS once
//     per workgroup, each wave preparing a share of the steps;
//   - the chunks of 4 steps are walked backwards as in ssm_scan_bwd.hip: the chunk's states are recomputed into
//     registers (from the window's start, or the state after two chunks kept in LDS), then the reverse recurrence runs;
//   - gB / gC are summed over the wave's lanes (its channels); q = sum_s gh B and sum_s g_arg A go to LDS per wave, and
//     after a barrier wave g adds the groups' parts for steps g, g + NG and writes gx, gdt.
// Sequences longer than a window first run forward once, leaving each window's start in memory.
// SG = 16, bf16: u B and gy C enter the states on the matrix core (operand layout of ssm_scan_fwd_mfma_kernel; exact in
// up to three bf16 pieces; see ssm_scan_group.hip for non-finite values).  SG = 8: on the VALU.
//
// Bound by VALU issue (about 30 slots per state update: 6 for each of three forward evaluations, 10 for the reverse
// step, 5 for the two sums across the wave) with few waves to hide it: registers allow 4 per SIMD at 8 states a lane and
// 3 at 16, LDS (160 KB a CU) workgroups of 12 waves at d_state 24, 32 and 48, 15, 14 and 16 at 40, 56 and 64 with 8 a
// lane; 9, 10, 6, 7 and 8 at 48, 80, 96, 112 and 128 with 16.  16 a lane spills (40 registers, 72 with the gate; fp32 76
// to 82), 8 a lane does not.  Measured on MI355X, us per call with the tail
// launch (before: states padded to a power of two over 2 or 4 lanes of a wave, 44 KB of LDS per two waves):
//   1024 x 16 x 384, S 48, bf16     701 -> 356 (block 804 -> 377)    512 x 16 x 512, S 64, fp32  472 -> 251
//   256 x 64 x 384, S 32, bf16      287 -> 226                       121 x 120 x 192, S 32, fp32 263 -> 179
//   64 x 16 x 768, S 96, bf16 block 332 -> 126                       128 x 16 x 256, S 32, fp32 43.6 -> 28.9
// Not kept: d_state 16 as two groups (1024 x 64 x 384: 416 -> 787), pointers instead of buffer resources (more registers),
// the outputs' inputs requested before the reverse steps (13 registers more: one wave per SIMD less).
#include "internal.h"
#include "ssm_scan_bwd_common.h"
#include "ssm_scan_bwd_group.h"

namespace hclsm {

typedef short s16x4_t __attribute__((ext_vector_type(4)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));

constexpr int BG_K = 4;                          // steps per chunk (their states stay in registers)
constexpr int BG_WIN = BG_WINDOW;                // steps per window (a checkpoint in memory at each window's start)
constexpr int BG_MAX_WAVES = 8;
constexpr int BG_MIN_S = 24;

struct BwdGroupArgs { int N, T, Dn, S, nwin; };

// The rank-1 operand of one lane: v as bf16 pieces whose sum is v (NP = 1: v is a bf16 value; 2: at most 16
// significant bits; 3: any).
template <int NP>
__device__ __forceinline__ void split_op(float v, s16x4_t& o) {
  const uint32_t p1 = __float_as_uint(v) & 0xffff0000u;
  o.x = (short)(p1 >> 16);
  if constexpr (NP >= 2) {
    const float r1 = v - __uint_as_float(p1);
    const uint32_t p2 = __float_as_uint(r1) & 0xffff0000u;
    o.y = (short)(p2 >> 16);
    if constexpr (NP >= 3) o.z = (short)(__float_as_uint(r1 - __uint_as_float(p2)) >> 16);
  }
}
__device__ __forceinline__ bool finite_f(float v) { return fabsf(v) <= __FLT_MAX__; }
__device__ __forceinline__ s16x4_t fill_op(uint16_t b, int np) {
  return s16x4_t{(short)b, (short)(np >= 2 ? b : 0), (short)(np >= 3 ? b : 0), 0};
}

template <int DT, int MODE, int SG>
__global__ void __launch_bounds__(64 * BG_MAX_WAVES) __attribute__((amdgpu_waves_per_eu(SG == 8 ? 4 : 3)))
ssm_scan_bwd_group_kernel(const typename Elem<DT>::T* __restrict__ x, const typename Elem<DT>::T* __restrict__ dt,
                          const float* __restrict__ A_log, const typename Elem<DT>::T* __restrict__ Bm,
                          const typename Elem<DT>::T* __restrict__ Cm, const float* __restrict__ Dskip,
                          const typename Elem<DT>::T* __restrict__ gy, typename Elem<DT>::T* __restrict__ gx,
                          typename Elem<DT>::T* __restrict__ gdt, BwdGate gate, float* __restrict__ ckpt,
                          float* __restrict__ gbc, float* __restrict__ gA_part, float* __restrict__ gD_part,
                          BwdGroupArgs a) {
  using TT = typename Elem<DT>::T;
  constexpr bool MM = DT == HCLSM_BF16 && SG == 16;
  constexpr int ES = (int)sizeof(TT);
  constexpr int K = BG_K;
  constexpr int VL = RSCount<SG, 1>::value;
  constexpr bool BLK = MODE >= HCLSM_SCAN_BLOCK, GATE = MODE == BWD_BLOCK_GATE;
  constexpr int NPU = MODE == HCLSM_SCAN_RAW ? 2 : 3;      // bf16 pieces of u = dt x
  constexpr int NPG = MODE == BWD_BLOCK_GATE ? 3 : 1;      // and of gy (g silu(gate) in fp32 there)
  const int l = threadIdx.x & 63;
  const int g = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int NG = blockDim.x >> 6;
  const int T = a.T, Dn = a.Dn, S = a.S;
  const int SH = S + 2;                          // pitch of the 16-bit rows: entry S is zero
  extern __shared__ __align__(16) float lds[];
  float* slot = lds + g * 2 * SG * 64;           // [2][SG][64] of this wave: start of the current chunk, of chunk 2
  float* sB = lds + NG * 2 * SG * 64;            // [BG_WIN][S] B rows of the window, fp32
  float* sC = sB + BG_WIN * S;                   // [BG_WIN][S] C rows (without the matrix core)
  float* red = MM ? sC : sC + BG_WIN * S;        // [K][2 S] sums over the channels: gB | gC
  float* sQ = red + K * 2 * S;                   // [K][2][NG][64] parts of q and gda2
  float* sDt = sQ + K * 2 * NG * 64;             // [BG_WIN][64] dt as the recurrence uses it,
  float* sU = sDt + BG_WIN * 64;                 //   dt x (0 on lanes without a channel)
  float* sG = sU + BG_WIN * 64;                  //   and the gradient of the scan output (0 there)
  uint16_t* sBh = reinterpret_cast<uint16_t*>(sG + BG_WIN * 64);   // [BG_WIN][SH], matrix core
  uint16_t* sCh = sBh + BG_WIN * SH;
  int* sOdd = reinterpret_cast<int*>(sCh + BG_WIN * SH);           // matrix core: a staged value is not finite

  const int s0 = g * SG;
  const int d = blockIdx.y * 64 + l;
  const bool act = d < Dn;
  const int dd = act ? d : Dn - 1;
  const int ii = l & 31;                         // matrix-core operand row: state s_row of half a_on
  const bool a_on = (((ii >> 2) & 1) == (l >> 5));
  const int op_col = a_on ? s0 + (ii & 3) + 4 * (ii >> 3) : S;

  float a2[SG];
#pragma unroll
  for (int j = 0; j < SG; ++j) {
    const float e = expf(A_log[(size_t)dd * S + s0 + j]);
    a2[j] = -((MODE != HCLSM_SCAN_RAW) ? fminf(fmaxf(e, 1e-6f), 1.0f) : e) * HCLSM_LOG2E;
  }
  const float dsk = Dskip ? Dskip[dd] : 0.f;
  if (MM && threadIdx.x == 0) *sOdd = 0;
  if constexpr (MM)
    for (int e = threadIdx.x; e < 2 * BG_WIN * 2; e += blockDim.x) (e & 1 ? sCh : sBh)[(e >> 2) * SH + S + ((e >> 1) & 1)] = 0;

  // The matrix core takes finite values only: a lane's column also meets the other half's channel with zero weights, and a
  // zero piece of u meets B.  From the first window with a value that is not finite on, `odd` is set and the products
  // with such a value are formed here instead (v: u or gy, w: the row's B or C), in the states' place; the operands have
  // 0 there.  What is finite comes out the same either way.
  bool odd = false;
  auto fix_up = [&](f32x16_t& st, float& v, uint16_t& w_op, const uint16_t* w) {
    const bool vf = finite_f(v);
#pragma unroll
    for (int j = 0; j < SG; ++j) {
      const float wj = bf16_bits_to_f32(w[j]);
      if (!(vf && finite_f(wj))) st[j] = fmaf(v, wj, st[j]);
    }
    v = vf ? v : 0.f;
    w_op = (w_op & 0x7f80) == 0x7f80 ? 0 : w_op;
  };
  f32x16_t gh;
  float gA[SG], gD = 0.f;
#pragma unroll
  for (int j = 0; j < SG; ++j) gA[j] = 0.f;
  const unsigned pitch = (unsigned)Dn * ES;
  const int slab = (int)(T * pitch);             // < 2^31: checked by the entry point
  const int vo = dd * ES;
  const int vo_st = act ? vo : 0x7ffffff0;       // past num_records: the store is dropped

  for (int n = blockIdx.x; n < a.N; n += gridDim.x) {
    const size_t row0 = (size_t)n * T;
    auto rsrc = [&](const void* p, int bytes) { return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, bytes, kRawBufferWord3); };
    const auto rx = rsrc(x + row0 * Dn, slab), rdt = rsrc(dt + row0 * Dn, slab), rgy = rsrc(gy + row0 * Dn, slab);
    const auto rgx = rsrc(gx + row0 * Dn, slab), rgdt = rsrc(gdt + row0 * Dn, slab);
    const auto rb = rsrc(Bm + row0 * S, T * S * ES), rc = rsrc(Cm + row0 * S, T * S * ES);
    const auto rgt = rsrc(GATE ? reinterpret_cast<const TT*>(gate.gate) + row0 * Dn : x + row0 * Dn, slab);
    const auto rpr = rsrc(GATE ? reinterpret_cast<const TT*>(gate.y_pre) + row0 * Dn : x + row0 * Dn, slab);
    const auto rgg = rsrc(GATE ? reinterpret_cast<TT*>(gate.g_gate) + row0 * Dn : gx + row0 * Dn, GATE ? slab : 0);

    // the rows of window w; steps past T read as zero
    bool seen = false;                           // this thread staged a value that is not finite (matrix core)
    auto look = [&](float v) { if constexpr (MM) seen |= !finite_f(v); };
    auto staged = [&]() {
      if (MM && seen) *sOdd = 1;
      __syncthreads();
      if constexpr (MM) odd = __builtin_amdgcn_readfirstlane(*sOdd);
    };
    auto stage = [&](int w) {
      for (int e = threadIdx.x; e < BG_WIN * S; e += blockDim.x) {
        const int off = (w * BG_WIN * S + e) * ES;
        if constexpr (MM) {
          const uint16_t b = __builtin_amdgcn_raw_buffer_load_b16(rb, off, 0, 0);
          const uint16_t c = __builtin_amdgcn_raw_buffer_load_b16(rc, off, 0, 0);
          const int r = e / S;
          sB[e] = bf16_bits_to_f32(b);
          look(sB[e]);
          look(bf16_bits_to_f32(c));
          sBh[r * SH + e - r * S] = b;
          sCh[r * SH + e - r * S] = c;
        } else {
          sB[e] = buf_ld<DT>(rb, off, 0);
          sC[e] = buf_ld<DT>(rc, off, 0);
        }
      }
    };
    // dt as the recurrence uses it; 0 for a missing step
    auto dt_of = [&](float v, bool live) {
      if constexpr (MODE == HCLSM_SCAN_MODEL) return live ? fminf(fmaxf(v, 1e-3f), 1.0f) : 0.f;
      else if constexpr (BLK) return live ? fminf(fmaxf(softplus_f(v), 1e-3f), 1.0f) : 0.f;
      else return v;
    };
    // a window's step values, wave g those of steps g, g + NG, ...: loads first, four steps at a time
    auto stage_values = [&](int w, bool with_g) {
      for (int r0 = g; r0 < BG_WIN; r0 += 4 * NG) {
        float xv[4], dv[4], gv[4], gt[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const int so = (int)((unsigned)(w * BG_WIN + r0 + k * NG) * pitch);   // past the slab for steps >= T: reads 0
          xv[k] = buf_ld<DT>(rx, vo, so);
          dv[k] = buf_ld<DT>(rdt, vo, so);
          if (with_g) {
            gv[k] = buf_ld<DT>(rgy, vo, so);
            if constexpr (GATE) gt[k] = buf_ld<DT>(rgt, vo, so);
          }
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const int r = r0 + k * NG;
          if (r < BG_WIN) {
            const float v = dt_of(dv[k], w * BG_WIN + r < T);
            sDt[r * 64 + l] = v;
            const float u = act ? v * xv[k] : 0.f;
            sU[r * 64 + l] = u;
            look(u);
            if (with_g) {
              const float gr = act ? (GATE ? gv[k] * silu_f(gt[k]) : gv[k]) : 0.f;
              sG[r * 64 + l] = gr;
              look(gr);
            }
          }
        }
      }
    };
    f32x16_t hc;
    // one forward step: hc = exp(dt A) hc + u B_r (r: row of the window)
    auto fwd_step = [&](int r, float dtv, float u) {
      if constexpr (MM) {
        uint16_t b = sBh[r * SH + op_col];
#pragma unroll
        for (int j = 0; j < SG; ++j) hc[j] *= fast_exp2(dtv * a2[j]);
        if (__builtin_expect(odd, 0)) fix_up(hc, u, b, sBh + r * SH + s0);
        s16x4_t bop = {0, 0, 0, 0};
        split_op<NPU>(u, bop);
        hc = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(fill_op(b, NPU), bop, hc, 0, 0, 0);
      } else {
#pragma unroll
        for (int j = 0; j < SG; ++j) hc[j] = fmaf(fast_exp2(dtv * a2[j]), hc[j], u * sB[r * S + s0 + j]);
      }
    };
    float* ck = ckpt + (size_t)n * (a.nwin - 1) * S * Dn + (size_t)s0 * Dn + dd;   // window w's start at w - 1
    auto ld_start = [&](int w) {
#pragma unroll
      for (int j = 0; j < SG; ++j) hc[j] = (w > 0 && act) ? ck[((size_t)(w - 1) * S + j) * Dn] : 0.f;
    };
    // the first nc chunks of the window forward; with keep2 the state after two goes to slot 1
    auto sweep = [&](int nc, bool keep2) {
      for (int c = 0; c < nc; ++c) {
#pragma unroll
        for (int i = 0; i < K; ++i) {
          __builtin_amdgcn_sched_barrier(0);
          fwd_step(c * K + i, sDt[(c * K + i) * 64 + l], sU[(c * K + i) * 64 + l]);
        }
        if (keep2 && c == 1)
#pragma unroll
          for (int j = 0; j < SG; ++j) slot[(SG + j) * 64 + l] = hc[j];
      }
    };

    if (a.nwin > 1) {   // window starts, forward
#pragma unroll
      for (int j = 0; j < 16; ++j) hc[j] = 0.f;
      for (int w = 0; w + 1 < a.nwin; ++w) {
        __syncthreads();
        stage(w);
        stage_values(w, false);
        staged();
        sweep(BG_WIN / K, false);
        if (act)
#pragma unroll
          for (int j = 0; j < SG; ++j) ck[((size_t)w * S + j) * Dn] = hc[j];
      }
    }
#pragma unroll
    for (int j = 0; j < 16; ++j) gh[j] = 0.f;

    for (int w = a.nwin - 1; w >= 0; --w) {
      __syncthreads();
      stage(w);
      stage_values(w, true);
      staged();
      const int left = T - w * BG_WIN;
      const int nch = left >= BG_WIN ? BG_WIN / K : (left + K - 1) / K;
      for (int c = nch - 1; c >= 0; --c) {
        const int t0 = w * BG_WIN + c * K;
        if (c == 2 && nch == 4) {
#pragma unroll
          for (int j = 0; j < SG; ++j) hc[j] = slot[(SG + j) * 64 + l];
        } else {
          ld_start(w);
          if (c > 0) sweep(c, c == 3);
        }
#pragma unroll
        for (int j = 0; j < SG; ++j) slot[j * 64 + l] = hc[j];
        // recompute the chunk's states into hk and reduce gC_t = sum_d gy_t h_t over the wave's channels
        float hk[K - 1][SG];
#pragma unroll
        for (int i = 0; i < K; ++i) {
          const int r = c * K + i;
          __builtin_amdgcn_sched_barrier(0);
          fwd_step(r, sDt[r * 64 + l], sU[r * 64 + l]);
          const float gv = sG[r * 64 + l];
          float v[SG];
#pragma unroll
          for (int j = 0; j < SG; ++j) {
            if (i < K - 1) hk[i < K - 1 ? i : 0][j] = hc[j];
            v[j] = gv * hc[j];
          }
          const int off = RS<SG, 1>::run(v, l);
#pragma unroll
          for (int e = 0; e < VL; ++e) red[i * 2 * S + S + s0 + off + e] = v[e];
        }
        asm volatile("" ::: "memory");   // the reverse steps recompute the gates (registers are the occupancy limit)
        // the chunk's part of gA, in the places of hk's states as they are used up: four steps summed first keep the chain
        // of additions over a walk short (error of gA_log against float64 at 512 x 16 x 512, S 64: 1.7e-7; step by step
        // 2.4e-7, one partial per sequence 1.8e-7; 354.8 -> 356.8 us at 1024 x 16 x 384, S 48, else equal)
        float gc[SG];
#pragma unroll
        for (int i = K - 1; i >= 0; --i) {
          const int r = c * K + i;
          __builtin_amdgcn_sched_barrier(0);
          const float dv = sDt[r * 64 + l], um = sU[r * 64 + l], gv = sG[r * 64 + l];
          if constexpr (MM) {
            float gf = gv;
            uint16_t c_op = sCh[r * SH + op_col];
            if (__builtin_expect(odd, 0)) fix_up(gh, gf, c_op, sCh + r * SH + s0);
            s16x4_t bop = {0, 0, 0, 0};
            split_op<NPG>(gf, bop);
            gh = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(fill_op(c_op, NPG), bop, gh, 0, 0, 0);
          }
          float v[SG], q = 0.f, gda2 = 0.f;     // gda2 = sum garg * A * log2(e); times ln 2 below
#pragma unroll
          for (int j = 0; j < SG; ++j) {
            if constexpr (!MM) gh[j] = fmaf(gv, sC[r * S + s0 + j], gh[j]);
            const float hp = (i > 0) ? hk[i > 0 ? i - 1 : 0][j] : slot[j * 64 + l];   // h_{t-1}
            q = fmaf(gh[j], sB[r * S + s0 + j], q);
            v[j] = gh[j] * um;                   // -> gB
            gh[j] *= fast_exp2(dv * a2[j]);      // carried to step t-1
            const float garg = gh[j] * hp;
            gda2 = fmaf(garg, a2[j], gda2);
            gc[j] = i == K - 1 ? garg * dv : fmaf(garg, dv, gc[j]);
            if (i == 0) gA[j] += gc[j];
          }
          sQ[((i * 2 + 0) * NG + g) * 64 + l] = q;
          sQ[((i * 2 + 1) * NG + g) * 64 + l] = gda2;
          const int off = RS<SG, 1>::run(v, l);
#pragma unroll
          for (int e = 0; e < VL; ++e) red[i * 2 * S + s0 + off + e] = v[e];
        }
        // what this wave's part of the outputs needs (steps g and g + NG of the chunk), in flight over the barrier
        constexpr int NI = K / 2;                // most of them (NG >= 2)
        float xe[NI], de[NI], ge[GATE ? NI : 1], te[GATE ? NI : 1], pe[GATE ? NI : 1];
#pragma unroll
        for (int k = 0; k < NI; ++k) {
          const int so = (int)((unsigned)(t0 + g + k * NG) * pitch);
          xe[k] = buf_ld<DT>(rx, vo, so);
          if constexpr (MODE != HCLSM_SCAN_RAW) de[k] = buf_ld<DT>(rdt, vo, so);
          if constexpr (GATE) {
            ge[k] = buf_ld<DT>(rgy, vo, so);
            te[k] = buf_ld<DT>(rgt, vo, so);
            pe[k] = buf_ld<DT>(rpr, vo, so);
          }
        }
        __syncthreads();
        for (int e = threadIdx.x; e < K * 2 * S; e += blockDim.x) {
          const int i = e / (2 * S);
          if (t0 + i < T) gbc[(((size_t)blockIdx.y * a.N + n) * T + t0) * 2 * S + e] = red[e];
        }
        // gx, gdt (and the gate's gradient) of this wave's steps: the parts of the groups in group order
#pragma unroll
        for (int k = 0; k < NI; ++k) {
          const int i = g + k * NG, t = t0 + i;
          if (i >= K) break;
          float q = 0.f, gda2 = 0.f;
          for (int p = 0; p < NG; ++p) {
            q += sQ[((i * 2 + 0) * NG + p) * 64 + l];
            gda2 += sQ[((i * 2 + 1) * NG + p) * 64 + l];
          }
          const float dv = sDt[(c * K + i) * 64 + l], gv = sG[(c * K + i) * 64 + l];
          float gdv = fmaf(gda2, HCLSM_LN2, q * xe[k]);
          const int so = t < T ? (int)((unsigned)t * pitch) : slab;   // a missing step stores nothing
          if constexpr (MODE == HCLSM_SCAN_MODEL) {
            if (!(de[k] >= 1e-3f && de[k] <= 1.0f)) gdv = 0.f;
          }
          if constexpr (BLK) {   // through the clamp (closed interval) and softplus
            const float sp = softplus_f(de[k]);
            gdv = (sp >= 1e-3f && sp <= 1.0f) ? gdv * __builtin_amdgcn_rcpf(1.f + __expf(-de[k])) : 0.f;
          }
          if constexpr (GATE) {
            const float sg = __builtin_amdgcn_rcpf(1.f + __expf(-te[k]));
            buf_st<DT>(ge[k] * pe[k] * sg * fmaf(te[k], 1.f - sg, 1.f), rgg, vo_st, so);
          }
          buf_st<DT>(fmaf(q, dv, dsk * gv), rgx, vo_st, so);
          buf_st<DT>(gdv, rgdt, vo_st, so);
          gD = fmaf(gv, xe[k], gD);
        }
        __syncthreads();
      }
    }
  }
  sQ[g * 64 + l] = gD;
  __syncthreads();
  if (g == 0) {
    gD = 0.f;
    for (int p = 0; p < NG; ++p) gD += sQ[p * 64 + l];
  }
  if (act) {
#pragma unroll
    for (int j = 0; j < SG; ++j) gA_part[((size_t)blockIdx.x * S + s0 + j) * Dn + d] = gA[j];
    if (g == 0) gD_part[(size_t)blockIdx.x * Dn + d] = gD;
  }
}

static size_t group_lds(int NG, int SG, int S, bool mm) {
  size_t f = (size_t)NG * 2 * SG * 64 + (size_t)BG_WIN * S * (mm ? 1 : 2) + (size_t)BG_K * 2 * S + (size_t)BG_K * 2 * NG * 64 + (size_t)3 * BG_WIN * 64;
  return f * 4 + (mm ? (size_t)2 * BG_WIN * (S + 2) * 2 + 4 : 0);
}

// Sequences one workgroup walks: the fewest rounds of resident workgroups times their length, half a sequence added
// to each round for its start (A_log, the partials of gA).
static int64_t walk_length(int64_t N, int64_t nblk, int64_t resident) {
  int64_t best = 1;
  double cost = 0.;
  for (int64_t per = 1; per <= 64 && per <= N; ++per) {
    const int64_t wgs = (N + per - 1) / per * nblk;
    const double c = (double)((wgs + resident - 1) / resident) * ((double)per + 0.5);
    if (per == 1 || c < cost) { best = per; cost = c; }
  }
  return best;
}

template <int DT, int MODE, int SG>
static int launch_group(const void* x, const void* dt, const float* A_log, const void* B, const void* C,
                        const float* Dskip, const void* gy, void* gx, void* gdt, BwdGate gate, float* ck, float* gbc,
                        float* ga, float* gd, int64_t N, int64_t T, int64_t Dn, int64_t S, int* parts, hipStream_t st) {
  using TT = typename Elem<DT>::T;
  const int NG = (int)(S / SG);
  const size_t lds = group_lds(NG, SG, (int)S, DT == HCLSM_BF16 && SG == 16);
  static std::atomic<int> cache[BG_MAX_WAVES + 1][HCLSM_MAX_DEVICES];
  const auto fn = ssm_scan_bwd_group_kernel<DT, MODE, SG>;
  int resident = 0;
  if (int rc = device_launch_setup((const void*)fn, 64 * NG, lds, 160 * 1024, cache[NG], &resident)) return rc;
  const int64_t nblk = (Dn + 63) / 64;
  const int64_t per = walk_length(N, nblk, resident);   // sequences a workgroup walks
  const int64_t gridx = (N + per - 1) / per;
  *parts = (int)gridx;
  BwdGroupArgs a{(int)N, (int)T, (int)Dn, (int)S, (int)((T + BG_WIN - 1) / BG_WIN)};
  hipLaunchKernelGGL(fn, dim3((unsigned)gridx, (unsigned)nblk), dim3(64 * NG), lds, st, (const TT*)x, (const TT*)dt,
                     A_log, (const TT*)B, (const TT*)C, Dskip, (const TT*)gy, (TT*)gx, (TT*)gdt, gate, ck, gbc, ga, gd,
                     a);
  HCLSM_LAUNCH_CHECK();
  return 0;
}

bool bwd_group_ok(int64_t T, int64_t Dn, int64_t S, int dtype) {
  if (dtype != HCLSM_BF16 && dtype != HCLSM_F32) return false;
  if (S % 8 != 0 || S < BG_MIN_S || S > 16 * BG_MAX_WAVES || (S > 8 * BG_MAX_WAVES && S % 16 != 0)) return false;
  const int64_t es = dtype == HCLSM_F32 ? 4 : 2;
  return T * Dn * es < (1LL << 31) && T * S * es < (1LL << 31) && (Dn + 63) / 64 <= 65535;
}

int bwd_group(int mode, const void* x, const void* dt, const float* A_log, const void* B, const void* C,
              const float* Dskip, const void* gy, void* gx, void* gdt, BwdGate gate, float* ck, float* gbc, float* ga,
              float* gd, int64_t N, int64_t T, int64_t Dn, int64_t S, int dtype, int* parts, hipStream_t st) {
#define HCLSM_BG(DT_, SG_, MODE_)                                                                                  \
  if (mode == MODE_)                                                                                               \
    return launch_group<DT_, MODE_, SG_>(x, dt, A_log, B, C, Dskip, gy, gx, gdt, gate, ck, gbc, ga, gd, N, T, Dn, S, \
                                         parts, st);
#define HCLSM_BG_M(DT_, SG_) \
  HCLSM_BG(DT_, SG_, HCLSM_SCAN_RAW) HCLSM_BG(DT_, SG_, HCLSM_SCAN_MODEL) HCLSM_BG(DT_, SG_, HCLSM_SCAN_BLOCK)
  int cus = 0;
  if (int rc = device_cus(&cus)) return rc;
  // 8 or 16 states a lane.  Past 64 states 8 a lane would need more than 8 waves.  The widths with a choice are 32, 48 and
  // 64; forward and backward together in us, 8 | 16 a lane:
  //   bf16 1024 x 16 x 384:  242 | 302   475 | 419   435 | 483     bf16 256 x 64 x 384:  281 | 432   533 | 526   499 | 654
  //   bf16 32 x 64 x 384:    151 | 169   152 | 174   155 | 175     fp32 512 x 16 x 512:         304 | 360   317 | 383
  // 16 a lane halves the waves and takes the rank-1 products off the VALU in bf16 (fp32 has no matrix core for them) but
  // spills 40 to 72 registers: it gains on full grids at 48 alone, the width whose workgroups of S/8 waves do not divide
  // the 16 wave slots that the registers of 8 a lane allow.  (Wave slots are not the whole reason: LDS leaves 12 of them
  // in use at 32 and at 48.)
  const bool gaps = S % 16 == 0 && 16 % (S / 8) != 0;
  const bool wide = S > 8 * BG_MAX_WAVES || (dtype == HCLSM_BF16 && gaps && N * ((Dn + 63) / 64) >= 4 * (int64_t)cus);
  if (wide) {
    if (dtype == HCLSM_BF16) { HCLSM_BG_M(HCLSM_BF16, 16) HCLSM_BG(HCLSM_BF16, 16, BWD_BLOCK_GATE) }
    else { HCLSM_BG_M(HCLSM_F32, 16) }
  } else {
    if (dtype == HCLSM_BF16) { HCLSM_BG_M(HCLSM_BF16, 8) HCLSM_BG(HCLSM_BF16, 8, BWD_BLOCK_GATE) }
    else { HCLSM_BG_M(HCLSM_F32, 8) }
  }
#undef HCLSM_BG_M
#undef HCLSM_BG
  return HCLSM_ERR_MODE;
}

}  // namespace hclsm
