// One Level-0 SSM block (SimplifiedSSMBlock, hclsm/dynamics/level0_ssm.py:30-107) in bf16 operands with fp32 residual
// stream and parameters: forward and backward as two calls of a few launches each.
//
//   u = LN(x); z = u W_in^T, gate = u W_gate^T; dt = z W_dt^T + b, B = z W_B^T, C = z W_C^T;
//   y = silu(gate) * scan(z, clamp(softplus(dt)), A_log, B, C); out = x + y W_out^T
//
// Forward: weight cast (and transposes for the backward), LayerNorm, two grouped GEMM launches, the scan, one GEMM.
// Backward: gy = g W_out; the scan's backward with the gate's chain rule; gz = gz_scan + gdt W_dt + gB W_B + gC W_C and
// gu = gz W_in + ggate W_gate as GEMMs over several operand pairs; LayerNorm's backward; all weight gradients in one
// grouped launch split over the rows, and one reduction.
//
// What it replaces took 63 launches per step of a 1024 x 16 layer of width 192 (d_state 48): the weight gradients as
// library GEMMs over 16384 rows without a row split (six of 98 us), ten elementwise passes for the gate, a cast per
// weight and operand, 2160 us in all; the host needed 1.1 to 1.3 ms for them whatever the size.  Now 14 launches and 683
// us: scan backward 390, forward 85, six GEMM launches 107, weight gradients 62 (239 with a branch per load, which left
// one load in flight), LayerNorm's backward 26, the rest 34 (each kernel in the trace; together 3% more than the call).
// Smaller layers are bound by the host here too: 512 x 16, width 128, d_state 32, 1360 -> 315 us.
#include "internal.h"
#include "mfma.h"
#include "scan_common.h"
#include "ssm_scan_bwd_group.h"

namespace hclsm {

constexpr int BK_LD = 72;   // LDS row pitch in 16-bit elements: 64 + 8

// ------------------------------------------------------------------------------------------ weight casts
struct CastJob { const float* src; uint16_t* dst; uint16_t* dst_t; int rows, cols; int64_t ld_t; int blk0; };
struct CastJobs { CastJob j[6]; int n; };

// Each workgroup: one 32 x 32 tile of one matrix; dst [rows][cols], dst_t (nullable) transposed with row stride ld_t.
__global__ void __launch_bounds__(256) block_cast_kernel(CastJobs js) {
  __shared__ uint16_t tile[32][34];
  int k = 0;
  while (k + 1 < js.n && (int)blockIdx.x >= js.j[k + 1].blk0) ++k;
  const CastJob jb = js.j[k];
  const int tc = (jb.cols + 31) / 32, t = blockIdx.x - jb.blk0, r0 = t / tc * 32, c0 = t % tc * 32;
  const int c = threadIdx.x & 31;
  for (int r = threadIdx.x >> 5; r < 32; r += 8)
    if (r0 + r < jb.rows && c0 + c < jb.cols) {
      const uint16_t v = f32_to_bf16_bits(jb.src[(int64_t)(r0 + r) * jb.cols + c0 + c]);
      jb.dst[(int64_t)(r0 + r) * jb.cols + c0 + c] = v;
      tile[r][c] = v;
    }
  if (jb.dst_t == nullptr) return;
  __syncthreads();
  for (int r = threadIdx.x >> 5; r < 32; r += 8)   // column c0 + r of the source, rows r0 + c
    if (c0 + r < jb.cols && r0 + c < jb.rows) jb.dst_t[(int64_t)(c0 + r) * jb.ld_t + r0 + c] = tile[c][r];
}

// ------------------------------------------------------------------------------------------ grouped GEMM
// Y[M, N] = sum over segments X_s W_s^T (+ bias) (+ add): 16-bit W [N, K_s], X 16-bit or fp32 (rounded while staged).
struct GemmSeg { const void* x; int64_t ldx; const uint16_t* w; int64_t ldw; int K, x_f32; };
struct GemmProb {
  GemmSeg seg[3];
  int nseg, N;
  void* y; int64_t ldy; int y_f32;
  const float* bias;
  const void* add; int64_t ldadd; int add_f32;
  int tile0;                     // first column tile of this problem within a row block
};
struct GemmGroup { GemmProb p[3]; int np, tiles_n, M; };

// 64 x 64 tile per workgroup, 64-wide K chunks through LDS with the next in flight, across the segments.  Tiles that
// share rows of X run on one XCD (workgroups are dealt to the 8 XCDs in turn).
__global__ void __launch_bounds__(256) block_gemm_kernel(GemmGroup gg) {
  __shared__ __align__(16) uint16_t As[64 * BK_LD];
  __shared__ __align__(16) uint16_t Bs[64 * BK_LD];
  const int total = gg.tiles_n * ((gg.M + 63) / 64), per = (total + 7) / 8;
  const int tile = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per || tile >= total) return;   // the whole workgroup, before any barrier
  const int tm = tile / gg.tiles_n, tn = tile % gg.tiles_n;
  int pi = 0;
  while (pi + 1 < gg.np && tn >= gg.p[pi + 1].tile0) ++pi;
  const GemmProb& P = gg.p[pi];
  const int m0 = tm * 64, n0 = (tn - P.tile0) * 64, M = gg.M, N = P.N;
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6, g = lane >> 4, li = lane & 15;
  const int wr = wid >> 1, wc = wid & 1;
  uint4 ra[2], rb[2];
  auto fetch = [&](int s, int k0) {
    const GemmSeg& S = P.seg[s];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int u = tid + 256 * i, kc = k0 + (u & 7) * 8;
      int r = m0 + (u >> 3), c = n0 + (u >> 3);
      r = r < M ? r : M - 1;
      c = c < N ? c : N - 1;
      const bool in = kc < S.K;                    // K % 8 == 0
      const int kk = in ? kc : 0;
      if (S.x_f32) {
        const float4* xp = reinterpret_cast<const float4*>(reinterpret_cast<const float*>(S.x) + (int64_t)r * S.ldx + kk);
        const float4 a = xp[0], b = xp[1];
        ra[i] = make_uint4(pack_bf16x2(a.x, a.y), pack_bf16x2(a.z, a.w), pack_bf16x2(b.x, b.y), pack_bf16x2(b.z, b.w));
      } else {
        ra[i] = *reinterpret_cast<const uint4*>(reinterpret_cast<const uint16_t*>(S.x) + (int64_t)r * S.ldx + kk);
      }
      rb[i] = *reinterpret_cast<const uint4*>(S.w + (int64_t)c * S.ldw + kk);
      if (!in) ra[i] = rb[i] = make_uint4(0, 0, 0, 0);
    }
  };
  f32x4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  int s = 0, k0 = 0;
  fetch(0, 0);
  while (true) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int u = tid + 256 * i, o = (u >> 3) * BK_LD + (u & 7) * 8;
      *reinterpret_cast<uint4*>(As + o) = ra[i];
      *reinterpret_cast<uint4*>(Bs + o) = rb[i];
    }
    __syncthreads();
    k0 += 64;
    if (k0 >= P.seg[s].K) { ++s; k0 = 0; }
    const bool more = s < P.nseg;
    if (more) fetch(s, k0);
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      bf16x8_t a[2], b[2];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        a[t] = MM<HCLSM_BF16>::load(As + (wr * 32 + 16 * t + li) * BK_LD + kk * 32 + 8 * g);
        b[t] = MM<HCLSM_BF16>::load(Bs + (wc * 32 + 16 * t + li) * BK_LD + kk * 32 + 8 * g);
      }
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = MM<HCLSM_BF16>::mfma(b[j], a[i], acc[i][j]);   // weights as A operand
    }
    if (!more) break;
  }
  // lane: row 16 i + li, columns 16 j + 4 g .. + 3
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int col = n0 + wc * 32 + 16 * j + 4 * g;
    if (col >= N) continue;                        // N % 4 == 0
    float4 bv = make_float4(0.f, 0.f, 0.f, 0.f);
    if (P.bias) {                                  // rounded to 16 bits, as the autocast linear's
      auto rnd = [](float v) { return bf16_bits_to_f32(f32_to_bf16_bits(v)); };
      bv = make_float4(rnd(P.bias[col]), rnd(P.bias[col + 1]), rnd(P.bias[col + 2]), rnd(P.bias[col + 3]));
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int row = m0 + wr * 32 + 16 * i + li;
      if (row >= M) continue;
      float v[4] = {acc[i][j][0] + bv.x, acc[i][j][1] + bv.y, acc[i][j][2] + bv.z, acc[i][j][3] + bv.w};
      if (P.add) {
        if (P.add_f32) {
          const float4 a = *reinterpret_cast<const float4*>(reinterpret_cast<const float*>(P.add) + (int64_t)row * P.ldadd + col);
          v[0] += a.x; v[1] += a.y; v[2] += a.z; v[3] += a.w;
        } else {
          const uint2 a = *reinterpret_cast<const uint2*>(reinterpret_cast<const uint16_t*>(P.add) + (int64_t)row * P.ldadd + col);
          v[0] += __uint_as_float(a.x << 16); v[1] += __uint_as_float(a.x & 0xffff0000u);
          v[2] += __uint_as_float(a.y << 16); v[3] += __uint_as_float(a.y & 0xffff0000u);
        }
      }
      if (P.y_f32)
        *reinterpret_cast<float4*>(reinterpret_cast<float*>(P.y) + (int64_t)row * P.ldy + col) = make_float4(v[0], v[1], v[2], v[3]);
      else
        *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(P.y) + (int64_t)row * P.ldy + col) =
            make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
    }
  }
}

// --------------------------------------------------------------------------------------- weight gradients
// gW[N, K] = sum over rows of G[row, N] X[row, K] (G 16-bit or fp32, rounded; X 16-bit), split over row
// ranges: part[split][off + n * K + k].  bias_off >= 0: also the column sums of G at part[split][bias_off + n].
struct WgProb { const void* g; int64_t ldg; int g_f32, N; const uint16_t* x; int64_t ldx; int K, tiles_x; int64_t off, bias_off; int tile0; };
struct WgGroup { WgProb p[6]; int np; int M, rows_per, splits; int64_t part_ld; float* part; };

// 64 x 64 tile of one gradient per workgroup.  Both operands are needed with the row index fastest: a thread loads 8
// rows x 2 columns as words, interleaves them into two 8-row vectors (8 v_perm_b32) and writes those to LDS.
__global__ void __launch_bounds__(256) block_wgrad_kernel(WgGroup wg) {
  __shared__ __align__(16) uint16_t Gs[64 * BK_LD];
  __shared__ __align__(16) uint16_t Xs[64 * BK_LD];
  __shared__ float bsum[4][64];
  const int tile = (int)blockIdx.x / wg.splits, split = (int)blockIdx.x - tile * wg.splits;
  int pi = 0;
  while (pi + 1 < wg.np && tile >= wg.p[pi + 1].tile0) ++pi;
  const WgProb& P = wg.p[pi];
  const int t = tile - P.tile0, n0 = t / P.tiles_x * 64, k0 = t % P.tiles_x * 64;
  const int r_begin = split * wg.rows_per;
  const int r_end = r_begin + wg.rows_per < wg.M ? r_begin + wg.rows_per : wg.M;
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6, g = lane >> 4, li = lane & 15;
  const int wr = wid >> 1, wc = wid & 1;
  const bool is_g = tid < 128;                     // threads 0..127 stage G, the others X
  const int cp = tid & 31, oct = (tid >> 5) & 3;   // columns 2 cp, 2 cp + 1; rows 8 oct .. and 32 + 8 oct ..
  const int col = (is_g ? n0 : k0) + 2 * cp;
  const bool col_in = col < (is_g ? P.N : P.K);    // both even
  const bool want_bias = P.bias_off >= 0 && k0 == 0 && is_g;
  uint32_t w[2][8];
  float b0 = 0.f, b1 = 0.f;
  // this thread's operand, one branch per chunk (a wave stages one operand): 16 loads in flight
  const bool f32 = __builtin_amdgcn_readfirstlane(is_g && P.g_f32) != 0;
  const int64_t ldr = is_g ? P.ldg : P.ldx;
  const uint16_t* p16 = (is_g ? reinterpret_cast<const uint16_t*>(P.g) : P.x) + (col_in ? col : 0);
  const float* p32 = reinterpret_cast<const float*>(P.g) + (col_in ? col : 0);
  auto fetch = [&](int r0) {
    int64_t ro[2][8];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int r = r0 + 32 * h + 8 * oct + e;
        ro[h][e] = (int64_t)(r < r_end ? r : r_end - 1) * ldr;
      }
    if (f32) {
      float2 f[2][8];
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int e = 0; e < 8; ++e) f[h][e] = *reinterpret_cast<const float2*>(p32 + ro[h][e]);
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int e = 0; e < 8; ++e) w[h][e] = pack_bf16x2(f[h][e].x, f[h][e].y);
    } else {
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int e = 0; e < 8; ++e) w[h][e] = *reinterpret_cast<const uint32_t*>(p16 + ro[h][e]);
    }
  };
  auto zero_tail = [&](int r0) {   // rows past the range and columns past the matrix contribute nothing
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (!col_in || r0 + 32 * h + 8 * oct + e >= r_end) w[h][e] = 0u;
  };
  f32x4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  fetch(r_begin);
  for (int r0 = r_begin; r0 < r_end; r0 += 64) {
    __syncthreads();
    zero_tail(r0);
    uint16_t* dst = (is_g ? Gs : Xs) + 2 * cp * BK_LD + 8 * oct;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      uint32_t lo[4], hi[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        lo[q] = __builtin_amdgcn_perm(w[h][2 * q + 1], w[h][2 * q], 0x05040100);
        hi[q] = __builtin_amdgcn_perm(w[h][2 * q + 1], w[h][2 * q], 0x07060302);
      }
      *reinterpret_cast<uint4*>(dst + 32 * h) = make_uint4(lo[0], lo[1], lo[2], lo[3]);
      *reinterpret_cast<uint4*>(dst + BK_LD + 32 * h) = make_uint4(hi[0], hi[1], hi[2], hi[3]);
    }
    if (want_bias)
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          b0 += __uint_as_float(w[h][e] << 16);
          b1 += __uint_as_float(w[h][e] & 0xffff0000u);
        }
    __syncthreads();
    if (r0 + 64 < r_end) fetch(r0 + 64);
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      bf16x8_t a[2], b[2];
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        a[q] = MM<HCLSM_BF16>::load(Gs + (wr * 32 + 16 * q + li) * BK_LD + kk * 32 + 8 * g);
        b[q] = MM<HCLSM_BF16>::load(Xs + (wc * 32 + 16 * q + li) * BK_LD + kk * 32 + 8 * g);
      }
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = MM<HCLSM_BF16>::mfma(b[j], a[i], acc[i][j]);   // X columns as rows
    }
  }
  float* part = wg.part + split * wg.part_ld;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int n = n0 + wr * 32 + 16 * i + li;
    if (n >= P.N) continue;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int k = k0 + wc * 32 + 16 * j + 4 * g;
      if (k < P.K)                                 // K % 4 == 0
        *reinterpret_cast<float4*>(part + P.off + (int64_t)n * P.K + k) =
            make_float4(acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]);
    }
  }
  if (P.bias_off >= 0 && k0 == 0) {                // uniform over the workgroup
    if (is_g) { bsum[oct][2 * cp] = b0; bsum[oct][2 * cp + 1] = b1; }
    __syncthreads();
    if (tid < 64 && n0 + tid < P.N) part[P.bias_off + n0 + tid] = bsum[0][tid] + bsum[1][tid] + bsum[2][tid] + bsum[3][tid];
  }
}

struct RedSeg { const float* src; int64_t ld; int n; float* dst; int cnt, blk0; };
struct RedGroup { RedSeg s[9]; int ns; };

// dst[i] = sum over k < n of src[k * ld + i]: 64 columns x 4 row groups per workgroup, added in a fixed order.
__global__ void __launch_bounds__(256) block_reduce_kernel(RedGroup rg) {
  __shared__ float red[4][64];
  int k = 0;
  while (k + 1 < rg.ns && (int)blockIdx.x >= rg.s[k + 1].blk0) ++k;
  const RedSeg S = rg.s[k];
  const int c = threadIdx.x & 63, q = threadIdx.x >> 6;
  const int i = ((int)blockIdx.x - S.blk0) * 64 + c;
  float acc = 0.f;
  if (i < S.cnt) {
#pragma unroll 8
    for (int r = q; r < S.n; r += 4) acc += S.src[r * S.ld + i];
  }
  red[q][c] = acc;
  __syncthreads();
  if (q == 0 && i < S.cnt) S.dst[i] = (red[0][c] + red[1][c]) + (red[2][c] + red[3][c]);
}

// ------------------------------------------------------------------------------------ LayerNorm, backward
constexpr int LB_Q = 4;        // float4 units per lane: rows of up to 1024
// gx = g + LN'(gu) (gx nullable); per workgroup the partial sums of ggamma = sum gu xhat and gbeta = sum gu: part[block][2][D].
__global__ void __launch_bounds__(256)
block_ln_bwd_kernel(const float* __restrict__ x, const float* __restrict__ gu, const float* __restrict__ g,
                    const float* __restrict__ gamma, float* __restrict__ gx, float* __restrict__ part, int M, int D,
                    float eps) {
  __shared__ float red[4][1024];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nu = D / 4;
  float4 gm[LB_Q], sg[LB_Q], sb[LB_Q];
#pragma unroll
  for (int q = 0; q < LB_Q; ++q) {
    const int u = lane + 64 * q;
    gm[q] = u < nu ? reinterpret_cast<const float4*>(gamma)[u] : make_float4(0.f, 0.f, 0.f, 0.f);
    sg[q] = sb[q] = make_float4(0.f, 0.f, 0.f, 0.f);
  }
  const float inv = 1.f / (float)D;
  auto wsum = [](float v) {
#pragma unroll
    for (int m = 1; m < 16; m <<= 1) v += __shfl_xor(v, m, 64);
    return rows4_sum(v);
  };
  for (int row = blockIdx.x * 4 + wid; row < M; row += gridDim.x * 4) {
    const float4* xp = reinterpret_cast<const float4*>(x + (int64_t)row * D);
    const float4* up = reinterpret_cast<const float4*>(gu + (int64_t)row * D);
    const float4* gp = reinterpret_cast<const float4*>(g + (int64_t)row * D);
    float4 xv[LB_Q], uv[LB_Q], gv[LB_Q];
    float s = 0.f;
#pragma unroll
    for (int q = 0; q < LB_Q; ++q) {
      const int u = lane + 64 * q;
      const bool in = u < nu;
      xv[q] = in ? xp[u] : make_float4(0.f, 0.f, 0.f, 0.f);
      uv[q] = in ? up[u] : make_float4(0.f, 0.f, 0.f, 0.f);
      gv[q] = in ? gp[u] : make_float4(0.f, 0.f, 0.f, 0.f);
      s += (xv[q].x + xv[q].y) + (xv[q].z + xv[q].w);
    }
    const float mean = wsum(s) * inv;
    float v = 0.f;
#pragma unroll
    for (int q = 0; q < LB_Q; ++q) {
      const bool in = lane + 64 * q < nu;
      xv[q].x = in ? xv[q].x - mean : 0.f; xv[q].y = in ? xv[q].y - mean : 0.f;
      xv[q].z = in ? xv[q].z - mean : 0.f; xv[q].w = in ? xv[q].w - mean : 0.f;
      v += (xv[q].x * xv[q].x + xv[q].y * xv[q].y) + (xv[q].z * xv[q].z + xv[q].w * xv[q].w);
    }
    const float rstd = 1.f / sqrtf(wsum(v) * inv + eps);
    float a = 0.f, b = 0.f;     // sums of gu gamma and of gu gamma xhat
#pragma unroll
    for (int q = 0; q < LB_Q; ++q) {
      xv[q].x *= rstd; xv[q].y *= rstd; xv[q].z *= rstd; xv[q].w *= rstd;
      sg[q].x += uv[q].x * xv[q].x; sg[q].y += uv[q].y * xv[q].y; sg[q].z += uv[q].z * xv[q].z; sg[q].w += uv[q].w * xv[q].w;
      sb[q].x += uv[q].x; sb[q].y += uv[q].y; sb[q].z += uv[q].z; sb[q].w += uv[q].w;
      uv[q].x *= gm[q].x; uv[q].y *= gm[q].y; uv[q].z *= gm[q].z; uv[q].w *= gm[q].w;
      a += (uv[q].x + uv[q].y) + (uv[q].z + uv[q].w);
      b += (uv[q].x * xv[q].x + uv[q].y * xv[q].y) + (uv[q].z * xv[q].z + uv[q].w * xv[q].w);
    }
    a = wsum(a) * inv;
    b = wsum(b) * inv;
    float4* op = reinterpret_cast<float4*>(gx + (int64_t)row * D);
#pragma unroll
    for (int q = 0; q < LB_Q; ++q) {
      const int u = lane + 64 * q;
      if (u < nu && gx != nullptr)
        op[u] = make_float4(gv[q].x + rstd * (uv[q].x - a - xv[q].x * b), gv[q].y + rstd * (uv[q].y - a - xv[q].y * b),
                            gv[q].z + rstd * (uv[q].z - a - xv[q].z * b), gv[q].w + rstd * (uv[q].w - a - xv[q].w * b));
    }
  }
#pragma unroll
  for (int which = 0; which < 2; ++which) {
    if (which) __syncthreads();
#pragma unroll
    for (int q = 0; q < LB_Q; ++q)
      if (lane + 64 * q < nu) reinterpret_cast<float4*>(red[wid])[lane + 64 * q] = which ? sb[q] : sg[q];
    __syncthreads();
    for (int i = threadIdx.x; i < D; i += 256)
      part[((int64_t)blockIdx.x * 2 + which) * D + i] = (red[0][i] + red[1][i]) + (red[2][i] + red[3][i]);
  }
}

// The gate's chain rule where the scan's backward does not take it (d_state 16): g_scan = gy silu(gate),
// g_gate = gy y_pre silu'(gate).  Pairs of 16-bit elements.
__global__ void __launch_bounds__(256)
block_gate_bwd_kernel(const uint32_t* __restrict__ gy, const uint32_t* __restrict__ gate, const uint32_t* __restrict__ yp,
                      uint32_t* __restrict__ g_scan, uint32_t* __restrict__ g_gate, int64_t n2) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n2; i += (int64_t)gridDim.x * 256) {
    const uint32_t a = gy[i], b = gate[i], c = yp[i];
    float o[2], h[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const float gv = __uint_as_float(k ? a & 0xffff0000u : a << 16), t = __uint_as_float(k ? b & 0xffff0000u : b << 16);
      const float y = __uint_as_float(k ? c & 0xffff0000u : c << 16), sg = __builtin_amdgcn_rcpf(1.f + __expf(-t));
      o[k] = gv * t * sg;
      h[k] = gv * y * sg * fmaf(t, 1.f - sg, 1.f);
    }
    g_scan[i] = pack_bf16x2(o[0], o[1]);
    g_gate[i] = pack_bf16x2(h[0], h[1]);
  }
}

// --------------------------------------------------------------------------------------------- layouts
struct BlkLayout {   // byte offsets; save: what the backward reads, scratch: the backward's own
  size_t u, z, gate, dt, b, c, y, y_pre, w, wt, ck, save;
  size_t gy, gys, gz0, gdt, gbc, gg, gz, gu, part, lnp, ga, scan, scratch;
  int64_t R, part_ld;
  int splits, rows_per, ln_blocks;
  bool group, pair16;
};

constexpr size_t up256(size_t v) { return (v + 255) / 256 * 256; }

static int blk_layout(int64_t N, int64_t T, int64_t d, int64_t di, int64_t S, bool train, BlkLayout* L) {
  if (N < 1 || T < 1 || d < 8 || di < 8 || S < 16) return HCLSM_ERR_UNSUPPORTED;
  if (d % 8 || di % 8 || S % 8 || d > 256 * LB_Q || di > 4096 || S > 128) return HCLSM_ERR_UNSUPPORTED;
  const int64_t R = N * T;
  if (R > (1LL << 24) || R * di >= (1LL << 30)) return HCLSM_ERR_UNSUPPORTED;
  L->R = R;
  L->group = bwd_group_ok(T, di, S, HCLSM_BF16);
  L->pair16 = S == 16;
  if (!L->group && !L->pair16) return HCLSM_ERR_UNSUPPORTED;
  size_t o = 0;
  auto take = [&](size_t bytes) { const size_t at = o; o += up256(bytes); return at; };
  const int64_t nw = 2 * di * d + di * di + 2 * S * di + d * di;
  L->u = take(R * d * 2); L->z = take(R * di * 2); L->gate = take(R * di * 2); L->dt = take(R * di * 2);
  L->b = take(R * S * 2); L->c = take(R * S * 2); L->y = take(R * di * 2);
  L->y_pre = take(train ? R * di * 2 : 0);
  L->w = take(nw * 2);
  L->wt = take(train ? nw * 2 : 0);
  const int64_t scan_ws = hclsm_ssm_scan_bwd_workspace(N, T, di, S);
  if (scan_ws < 0) return (int)scan_ws;
  const int64_t ck_bytes = L->pair16 ? scan_bwd_ck_bytes(N, T, di, S) : 0;   // the forward leaves the scan's checkpoints
  L->ck = take(train ? ck_bytes : 0);
  L->save = o;
  o = 0;
  L->gy = take(R * di * 2); L->gys = take(L->group ? 0 : R * di * 2); L->gz0 = take(R * di * 2); L->gdt = take(R * di * 2);
  L->gbc = take(2 * up256(R * S * 2)); L->gg = take(R * di * 2); L->gz = take(R * di * 2); L->gu = take(R * d * 4);
  L->part_ld = nw + di;
  // row ranges of the weight gradients: at least 512 rows each, up to 16 (8: 72 us, 16: 63 us at 16384
  // rows of a 192-wide block); splits are dealt to the XCDs in turn, so the tiles of a row range share one L2
  int sp = (int)(R / 512);
  sp = sp < 1 ? 1 : sp > 16 ? 16 : sp;
  L->rows_per = (int)(((R + sp - 1) / sp + 63) / 64 * 64);
  L->splits = (int)((R + L->rows_per - 1) / L->rows_per);
  L->part = take((size_t)L->splits * L->part_ld * 4);
  L->ln_blocks = (int)((R + 15) / 16 < 256 ? (R + 15) / 16 : 256);
  L->lnp = take((size_t)L->ln_blocks * 2 * d * 4);
  L->ga = take(di * S * 4);
  L->scan = take(scan_ws - ck_bytes);
  L->scratch = o;
  return 0;
}

template <typename U>
struct BlkW {   // 16-bit weights and their transposes inside the save buffer
  U *in, *gate, *dt, *b, *c, *out, *in_t, *gate_t, *dt_t, *bc_t, *out_t;
};
template <typename U, typename Byte>
static BlkW<U> blk_weights(Byte* save, const BlkLayout& L, int64_t d, int64_t di, int64_t S) {
  BlkW<U> w;
  U* p = reinterpret_cast<U*>(save + L.w);
  w.in = p; p += di * d; w.gate = p; p += di * d; w.dt = p; p += di * di; w.b = p; p += S * di; w.c = p; p += S * di; w.out = p;
  p = reinterpret_cast<U*>(save + L.wt);
  w.in_t = p; p += di * d; w.gate_t = p; p += di * d; w.dt_t = p; p += di * di; w.bc_t = p; p += 2 * S * di; w.out_t = p;
  return w;
}

static GemmProb prob(int64_t N, void* y, int64_t ldy, int y_f32) {
  GemmProb p = {};
  p.N = (int)N; p.y = y; p.ldy = ldy; p.y_f32 = y_f32;
  return p;
}
static void add_seg(GemmProb& p, const void* x, int64_t ldx, const uint16_t* w, int64_t ldw, int64_t K, int x_f32 = 0) {
  p.seg[p.nseg++] = GemmSeg{x, ldx, w, ldw, (int)K, x_f32};
}
static int run_gemm(GemmGroup& g, int64_t M, hipStream_t st) {
  g.M = (int)M;
  int t = 0;
  for (int i = 0; i < g.np; ++i) { g.p[i].tile0 = t; t += (g.p[i].N + 63) / 64; }
  g.tiles_n = t;
  const int64_t total = t * ((M + 63) / 64);
  hipLaunchKernelGGL(block_gemm_kernel, dim3((unsigned)((total + 7) / 8 * 8)), dim3(256), 0, st, g);
  HCLSM_LAUNCH_CHECK();
  return 0;
}

static bool al16p(const void* p) { return ((uintptr_t)p & 15) == 0; }
static int blk_check(const HclsmBlockParams* P, const void* x, const void* o) {
  if (!P || !x || !o || !P->ln_w || !P->ln_b || !P->w_in || !P->w_gate || !P->w_dt || !P->b_dt || !P->w_b || !P->w_c ||
      !P->a_log || !P->w_out)
    return HCLSM_ERR_NULL;
  if (!al16p(x) || !al16p(o) || !al16p(P->ln_w) || !al16p(P->ln_b) || !al16p(P->a_log)) return HCLSM_ERR_UNSUPPORTED;
  return 0;
}

}  // namespace hclsm

using namespace hclsm;

extern "C" int64_t hclsm_ssm_block_save(int64_t batch, int64_t T, int64_t d_model, int64_t d_inner, int64_t d_state,
                                        int train) {
  BlkLayout L;
  const int rc = blk_layout(batch, T, d_model, d_inner, d_state, train != 0, &L);
  return rc ? rc : (int64_t)L.save;
}
extern "C" int64_t hclsm_ssm_block_scratch(int64_t batch, int64_t T, int64_t d_model, int64_t d_inner, int64_t d_state) {
  BlkLayout L;
  const int rc = blk_layout(batch, T, d_model, d_inner, d_state, true, &L);
  return rc ? rc : (int64_t)L.scratch;
}

extern "C" int hclsm_ssm_block_forward(const HclsmBlockParams* P, const float* x, float* out, int64_t batch, int64_t T,
                                       int64_t d, int64_t di, int64_t S, int train, void* save, int64_t save_bytes,
                                       void* stream) {
  BlkLayout L;
  int rc = blk_layout(batch, T, d, di, S, train != 0, &L);
  if (rc) return rc;
  if ((rc = blk_check(P, x, out))) return rc;
  if (!save) return HCLSM_ERR_NULL;
  if (save_bytes < (int64_t)L.save) return HCLSM_ERR_SHAPE;
  if (((uintptr_t)save & 255) != 0) return HCLSM_ERR_UNSUPPORTED;
  hipStream_t st = (hipStream_t)stream;
  char* s = reinterpret_cast<char*>(save);
  const BlkW<uint16_t> w = blk_weights<uint16_t>(s, L, d, di, S);
  CastJobs js = {};
  auto job = [&](const float* src, uint16_t* dst, uint16_t* dst_t, int64_t rows, int64_t cols, int64_t ld_t) {
    const int b0 = js.n ? js.j[js.n - 1].blk0 + ((js.j[js.n - 1].rows + 31) / 32) * ((js.j[js.n - 1].cols + 31) / 32) : 0;
    js.j[js.n++] = CastJob{src, dst, train ? dst_t : nullptr, (int)rows, (int)cols, ld_t, b0};
    return b0 + (int)(((rows + 31) / 32) * ((cols + 31) / 32));
  };
  job(P->w_in, w.in, w.in_t, di, d, di);
  job(P->w_gate, w.gate, w.gate_t, di, d, di);
  job(P->w_dt, w.dt, w.dt_t, di, di, di);
  job(P->w_b, w.b, w.bc_t, S, di, 2 * S);          // [W_B; W_C]^T: di rows of 2 S
  job(P->w_c, w.c, w.bc_t + S, S, di, 2 * S);
  const int nb = job(P->w_out, w.out, w.out_t, d, di, d);
  hipLaunchKernelGGL(block_cast_kernel, dim3((unsigned)nb), dim3(256), 0, st, js);
  HCLSM_LAUNCH_CHECK();
  rc = layer_norm_rows(x, d, P->ln_w, P->ln_b, s + L.u, d, L.R, d, 1e-5f, HCLSM_F32, HCLSM_BF16, nullptr, 0, st);
  if (rc) return rc;
  GemmGroup g = {};
  g.np = 2;
  g.p[0] = prob(di, s + L.z, di, 0);
  add_seg(g.p[0], s + L.u, d, w.in, d, d);
  g.p[1] = prob(di, s + L.gate, di, 0);
  add_seg(g.p[1], s + L.u, d, w.gate, d, d);
  if ((rc = run_gemm(g, L.R, st))) return rc;
  g = {};
  g.np = 3;
  g.p[0] = prob(di, s + L.dt, di, 0);
  add_seg(g.p[0], s + L.z, di, w.dt, di, di);
  g.p[0].bias = P->b_dt;
  g.p[1] = prob(S, s + L.b, S, 0);
  add_seg(g.p[1], s + L.z, di, w.b, di, di);
  g.p[2] = prob(S, s + L.c, S, 0);
  add_seg(g.p[2], s + L.z, di, w.c, di, di);
  if ((rc = run_gemm(g, L.R, st))) return rc;
  void* y_pre = train ? s + L.y_pre : nullptr;
  if (train && L.pair16)
    rc = scan_fwd_ckpt(SCAN_BLOCK, s + L.z, s + L.dt, P->a_log, s + L.b, s + L.c, nullptr, s + L.y, nullptr, batch, T, di,
                       S, HCLSM_BF16, s + L.gate, y_pre, reinterpret_cast<float*>(s + L.ck), st);
  else
    rc = hclsm_ssm_block_scan_fwd(s + L.z, s + L.dt, P->a_log, s + L.b, s + L.c, s + L.gate, s + L.y, y_pre, nullptr,
                                  batch, T, di, S, HCLSM_BF16, stream);
  if (rc) return rc;
  g = {};
  g.np = 1;
  g.p[0] = prob(d, out, d, 1);
  add_seg(g.p[0], s + L.y, di, w.out, di, di);
  g.p[0].add = x; g.p[0].ldadd = d; g.p[0].add_f32 = 1;
  return run_gemm(g, L.R, st);
}

extern "C" int hclsm_ssm_block_backward(const HclsmBlockParams* P, const float* x, const float* g, float* gx,
                                        const HclsmBlockGrads* G, int64_t batch, int64_t T, int64_t d, int64_t di,
                                        int64_t S, const void* save, int64_t save_bytes, void* scratch,
                                        int64_t scratch_bytes, void* stream) {
  BlkLayout L;
  int rc = blk_layout(batch, T, d, di, S, true, &L);
  if (rc) return rc;
  if (!P || !P->ln_w || !P->a_log || !x || !g || !G || !save || !scratch) return HCLSM_ERR_NULL;
  if (save_bytes < (int64_t)L.save || scratch_bytes < (int64_t)L.scratch) return HCLSM_ERR_SHAPE;
  if (((uintptr_t)save & 255) || ((uintptr_t)scratch & 255) || !al16p(x) || !al16p(g) || !al16p(gx) || !al16p(P->ln_w) ||
      !al16p(P->a_log))
    return HCLSM_ERR_UNSUPPORTED;
  // what the wanted gradients need: gu (the LayerNorm's), gz, the scan's backward
  const bool need_u = gx || G->ln_w || G->ln_b, need_z = need_u || G->w_in;
  const bool need_scan = need_z || G->w_gate || G->w_dt || G->b_dt || G->w_b || G->w_c || G->a_log;
  float* gA = G->a_log ? G->a_log : reinterpret_cast<float*>(reinterpret_cast<char*>(scratch) + L.ga);
  hipStream_t st = (hipStream_t)stream;
  const char* s = reinterpret_cast<const char*>(save);
  char* q = reinterpret_cast<char*>(scratch);
  const BlkW<const uint16_t> w = blk_weights<const uint16_t>(s, L, d, di, S);
  uint16_t* gB = reinterpret_cast<uint16_t*>(q + L.gbc);
  uint16_t* gC = reinterpret_cast<uint16_t*>(q + L.gbc + up256(L.R * S * 2));
  GemmGroup gg = {};
  if (need_scan) {
    gg.np = 1;
    gg.p[0] = prob(di, q + L.gy, di, 0);
    add_seg(gg.p[0], g, d, w.out_t, d, d, 1);
    if ((rc = run_gemm(gg, L.R, st))) return rc;
    if (L.group) {
      BwdGate gate;
      gate.gate = s + L.gate; gate.y_pre = s + L.y_pre; gate.g_gate = q + L.gg;
      rc = scan_bwd_block(s + L.z, s + L.dt, P->a_log, s + L.b, s + L.c, q + L.gy, q + L.gz0, q + L.gdt, gA, gB, gC,
                          batch, T, di, S, HCLSM_BF16, gate, nullptr, q + L.scan, (int64_t)(L.scratch - L.scan), st);
    } else {
      const int64_t n2 = L.R * di / 2;
      const int64_t nb = (n2 + 255) / 256;
      hipLaunchKernelGGL(block_gate_bwd_kernel, dim3((unsigned)(nb < 4096 ? nb : 4096)), dim3(256), 0, st,
                         (const uint32_t*)(q + L.gy), (const uint32_t*)(s + L.gate), (const uint32_t*)(s + L.y_pre),
                         (uint32_t*)(q + L.gys), (uint32_t*)(q + L.gg), n2);
      HCLSM_LAUNCH_CHECK();
      rc = scan_bwd_block(s + L.z, s + L.dt, P->a_log, s + L.b, s + L.c, q + L.gys, q + L.gz0, q + L.gdt, gA, gB, gC,
                          batch, T, di, S, HCLSM_BF16, BwdGate(), reinterpret_cast<const float*>(s + L.ck), q + L.scan,
                          (int64_t)(L.scratch - L.scan), st);
    }
    if (rc) return rc;
  }
  if (need_z) {
    gg = {};
    gg.np = 1;
    gg.p[0] = prob(di, q + L.gz, di, 0);
    add_seg(gg.p[0], q + L.gdt, di, w.dt_t, di, di);
    add_seg(gg.p[0], gB, S, w.bc_t, 2 * S, S);
    add_seg(gg.p[0], gC, S, w.bc_t + S, 2 * S, S);
    gg.p[0].add = q + L.gz0; gg.p[0].ldadd = di;
    if ((rc = run_gemm(gg, L.R, st))) return rc;
  }
  float* lnp = reinterpret_cast<float*>(q + L.lnp);
  if (need_u) {
    gg = {};
    gg.np = 1;
    gg.p[0] = prob(d, q + L.gu, d, 1);
    add_seg(gg.p[0], q + L.gz, di, w.in_t, di, di);
    add_seg(gg.p[0], q + L.gg, di, w.gate_t, di, di);
    if ((rc = run_gemm(gg, L.R, st))) return rc;
    hipLaunchKernelGGL(block_ln_bwd_kernel, dim3((unsigned)L.ln_blocks), dim3(256), 0, st, x, (const float*)(q + L.gu), g,
                       P->ln_w, gx, lnp, (int)L.R, (int)d, 1e-5f);
    HCLSM_LAUNCH_CHECK();
  }
  // weight gradients: those that are wanted (the bias's alone: the first column tile of its matrix)
  WgGroup wg = {};
  wg.M = (int)L.R; wg.rows_per = L.rows_per; wg.splits = L.splits; wg.part_ld = L.part_ld;
  wg.part = reinterpret_cast<float*>(q + L.part);
  RedGroup rg = {};
  int tiles = 0, rblk = 0;
  int64_t off = 0;
  auto red = [&](const float* src, int64_t ld, int n, float* dst, int64_t cnt) {
    if (!dst) return;
    rg.s[rg.ns++] = RedSeg{src, ld, n, dst, (int)cnt, rblk};
    rblk += (int)((cnt + 63) / 64);
  };
  auto wgrad = [&](const void* ga, int64_t N, int g_f32, const void* xa, int64_t K, float* dst, float* bias) {
    if (dst || bias) {
      const int tx = dst ? (int)((K + 63) / 64) : 1;
      wg.p[wg.np++] = WgProb{ga, N, g_f32, (int)N, (const uint16_t*)xa, K, (int)K, tx, off, bias ? L.part_ld - di : -1, tiles};
      tiles += tx * (int)((N + 63) / 64);
      red(wg.part + off, L.part_ld, L.splits, dst, N * K);
      red(wg.part + L.part_ld - di, L.part_ld, L.splits, bias, N);
    }
    off += N * K;
  };
  wgrad(q + L.gdt, di, 0, s + L.z, di, G->w_dt, G->b_dt);
  wgrad(q + L.gz, di, 0, s + L.u, d, G->w_in, nullptr);
  wgrad(q + L.gg, di, 0, s + L.u, d, G->w_gate, nullptr);
  wgrad(g, d, 1, s + L.y, di, G->w_out, nullptr);
  wgrad(gB, S, 0, s + L.z, di, G->w_b, nullptr);
  wgrad(gC, S, 0, s + L.z, di, G->w_c, nullptr);
  red(lnp, 2 * d, L.ln_blocks, G->ln_w, d);
  red(lnp + d, 2 * d, L.ln_blocks, G->ln_b, d);
  if (wg.np) {
    hipLaunchKernelGGL(block_wgrad_kernel, dim3((unsigned)(tiles * L.splits)), dim3(256), 0, st, wg);
    HCLSM_LAUNCH_CHECK();
  }
  if (rg.ns) {
    hipLaunchKernelGGL(block_reduce_kernel, dim3((unsigned)rblk), dim3(256), 0, st, rg);
    HCLSM_LAUNCH_CHECK();
  }
  return 0;
}
