// The state-group backward scan (ssm_scan_bwd_group.hip), as the entry points of ssm_scan_bwd.hip call it.
#pragma once

#include "common.h"

namespace hclsm {

constexpr int BG_WINDOW = 16;   // steps between the states kept in memory
// HCLSM_SCAN_BLOCK with the output gate's chain rule in the kernel: gy is the gradient of silu(gate) * y.
constexpr int BWD_BLOCK_GATE = HCLSM_SCAN_BLOCK + 1;
struct BwdGate {
  const void* gate = nullptr;    // [batch][T][d_inner], I/O type
  const void* y_pre = nullptr;   // the scan output before gating
  void* g_gate = nullptr;        // gradient of gate
};

// Whether the kernel takes these arguments.
bool bwd_group_ok(int64_t T, int64_t Dn, int64_t S, int dtype);
// Launches it; *parts gets the number of gA / gD partials written ([parts][S][Dn] and [parts][Dn], at most N).
// ck: (ceil(T / BG_WINDOW) - 1) * S * Dn floats per sequence; gbc: [ceil(Dn / 64)][N * T][2 S].
int bwd_group(int mode, const void* x, const void* dt, const float* A_log, const void* B, const void* C,
              const float* Dskip, const void* gy, void* gx, void* gdt, BwdGate gate, float* ck, float* gbc, float* ga,
              float* gd, int64_t N, int64_t T, int64_t Dn, int64_t S, int dtype, int* parts, hipStream_t st);

// The block-mode backward as composite entry points call it (ssm_scan_bwd.hip): with gate set, gy is the gradient of the
// gated output (shapes of bwd_group_ok).  ck (nullable): the checkpointing forward's states, scan_bwd_ck_bytes of them, only
// read; ws then holds the partial sums alone, hclsm_ssm_scan_bwd_workspace - scan_bwd_ck_bytes.
int64_t scan_bwd_ck_bytes(int64_t batch, int64_t T, int64_t d_inner, int64_t d_state);
int scan_bwd_block(const void* z, const void* dt_in, const float* A_log, const void* B, const void* C, const void* gy,
                   void* gz, void* gdt, float* gA_log, void* gB, void* gC, int64_t batch, int64_t T, int64_t d_inner,
                   int64_t d_state, int dtype, BwdGate gate, const float* ck, void* ws, int64_t ws_bytes, hipStream_t st);

}  // namespace hclsm
