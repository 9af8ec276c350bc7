"""The state-group forward scan (d_state split over the waves of a workgroup) against the numpy oracle, at the edges
of its channel blocks (64), chunks (4 steps) and state groups (8 / 16), and its handling of non-finite inputs."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle.ssm_scan import normwise_rel_err, ssm_scan_ref

pytestmark = pytest.mark.gpu

# bf16 output: one rounding (2^-9) of a value accumulated in fp32; the final state stays fp32
TOL = {torch.float32: 1e-5, torch.bfloat16: 4e-3}


def _np(t):
    return t.detach().double().cpu().numpy()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("N,T,Dn,S", [
    (1, 1, 1, 16),         # d_state 16: one lane per channel
    (1, 1, 1, 24),         # smallest of the state groups
    (2, 3, 63, 24),        # T below the chunk, a group count that does not divide it
    (3, 4, 64, 32),
    (2, 5, 65, 48),        # one past the chunk and the channel block
    (2, 9, 130, 64),
    (1, 17, 70, 96),
    (1, 8, 64, 128),       # most groups
    (260, 6, 96, 48),      # enough waves for the matrix-core form
    (130, 7, 129, 128),
])
@pytest.mark.parametrize("mode", ["raw", "model"])
def test_matches_oracle(N, T, Dn, S, dtype, mode):
    from hclsm_amd.kernels import fused_ssm_scan_hip
    from hclsm_amd.workloads import scan_inputs
    d = scan_inputs(N, T, Dn, S, dtype=dtype, seed=N + T + Dn + S)
    if mode == "model":
        d["A_log"] = -d["A_log"]
    y, h = fused_ssm_scan_hip(*(d[k].cuda() for k in ("x", "dt", "A_log", "B", "C")), D=d["D"].cuda(),
                              clamp_mode=mode, return_h_final=True)
    ref, href = ssm_scan_ref(*(_np(d[k]) for k in ("x", "dt", "A_log", "B", "C")), D=_np(d["D"]), clamp_mode=mode,
                             return_h_final=True)
    assert normwise_rel_err(_np(y), ref) <= TOL[dtype]
    assert normwise_rel_err(_np(h), href) <= 1e-5


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_nonfinite_inputs_stay_in_their_channel(dtype):
    """An infinity or NaN of one channel reaches that channel's later outputs and no other's; A_log = -inf (no decay)
    is a valid exponent."""
    from hclsm_amd.kernels import fused_ssm_scan_hip
    from hclsm_amd.workloads import scan_inputs
    N, T, Dn, S = 260, 6, 128, 48
    d = {k: v.cuda() for k, v in scan_inputs(N, T, Dn, S, dtype=dtype, seed=3).items()}
    d["A_log"][5, 3] = -float("inf")
    args = lambda: [d[k] for k in ("x", "dt", "A_log", "B", "C")]
    clean = fused_ssm_scan_hip(*args(), clamp_mode="raw")
    assert torch.isfinite(clean).all()
    for bad in (float("inf"), -float("inf"), float("nan")):
        d["x"][7, 2, 40] = bad
        got = fused_ssm_scan_hip(*args(), clamp_mode="raw")
        where = ~torch.isfinite(got)
        want = torch.zeros_like(where)
        want[7, 2:, 40] = True
        assert torch.equal(where, want)
        assert torch.equal(got[~want], clean[~want])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("N,T,Dn,S", [(2, 6, 70, 48), (260, 5, 66, 48)])
def test_block_mode(N, T, Dn, S, dtype):
    """softplus, clamp and gate in the kernel: against the scan oracle with the same steps in float64."""
    from hclsm_amd.kernels import ssm_block_scan
    from hclsm_amd.workloads import scan_inputs
    d = scan_inputs(N, T, Dn, S, dtype=dtype, seed=11)
    g = torch.Generator().manual_seed(12)
    dt_in = (torch.randn(N, T, Dn, generator=g) * 2 - 2).to(dtype)
    gate = torch.randn(N, T, Dn, generator=g).to(dtype)
    with torch.no_grad():
        y = ssm_block_scan(*(t.cuda() for t in (d["x"], dt_in, -d["A_log"], d["B"], d["C"], gate)))
    dt = np.clip(np.logaddexp(0.0, _np(dt_in)), 1e-3, 1.0)
    ref = ssm_scan_ref(_np(d["x"]), dt, -_np(d["A_log"]), _np(d["B"]), _np(d["C"]), clamp_mode="model")
    ref = ref * _np(gate) / (1.0 + np.exp(-_np(gate)))
    assert normwise_rel_err(_np(y), ref) <= TOL[dtype]
