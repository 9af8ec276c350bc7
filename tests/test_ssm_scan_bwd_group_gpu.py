"""The state-group backward scan against the float64 oracle at the edges of its windows (16 steps), chunks (4),
channel blocks (64), state groups (8 / 16) and sequence walk."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle.ssm_scan import normwise_rel_err, ssm_scan_bwd_ref

pytestmark = pytest.mark.gpu


def _np(t):
    return t.detach().double().cpu().numpy()


def _case(N, T, Dn, S, dtype, mode, seed):
    from hclsm_amd.workloads import scan_inputs
    d = scan_inputs(N, T, Dn, S, dtype=dtype, seed=seed)
    if mode == "model":
        d["A_log"] = -d["A_log"]
    gy = torch.randn(N, T, Dn, generator=torch.Generator().manual_seed(seed + 1)).to(dtype)
    return d, gy


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("N,T,Dn,S", [
    (1, 1, 1, 24),          # smallest
    (2, 4, 64, 32),         # one chunk
    (2, 5, 65, 40),         # one past a chunk and a channel block
    (1, 16, 63, 64),        # one window
    (2, 17, 70, 48),        # one past it
    (2, 35, 96, 32),        # last window of three steps
    (1, 13, 64, 96),        # past 64 states
    (1, 20, 66, 128),       # most states
    (1100, 9, 64, 48),      # 16 states a lane, sequences walked by one workgroup
])
@pytest.mark.parametrize("mode", ["raw", "model"])
def test_matches_oracle(N, T, Dn, S, dtype, mode):
    from hclsm_amd import _lib
    from hclsm_amd.kernels.ssm_scan_bwd import scan_backward
    d, gy = _case(N, T, Dn, S, dtype, mode, N + T + Dn + S)
    code = _lib.SCAN_RAW if mode == "raw" else _lib.SCAN_MODEL
    got = scan_backward(*(d[k].cuda() for k in ("x", "dt", "A_log", "B", "C", "D")), gy.cuda(), code)
    ref = ssm_scan_bwd_ref(*(_np(d[k]) for k in ("x", "dt", "A_log", "B", "C")), _np(gy), D=_np(d["D"]),
                           clamp_mode=mode)
    for name, g in got.items():
        # fp32 results: sums of fp32 products; bf16 ones: one rounding of such a sum (2^-9)
        tol = 1e-5 if g.dtype == torch.float32 else 4e-3
        err = normwise_rel_err(_np(g), ref[name])
        assert err <= tol, f"{name}: {err:.3e}"


@pytest.mark.parametrize("dtype,N", [(torch.float32, 3), (torch.bfloat16, 3), (torch.bfloat16, 1100)])
def test_nonfinite_inputs_stay_in_their_channel(dtype, N):
    """An infinity or NaN of one channel's x or gy leaves the other channels' gx, gdt and gA_log untouched."""
    from hclsm_amd import _lib
    from hclsm_amd.kernels.ssm_scan_bwd import scan_backward
    d, gy = _case(N, 9, 64, 48, dtype, "raw", 5)
    args = [d[k].cuda() for k in ("x", "dt", "A_log", "B", "C")]
    clean = scan_backward(*args, None, gy.cuda(), _lib.SCAN_RAW)
    for which in ("x", "gy"):
        for bad in (float("inf"), float("nan")):
            x, g = args[0].clone(), gy.cuda().clone()
            (x if which == "x" else g)[1, 6, 40] = bad
            got = scan_backward(x, *args[1:], None, g, _lib.SCAN_RAW)
            assert not torch.isfinite(got["x" if which == "gy" else "dt"][1, :, 40]).all()
            for name in ("x", "dt"):
                keep = torch.ones_like(got[name], dtype=torch.bool)
                keep[1, :, 40] = False
                assert torch.equal(got[name][keep], clean[name][keep]), (which, bad, name)
            rows = torch.arange(64, device="cuda") != 40
            assert torch.equal(got["A_log"][rows], clean["A_log"][rows])


@pytest.mark.parametrize("N,T,Dn,S", [(512, 16, 512, 64), (1024, 16, 384, 48)])
def test_gA_log_sums_over_a_walk(N, T, Dn, S):
    """gA_log where a workgroup walks 4 to 8 sequences: the rounding of its sums.  An fp32 addition of random terms
    rounds by 2.4e-8 (rms), a chain of k by 2.4e-8 sqrt(k / 2), and the terms themselves are good to 1.45e-7.  The walk's
    chain is 32 sums of four steps at most: 1.75e-7 in all; step by step it is 128: 2.4e-7.  (One partial per sequence and
    a chain of 32 of them: 1.9e-7.)"""
    from hclsm_amd import _lib
    from hclsm_amd.kernels.ssm_scan_bwd import scan_backward
    d, gy = _case(N, T, Dn, S, torch.float32, "raw", N + S)
    x, dt, A_log, B, C = (d[k].cuda() for k in ("x", "dt", "A_log", "B", "C"))
    gy = gy.cuda()
    got = scan_backward(x, dt, A_log, B, C, None, gy, _lib.SCAN_RAW)["A_log"].double()
    al = A_log.double().requires_grad_()
    A, h, loss = -torch.exp(al), torch.zeros(N, Dn, S, dtype=torch.float64, device="cuda"), 0.0
    for t in range(T):
        h = torch.exp(dt[:, t, :, None].double() * A) * h + (dt[:, t].double() * x[:, t].double())[..., None] * B[:, t, None].double()
        loss = loss + ((h * C[:, t, None].double()).sum(-1) * gy[:, t].double()).sum()
    want, = torch.autograd.grad(loss, al)
    err = float((got - want).norm() / want.norm())
    assert err <= 1.9e-7, f"{err:.3e}"
