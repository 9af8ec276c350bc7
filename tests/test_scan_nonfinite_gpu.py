"""Infinities and NaN through the state-group scans: which values they reach, and with which sign, against the oracle
and against the same sequence on a grid too small for the matrix-core form."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle.ssm_scan import normwise_rel_err, ssm_scan_ref

pytestmark = pytest.mark.gpu

INF, NAN = float("inf"), float("nan")


def _np(t):
    return t.detach().double().cpu().numpy()


def _same(got, ref, tol, what):
    """The same values not finite, of the same sign, and the finite ones within tol of the largest."""
    got, ref = _np(got), (_np(ref) if isinstance(ref, torch.Tensor) else ref)
    for f in (np.isnan, np.isposinf, np.isneginf):
        assert np.array_equal(f(got), f(ref)), (what, f.__name__, int((f(got) != f(ref)).sum()))
    ok = np.isfinite(ref)
    assert normwise_rel_err(got[ok], ref[ok]) <= tol, what


def _inputs(N, T, Dn, S, dtype, mode, seed):
    from hclsm_amd.workloads import scan_inputs
    d = scan_inputs(N, T, Dn, S, dtype=dtype, seed=seed)
    if mode == "model":
        d["A_log"] = -d["A_log"]
    d["B"][:, :, 3] = 0                       # inf * 0
    d["B"][:, :, 5] *= 16                     # both signs past 1
    n, c = N - 2, Dn // 2
    d["x"][n, 1, c] = INF                     # one channel of each half of a wave, two signs, a later NaN
    d["x"][n, 2, c + 32 if c + 32 < Dn else c - 32] = -INF
    d["x"][n + 1, 3, 0] = NAN
    d["B"][0, 2, 1], d["B"][0, 2, S - 1] = INF, -INF
    d["B"][1, T - 1, 7] = NAN
    if mode == "raw":
        d["dt"][2 % N, 1, 9], d["x"][2 % N, 1, 9] = 3e38, -3e38       # their product overflows
    return d


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("N,T,Dn,S", [(260, 6, 128, 32), (260, 5, 128, 48), (130, 9, 128, 64), (130, 7, 129, 128),
                                      (3, 6, 128, 48)])
@pytest.mark.parametrize("mode", ["raw", "model"])
def test_forward(N, T, Dn, S, dtype, mode):
    from hclsm_amd.kernels import fused_ssm_scan_hip
    d = _inputs(N, T, Dn, S, dtype, mode, N + S)
    run = lambda rows: fused_ssm_scan_hip(*(d[k][rows].cuda() for k in ("x", "dt")), d["A_log"].cuda(),
                                          *(d[k][rows].cuda() for k in ("B", "C")), clamp_mode=mode, return_h_final=True)
    y, h = run(slice(None))
    tol = 1e-5 if dtype == torch.float32 else 4e-3             # one rounding of the output (2^-9)
    keep = [n for n in range(N) if n != 2 or mode == "model"]  # (the oracle's float64 product does not overflow)
    with np.errstate(all="ignore"):
        ref, href = ssm_scan_ref(*(_np(d[k][keep]) for k in ("x", "dt")), _np(d["A_log"]),
                                 *(_np(d[k][keep]) for k in ("B", "C")), clamp_mode=mode, return_h_final=True)
    _same(h[keep], href, 1e-5, "h_final")
    _same(y[keep], ref, tol, "y")
    for n in (0, 1, 2, N - 2, N - 1):                          # alone: 8 states a lane
        y1, h1 = run(slice(n, n + 1))
        _same(h[n:n + 1], h1, 1e-5, ("h_final", n))
        _same(y[n:n + 1], y1, tol, ("y", n))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_block_forward(dtype):
    from hclsm_amd.kernels import ssm_block_scan
    N, T, Dn, S = 260, 6, 128, 48
    d = _inputs(N, T, Dn, S, dtype, "model", 5)
    g = torch.Generator().manual_seed(6)
    dt_in = (torch.randn(N, T, Dn, generator=g) * 2 - 2).to(dtype)
    gate = torch.randn(N, T, Dn, generator=g).to(dtype)
    with torch.no_grad():
        run = lambda r: ssm_block_scan(*(t.cuda() for t in (d["x"][r], dt_in[r], d["A_log"], d["B"][r], d["C"][r], gate[r])))
        y = run(slice(None))
        for n in (0, 1, N - 2, N - 1):
            _same(y[n:n + 1], run(slice(n, n + 1)), 4e-3, n)


@pytest.mark.parametrize("which", ["x", "gy", "B", "C"])
@pytest.mark.parametrize("N,T,Dn,S", [(1100, 9, 64, 48), (1100, 18, 64, 48), (300, 7, 129, 96)])
@pytest.mark.parametrize("mode", ["raw", "model"])
def test_backward(N, T, Dn, S, mode, which):
    """16 states a lane (wide grids) against the same sequences on a grid too small for it (8 a lane; past 64 states the
    fp32 kernel on the same values)."""
    from hclsm_amd import _lib
    from hclsm_amd.kernels.ssm_scan_bwd import scan_backward
    from hclsm_amd.workloads import scan_inputs
    d = scan_inputs(N, T, Dn, S, dtype=torch.bfloat16, seed=N + S)
    if mode == "model":
        d["A_log"] = -d["A_log"]
    d["gy"] = torch.randn(N, T, Dn, generator=torch.Generator().manual_seed(1)).to(torch.bfloat16)
    d["B"][:, :, 3] = 0
    d["C"][:, :, 4] = 0
    rows = [0, 1, N // 2, N - 1]
    for n, bad in zip(rows, (INF, -INF, NAN, INF)):
        d[which][n, T // 2 if n else T - 1, (5 + 40 * (n & 1)) % S] = bad
    code = _lib.SCAN_RAW if mode == "raw" else _lib.SCAN_MODEL

    def run(pick, dtype):
        v = [d[k][pick].cuda().to(dtype) for k in ("x", "dt", "B", "C", "gy")]
        return scan_backward(v[0], v[1], d["A_log"].cuda(), v[2], v[3], None, v[4], code)

    got = run(slice(None), torch.bfloat16)
    for n in rows + [2]:
        ref = run(slice(n, n + 1), torch.bfloat16 if S <= 64 else torch.float32)
        for k in ("x", "dt", "B", "C"):
            _same(got[k][n:n + 1], ref[k], 4e-3, (k, n))
    # gA_log: not finite where any sequence's is
    odd = torch.zeros_like(got["A_log"], dtype=torch.bool)
    for n in rows:
        odd |= ~torch.isfinite(run(slice(n, n + 1), torch.float32)["A_log"])
    assert torch.equal(~torch.isfinite(got["A_log"]), odd)
