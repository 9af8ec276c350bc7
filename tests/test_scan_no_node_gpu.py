"""The scan without an autograd node against the same call with one: same values, and every form that needs the node
(gradients, function transforms, forward-mode AD) still gets it."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


def _inputs(io, dev="cuda", S=16):
    g = torch.Generator().manual_seed(3)
    x, dt = (torch.randn(3, 9, 40, generator=g) for _ in range(2))
    A = torch.rand(40, S, generator=g).log()
    B, C = (torch.randn(3, 9, S, generator=g) for _ in range(2))
    D = torch.randn(40, generator=g)
    return [t.to(dev) for t in (x.to(io), dt.abs().to(io), A, B.to(io), C.to(io), D)]


@pytest.mark.parametrize("io", [torch.float32, torch.float16])
@pytest.mark.parametrize("form", ["contiguous", "strided", "mixed"])
@pytest.mark.parametrize("skip", [False, True])
def test_same_values(io, form, skip):
    from hclsm_amd.kernels import ssm_scan_fn
    x, dt, A, B, C, D = _inputs(io)
    if form == "strided":
        x, B, A = (t.transpose(-1, -2).contiguous().transpose(-1, -2) for t in (x, B, A))
    if form == "mixed":
        dt, A = dt.float(), A.to(torch.float64)
    D = D if skip else None
    xg = x.clone(memory_format=torch.preserve_format).requires_grad_()
    y1, h1 = ssm_scan_fn(xg, dt, A, B, C, D=D, return_h_final=True)      # with the node
    y0, h0 = ssm_scan_fn(x, dt, A, B, C, D=D, return_h_final=True)       # nothing to record
    with torch.no_grad():
        y2 = ssm_scan_fn(xg, dt, A, B, C, D=D)
    with torch.inference_mode():
        y3 = ssm_scan_fn(x, dt, A, B, C, D=D)
    assert y1.requires_grad and not h1.requires_grad and not y0.requires_grad and not y2.requires_grad
    assert y0.dtype == x.dtype and h0.dtype == torch.float32
    for a, b in ((y0, y1), (h0, h1), (y2, y1), (y3, y1)):
        assert torch.equal(a, b)


def test_transforms_still_see_the_function():
    from hclsm_amd.kernels import ssm_scan_fn
    x, dt, A, B, C, _ = _inputs(torch.float32)
    with pytest.raises(RuntimeError):     # an autograd function without a vmap rule
        torch.func.vmap(lambda v: ssm_scan_fn(v, dt, A, B, C))(x[None])
    import torch.autograd.forward_ad as fwAD
    with fwAD.dual_level():
        with pytest.raises((RuntimeError, NotImplementedError)):      # nor one for forward-mode AD
            ssm_scan_fn(fwAD.make_dual(x, torch.ones_like(x)), dt, A, B, C)
