"""The fused Level-0 block (bf16 autocast: one library call forward, one backward) against the module's float64 math, at
the edges of its tiles, and where the module has to keep its own ops."""

from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


def _block(d, S, seed, expand=2):
    from hclsm_amd.dynamics import SimplifiedSSMBlock
    torch.manual_seed(seed)
    m = SimplifiedSSMBlock(d, S, expand).cuda()
    with torch.no_grad():
        m.dt_proj.bias.sub_(1.0)
        m.norm.weight.add_(0.1 * torch.randn_like(m.norm.weight))
        m.norm.bias.add_(0.1 * torch.randn_like(m.norm.bias))
    return m


def _exact(m, x, g):
    p = {k: v.detach().double().requires_grad_() for k, v in m.named_parameters()}
    x = x.detach().double().requires_grad_()
    u = F.layer_norm(x, (x.shape[-1],), p["norm.weight"], p["norm.bias"])
    z, gate = F.linear(u, p["in_proj.weight"]), F.silu(F.linear(u, p["gate_proj.weight"]))
    dt = F.softplus(F.linear(z, p["dt_proj.weight"], p["dt_proj.bias"])).clamp(1e-3, 1.0)
    B, C = F.linear(z, p["B_proj.weight"]), F.linear(z, p["C_proj.weight"])
    A = -torch.exp(p["A_log"]).clamp(1e-6, 1.0)
    h, ys = z.new_zeros(z.shape[0], z.shape[2], A.shape[1]), []
    for t in range(z.shape[1]):
        h = torch.exp(dt[:, t, :, None] * A) * h + (dt[:, t] * z[:, t])[..., None] * B[:, t, None, :]
        ys.append((h * C[:, t, None, :]).sum(-1))
    y = x + F.linear(torch.stack(ys, 1) * gate, p["out_proj.weight"])
    grads = torch.autograd.grad(y, [x] + list(p.values()), g.double())
    return y.detach(), dict(zip(["x"] + list(p), grads))


def _rel(a, b):
    b = b.detach()
    n = float(b.norm())
    return float((a.detach().double() - b).norm()) / (n if n > 0 else 1.0)   # (one step: A_log has no gradient)


@pytest.mark.parametrize("N,T,d,S,expand", [
    (1, 1, 8, 16, 1),         # smallest
    (3, 5, 40, 24, 2),        # widths that are not multiples of the 64-wide tiles
    (2, 33, 64, 16, 2),       # d_state 16: checkpoints from the forward
    (5, 13, 128, 32, 2),
    (70, 16, 192, 48, 2),     # rows past one weight-gradient split
    (2, 17, 96, 128, 3),      # widest state
    (1, 20, 1024, 64, 1),     # widest row
])
def test_forward_and_gradients(N, T, d, S, expand):
    from hclsm_amd.kernels.ssm_block import block_params
    m = _block(d, S, N + T + d + S, expand)
    gen = torch.Generator("cuda").manual_seed(d)
    x = torch.randn(N, T, d, generator=gen, device="cuda").requires_grad_()
    g = torch.randn(N, T, d, generator=gen, device="cuda")
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert block_params(m, x) is not None
        y = m(x)
        with torch.no_grad():
            assert torch.equal(m(x), y)              # the same kernels without grad
    assert type(y.grad_fn).__name__ == "_BlockBackward"
    names = ["x"] + [n for n, _ in m.named_parameters()]
    grads = torch.autograd.grad(y, [x] + list(m.parameters()), g)
    ye, ge = _exact(m, x, g)
    # bf16 operands (2^-9 each) through up to four chained products; the step size's gradients are sums of both signs
    assert _rel(y, ye) <= 2e-2
    for n, v in zip(names, grads):
        assert v.dtype == torch.float32
        assert _rel(v, ge[n]) <= 6e-2, (n, _rel(v, ge[n]))


def test_partial_gradients_and_checkpointing():
    m = _block(64, 32, 3)
    m.in_proj.weight.requires_grad_(False)
    x = torch.randn(2, 9, 64, device="cuda")
    with torch.autocast("cuda", dtype=torch.bfloat16):
        y = m(x)
    y.sum().backward()
    assert m.in_proj.weight.grad is None
    ref = {n: p.grad.clone() for n, p in m.named_parameters() if p.grad is not None}
    m.zero_grad()
    with torch.autocast("cuda", dtype=torch.bfloat16):
        y2 = torch.utils.checkpoint.checkpoint(m, x, use_reentrant=False)
    y2.sum().backward()
    assert torch.equal(y, y2)
    for n, p in m.named_parameters():
        if p.grad is not None:
            assert torch.equal(p.grad, ref[n])


def test_module_ops_stay_where_they_are_observable():
    """Hooks on a submodule, other submodule types, double-precision parts and fp32 (no autocast) keep the module path."""
    from hclsm_amd.kernels.ssm_block import block_params
    m = _block(64, 32, 4)
    x = torch.randn(2, 5, 64, device="cuda")
    assert block_params(m, x) is None                # no autocast
    with torch.autocast("cuda", dtype=torch.float16):
        assert block_params(m, x) is None
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert block_params(m, x) is not None
        seen = []
        h = m.B_proj.register_forward_hook(lambda mod, i, o: seen.append(o.shape))
        assert block_params(m, x) is None
        m(x)
        h.remove()
        assert seen
        m2 = _block(64, 32, 5)
        m2.dt_proj = torch.nn.Sequential(m2.dt_proj)
        assert block_params(m2, x) is None
        m2(x)
        assert block_params(m, x.half()) is None
