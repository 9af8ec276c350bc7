"""The fused Level-0 block inside a larger autograd graph: incoming gradients and saved tensors at any address, the saved
forward left as it is; and beside the module's own ops."""

from __future__ import annotations

import pytest
import torch

from test_ssm_block_gpu import _block, _exact, _rel

pytestmark = pytest.mark.gpu


def _grads(m, x, loss):
    m.zero_grad()
    x.grad = None
    loss.backward()
    return [x.grad.clone()] + [p.grad.clone() for p in m.parameters()]


def _run(m, x):
    with torch.autocast("cuda", dtype=torch.bfloat16):
        y = m(x)
    assert type(y.grad_fn).__name__ == "_BlockBackward"
    return y


@pytest.mark.parametrize("S", [16, 48])
@pytest.mark.parametrize("shift", [1, 2, 3])
def test_gradient_at_an_odd_address(S, shift):
    """The backward of a cat hands a contiguous view at any multiple of 4 bytes over."""
    m = _block(64, S, 1)
    x = torch.randn(3, 9, 64, device="cuda").requires_grad_()
    aux = torch.randn(shift, device="cuda").requires_grad_()
    w = torch.randn(shift + x.numel(), device="cuda")
    assert w[shift:].data_ptr() % 16
    got = _grads(m, x, (torch.cat([aux, _run(m, x).reshape(-1)]) * w).sum())
    ref = _grads(m, x, (_run(m, x).reshape(-1) * w[shift:].clone()).sum())
    for a, b in zip(got, ref):
        assert torch.equal(a, b)


def test_saved_tensors_at_an_odd_address():
    """Saved-tensor hooks that hand back copies inside a larger buffer, one element past its start."""
    m = _block(64, 32, 2)
    x = torch.randn(2, 7, 64, device="cuda").requires_grad_()
    g = torch.randn_like(x)

    def pack(t):
        buf = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
        buf[1:].copy_(t.detach().reshape(-1))
        return buf, t.shape

    ref = _grads(m, x, (_run(m, x) * g).sum())
    with torch.autograd.graph.saved_tensors_hooks(pack, lambda h: h[0][1:].view(h[1])):
        y = _run(m, x)
    got = _grads(m, x, (y * g).sum())
    for a, b in zip(got, ref):
        assert torch.equal(a, b)


@pytest.mark.parametrize("S", [16, 48])
def test_the_backward_only_reads_what_the_forward_saved(S):
    """A second backward over the same saved forward finds what the first one found."""
    m = _block(64, S, 3)
    x = torch.randn(40, 19, 64, device="cuda").requires_grad_()
    y = _run(m, x)
    ps = [x] + list(m.parameters())
    g = torch.randn_like(x)
    saved = [t.clone() for t in y.grad_fn.saved_tensors]
    ref = torch.autograd.grad(y, ps, g, retain_graph=True)
    for a, b in zip(y.grad_fn.saved_tensors, saved):
        assert torch.equal(a, b)
    again = torch.autograd.grad(y, ps, g)
    for a, b in zip(again, ref):
        assert torch.equal(a, b)


_PARAMS = {"norm.weight": "ln_w", "norm.bias": "ln_b", "in_proj.weight": "w_in", "gate_proj.weight": "w_gate",
           "dt_proj.weight": "w_dt", "dt_proj.bias": "b_dt", "B_proj.weight": "w_b", "C_proj.weight": "w_c",
           "A_log": "a_log", "out_proj.weight": "w_out"}


@pytest.mark.parametrize("S", [16, 48])
@pytest.mark.parametrize("wanted", [["x"], *([n] for n in _PARAMS), ["x", "A_log"], ["in_proj.weight", "dt_proj.bias"],
                                    [n for n in _PARAMS if n != "dt_proj.weight"]])
def test_only_the_wanted_gradients_are_formed(S, wanted, monkeypatch):
    """Frozen inputs and parameters reach the library as null pointers; the others' gradients do not change."""
    from hclsm_amd import _lib
    from hclsm_amd.kernels import ssm_block
    m = _block(72, S, 4)                                     # widths past one tile
    x = torch.randn(5, 11, 72, device="cuda").requires_grad_()
    g = torch.randn_like(x)
    names = {"x": x, **dict(m.named_parameters())}
    ref = dict(zip(names, torch.autograd.grad(_run(m, x), list(names.values()), g)))
    for n, t in names.items():
        t.requires_grad_(n in wanted)
    seen = []

    class Recorder:
        def __getattr__(self, name):
            fn = getattr(_lib.lib(), name)
            if name != "hclsm_ssm_block_backward":
                return fn

            def call(*a):
                sg = a[4]._obj
                seen.append({"x": a[3], **{n: getattr(sg, c) for n, c in _PARAMS.items()}})
                return fn(*a)
            return call

    class Lib:
        def __getattr__(self, name):
            return (lambda: Recorder()) if name == "lib" else getattr(_lib, name)

    monkeypatch.setattr(ssm_block, "_lib", Lib())
    got = torch.autograd.grad(_run(m, x), [names[n] for n in wanted], g)
    for n, v in zip(wanted, got):
        assert torch.equal(v, ref[n]), n
    assert len(seen) == 1
    assert {n for n, p in seen[0].items() if p} == set(wanted)


@pytest.mark.parametrize("S", [16, 48])
def test_parameters_changed_before_the_backward(S):
    """Matrices that the forward rounded to bf16 may change afterwards (a step of one loss before the backward of the
    next, as with the module's ops); those that the backward reads itself may not."""
    m = _block(64, S, 5)
    x = torch.randn(3, 9, 64, device="cuda").requires_grad_()
    g = torch.randn_like(x)
    ps = [x] + list(m.parameters())
    ref = torch.autograd.grad(_run(m, x), ps, g)
    kept = {n: p.detach().clone() for n, p in m.named_parameters()}
    y = _run(m, x)
    with torch.no_grad():
        for n, p in m.named_parameters():
            if n not in ("norm.weight", "A_log"):
                p.add_(1.0)
    for a, b in zip(torch.autograd.grad(y, ps, g), ref):
        assert torch.equal(a, b)
    for name in ("norm.weight", "A_log"):
        m.load_state_dict(kept)
        y = _run(m, x)
        with torch.no_grad():
            m.get_parameter(name).add_(1.0)
        with pytest.raises(RuntimeError, match="modified by an inplace operation"):
            torch.autograd.grad(y, ps, g)


def test_a_submodules_own_forward_is_called():
    """Libraries that wrap modules set `forward` on the instance: the module's ops run it."""
    m = _block(64, 32, 6)
    x = torch.randn(2, 5, 64, device="cuda")
    with torch.autocast("cuda", dtype=torch.bfloat16), torch.no_grad():
        plain = m(x)
        for name in ("norm", "B_proj", "out_proj"):
            sub, seen = getattr(m, name), []
            sub.forward = lambda *a, f=type(sub).forward, sub=sub: seen.append(1) or f(sub, *a)
            y = m(x)
            del sub.forward
            assert seen or name == "out_proj"      # (the module reads out_proj's weight itself)
            assert (y - plain).norm() <= 2e-2 * plain.norm()


def _both_ways(m, x, g):
    """Output and gradients of the fused block and of the module's ops, and the same in float64."""
    ps = [x] + list(m.parameters())
    out = []
    for hooked in (False, True):
        h = m.B_proj.register_forward_hook(lambda mod, i, o: None) if hooked else None    # keeps the module's ops
        with torch.autocast("cuda", dtype=torch.bfloat16):
            y = m(x)
        if h:
            h.remove()
        assert (type(y.grad_fn).__name__ == "_BlockBackward") != hooked
        out.append((y.detach(), *torch.autograd.grad(y, ps, g)))
    ye, ge = _exact(m, x, g)
    return out, (ye, *ge.values())


@pytest.mark.parametrize("N,T,d,S,expand", [
    (70, 16, 192, 48, 2), (64, 33, 128, 16, 2), (40, 13, 128, 32, 2), (20, 17, 96, 128, 3), (300, 16, 192, 48, 2)])
def test_no_further_from_float64_than_the_modules_ops(N, T, d, S, expand):
    """The fused block makes a part of the module's roundings: its errors are no larger.  The two share the roundings
    that weigh most (operands, the inputs of the scan), so their errors differ little; a tenth is left to chance."""
    m = _block(d, S, N + S, expand)
    gen = torch.Generator("cuda").manual_seed(N)
    x = torch.randn(N, T, d, generator=gen, device="cuda").requires_grad_()
    g = torch.randn(N, T, d, generator=gen, device="cuda")
    (fused, module), exact = _both_ways(m, x, g)
    for name, a, b, e in zip(["y", "x"] + [n for n, _ in m.named_parameters()], fused, module, exact):
        assert _rel(a, e) <= 1.1 * _rel(b, e), (name, _rel(a, e), _rel(b, e))


@pytest.mark.parametrize("d,S", [(64, 72), (64, 8), (36, 32), (64, 20)])
def test_widths_that_keep_the_modules_ops(d, S):
    """d_state past 64 that is no multiple of 16, below 16, or widths that are no multiples of 8."""
    from hclsm_amd.kernels.ssm_block import ssm_block
    m = _block(d, S, 8)
    x = torch.randn(3, 9, d, device="cuda").requires_grad_()
    g = torch.randn_like(x)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert ssm_block(m, x) is None
        y = m(x)
    grads = torch.autograd.grad(y, [x] + list(m.parameters()), g)
    ye, ge = _exact(m, x, g)
    assert _rel(y, ye) <= 2e-2
    for v, n in zip(grads, ge):
        assert _rel(v, ge[n]) <= 6e-2, n
