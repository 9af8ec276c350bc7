"""A whole SimplifiedSSMBlock (hclsm/dynamics/level0_ssm.py:30-107) under a bf16 autocast on MI355X
(libhclsm_amd.so: hclsm_ssm_block_forward / hclsm_ssm_block_backward): one library call each way, with bf16 operands
and intermediates where the module's ops have them, fp32 residual stream, parameters and gradients.  The output
projection, the parts of z's gradient and the weight gradients, which the module's ops round to bf16 one by one, are
summed in fp32, and every sum has its own order: results differ from the module's ops in bf16 roundings.
"""

from __future__ import annotations

import ctypes

import torch
import torch.nn as nn

from hclsm_amd import _lib

_NAMES = ("ln_w", "ln_b", "w_in", "w_gate", "w_dt", "b_dt", "w_b", "w_c", "a_log", "w_out")


class _Ptrs(ctypes.Structure):
    """Mirror of the C structs HclsmBlockParams / HclsmBlockGrads (the same ten pointers)."""
    _fields_ = [(n, ctypes.c_void_p) for n in _NAMES]


def _ptrs(tensors) -> _Ptrs:
    return _Ptrs(*(None if t is None else t.data_ptr() for t in tensors))


def _shapes(d: int, di: int, S: int) -> tuple:
    """The parameters' shapes in _NAMES order."""
    return (d,), (d,), (di, d), (di, d), (di, di), (di,), (S, di), (S, di), (di, S), (d, di)


def _params(m, cls):
    """(weight, bias) of a submodule that is a plain cls to which nothing is attached (no hook, and no forward of the
    instance's own, as wrapping libraries set), else (None, None).  What m.weight finds, an entry of the instance or
    else a parameter, without the 0.5 us that the attribute of a module costs."""
    if type(m) is not cls:
        return None, None
    d = m.__dict__
    if "forward" in d or d["_forward_hooks"] or d["_forward_pre_hooks"] or d["_backward_hooks"] or d["_backward_pre_hooks"]:
        return None, None
    ps = d["_parameters"]
    return d["weight"] if "weight" in d else ps.get("weight"), d["bias"] if "bias" in d else ps.get("bias")


def block_params(m, x):
    """The block's parameters in _NAMES order where the fused block computes what the module's ops would (bf16 autocast,
    fp32 input and parameters, plain submodules nobody hooks into, no tracing or function transform), else None."""
    if not (x.is_cuda and x.dtype == torch.float32 and x.dim() == 3 and x.numel() > 0 and type(x) in (torch.Tensor, nn.Parameter)):
        return None
    if not torch.is_autocast_enabled("cuda") or torch.get_autocast_dtype("cuda") != torch.bfloat16:
        return None
    if torch.compiler.is_compiling() or torch.jit.is_tracing() or torch._C._are_functorch_transforms_active():
        return None
    if torch.autograd.forward_ad._current_level >= 0:
        return None
    mm = nn.modules.module
    if mm._global_forward_hooks or mm._global_forward_pre_hooks or mm._global_backward_hooks or mm._global_backward_pre_hooks:
        return None
    norm = m.norm
    ln_w, ln_b = _params(norm, nn.LayerNorm)
    if ln_b is None or norm.eps != 1e-5:
        return None
    (w_in, b0), (w_gate, b1), (w_dt, b_dt), (w_b, b2), (w_c, b3), (w_out, b4) = [
        _params(p, nn.Linear) for p in (m.in_proj, m.gate_proj, m.dt_proj, m.B_proj, m.C_proj, m.out_proj)]
    if not (b0 is b1 is b2 is b3 is b4 is None):
        return None
    ps = (ln_w, ln_b, w_in, w_gate, w_dt, b_dt, w_b, w_c, m.A_log, w_out)    # (a None among them ends below)
    dev = x.device
    if any(type(p) not in (nn.Parameter, torch.Tensor) or p.dtype != torch.float32 or p.device != dev or
           not p.is_contiguous() for p in ps):
        return None
    if ps[8].dim() != 2:
        return None
    d, (di, S) = x.shape[2], ps[8].shape
    if any(p.shape != s for p, s in zip(ps, _shapes(d, di, S))):
        return None
    return ps


def _aligned(t, n: int = 16):
    """t contiguous at a multiple of n bytes: t itself, or a copy (torch allocates at 512).  Gradients and unpacked saved
    tensors may be contiguous views at any offset, where the forward's inputs were checked."""
    t = t.contiguous()
    return t if t.data_ptr() % n == 0 else t.clone()


def _save_buffer(x, ps, train: bool):
    N, T, d = x.shape
    nb = int(_lib.lib().hclsm_ssm_block_save(N, T, d, ps[8].shape[0], ps[8].shape[1], int(train)))
    return None if nb < 0 else torch.empty(nb, dtype=torch.uint8, device=x.device)


def _forward(x, ps, save, train: bool):
    N, T, d = x.shape
    out = torch.empty_like(x)
    st = _ptrs(ps)
    return out, _lib.lib().hclsm_ssm_block_forward(
        ctypes.byref(st), x.data_ptr(), out.data_ptr(), N, T, d, ps[8].shape[0], ps[8].shape[1], int(train),
        save.data_ptr(), save.numel(), _lib.stream_of(x))


class _Block(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, save, *ps):
        out, rc = _forward(x, ps, save, True)
        _lib.check(rc, "hclsm_ssm_block_forward")
        ctx.save_for_backward(x, save, ps[0], ps[8])   # (the backward's other parameters are in save, rounded)
        return out

    @staticmethod
    @torch.autograd.function.once_differentiable
    def backward(ctx, g):
        x, save, ln_w, a_log = (_aligned(t, 256 if t.dtype == torch.uint8 else 16) for t in ctx.saved_tensors)
        N, T, d = x.shape
        di, S = a_log.shape
        g = _aligned(g.to(torch.float32))
        L = _lib.lib()
        scratch = torch.empty(int(L.hclsm_ssm_block_scratch(N, T, d, di, S)), dtype=torch.uint8, device=x.device)
        need = ctx.needs_input_grad               # (x, save, parameters): the others are not formed
        gx = torch.empty_like(x) if need[0] else None
        grads = [x.new_empty(s) if n else None for s, n in zip(_shapes(d, di, S), need[2:])]
        st, sg = _Ptrs(ln_w=ln_w.data_ptr(), a_log=a_log.data_ptr()), _ptrs(grads)
        rc = L.hclsm_ssm_block_backward(ctypes.byref(st), x.data_ptr(), g.data_ptr(), _lib.ptr(gx), ctypes.byref(sg), N, T,
                                        d, di, S, save.data_ptr(), save.numel(), scratch.data_ptr(), scratch.numel(),
                                        _lib.stream_of(x))
        _lib.check(rc, "hclsm_ssm_block_backward")
        return (gx, None, *grads)


def ssm_block(m, x):
    """The block's output, or None where this path does not apply (the caller runs the module's ops)."""
    ps = block_params(m, x)
    if ps is None:
        return None
    xc = x.contiguous()
    train = torch.is_grad_enabled() and (xc.requires_grad or any(p.requires_grad for p in ps))
    save = _save_buffer(xc, ps, train)
    if save is None or (xc.data_ptr() | ps[0].data_ptr() | ps[1].data_ptr() | ps[8].data_ptr()) & 15:
        return None
    if train:
        return _Block.apply(xc, save, *ps)
    out, rc = _forward(xc, ps, save, False)
    if rc == _lib.ERR_UNSUPPORTED:
        return None
    _lib.check(rc, "hclsm_ssm_block_forward")
    return out
