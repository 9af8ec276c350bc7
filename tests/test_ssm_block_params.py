"""What the fused Level-0 block takes as a plain submodule's parameters: what its attributes give, or nothing."""

from __future__ import annotations

import torch
import torch.nn as nn
from torch.nn.utils import parametrizations

from hclsm_amd.kernels.ssm_block import _params


def _same(m, cls):
    w, b = _params(m, cls)
    assert w is m.weight and b is m.bias


def test_what_the_attributes_give():
    _same(nn.Linear(4, 4), nn.Linear)
    _same(nn.Linear(4, 4, bias=False), nn.Linear)
    _same(nn.LayerNorm(4), nn.LayerNorm)
    _same(nn.LayerNorm(4, elementwise_affine=False), nn.LayerNorm)
    m = nn.Linear(4, 4)
    w, b = m.weight, m.bias
    m._parameters.clear()                     # as replicas of a module keep theirs: tensors of the instance
    m.weight, m.bias = w.detach().clone(), b.detach().clone()
    _same(m, nn.Linear)


def test_nothing_of_what_is_not_plain():
    class Own(nn.Linear):
        pass

    hooked = [nn.Linear(4, 4) for _ in range(5)]
    hooked[0].register_forward_hook(lambda *a: None)
    hooked[1].register_forward_pre_hook(lambda *a: None)
    hooked[2].register_full_backward_hook(lambda *a: None)
    hooked[3].register_full_backward_pre_hook(lambda *a: None)
    hooked[4].forward = torch.relu
    gone = nn.Linear(4, 4)
    del gone.weight
    for m in (*hooked, Own(4, 4), parametrizations.weight_norm(nn.Linear(4, 4)), nn.LayerNorm(4), None, torch.relu):
        assert _params(m, nn.Linear) == (None, None)
    assert _params(gone, nn.Linear)[0] is None
