"""Pair costs at the edges of the weight-resident kernel's units (8-column tiles, 4-row groups, 32 staged rows, frames
sharing a unit, row ranges) against the same cost in float64 of the operands rounded as the kernel rounds them."""

from __future__ import annotations

from types import SimpleNamespace

import pytest
import torch

pytestmark = pytest.mark.gpu


def _cost64(m, a, b, al, bl, dtype):
    """The cost with both layers' operands rounded to dtype and everything else in float64."""
    def r(x):
        return x.to(dtype).double()
    D = a.shape[-1]
    a, b = a.clamp(-50, 50), b.clamp(-50, 50)
    w1, w2 = r(m.match_mlp[0].weight), r(m.match_mlp[2].weight)
    u = r(a) @ w1[:, :D].T + m.match_mlp[0].bias.double()
    v = r(b) @ w1[:, D:2 * D].T
    d = r((a[:, :, None] - b[:, None]).abs())
    h = (u[:, :, None] + v[:, None] + d @ w1[:, 2 * D:].T).relu()
    h = (r(h.float()) @ w2.T + m.match_mlp[2].bias.double()).relu()
    s = (h @ m.match_mlp[4].weight.double().T + m.match_mlp[4].bias.double()).squeeze(-1)
    return -(s - 1e4 * (al < 0.5).double()[:, :, None] - 1e4 * (bl < 0.5).double()[:, None])


@pytest.mark.parametrize("F,N,D,dtype", [
    (1, 1, 64, torch.bfloat16),       # one pair
    (5, 8, 64, torch.bfloat16),       # four frames a unit, the last unit short
    (3, 9, 128, torch.bfloat16),      # two frames a unit, a column and row group beyond the first
    (7, 16, 192, torch.float16),
    (2, 31, 192, torch.bfloat16),     # padding in every direction; few units: row ranges
    (300, 17, 64, torch.bfloat16),    # many frames, three column tiles
    (40, 33, 192, torch.bfloat16),    # a second unit across the columns, one column in it
    (2, 128, 128, torch.float16),
])
def test_cost_edges(F, N, D, dtype):
    from hclsm_amd.kernels.slot_tracker import TrackerWeights, track_cost
    from hclsm_amd.objects import SlotTracker
    torch.manual_seed(F + N)
    m = SlotTracker(SimpleNamespace(d_slot=D, n_max_slots=N)).cuda()
    a, b = (torch.randn(F, N, D, device="cuda") * 2 for _ in range(2))
    al, bl = ((torch.rand(F, N, device="cuda") > 0.2).float() for _ in range(2))
    with torch.no_grad():
        got = track_cost(a, b, al, bl, TrackerWeights.from_module(m, dtype)).double()
        ref = _cost64(m, a, b, al, bl, dtype)
        live = (al > 0.5)[:, :, None] & (bl > 0.5)[:, None]
        # the hidden layer is rounded from an fp32 sum on one side and a float64 sum on the other: a value near a
        # rounding boundary moves by one unit, 2^-8 (bf16) of it, and D such terms meet in a sum of random signs
        scale = (ref[live].abs().mean() + 1).item() if live.any() else 1.0
        eps = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
        assert not live.any() or (got - ref)[live].abs().max().item() <= eps * scale
        dead = ~live
        if dead.any():   # an fp32 sum next to the penalty of 1e4 or 2e4: units of 2^-10 or 2^-9
            assert (got - ref)[dead].abs().max().item() <= 2.0 ** -9 + eps * scale
