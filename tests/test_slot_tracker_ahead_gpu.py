"""Frame pairs matched ahead of the tracking loop: a few clips (pairs ahead) against the same clips repeated past the
device's compute units (the loop alone), bit for bit, on decisive, undecided, tied and degenerate matches."""

from __future__ import annotations

from types import SimpleNamespace

import pytest
import torch

pytestmark = pytest.mark.gpu


def _tracker(D, N, decisive, seed):
    from hclsm_amd.objects import SlotTracker
    torch.manual_seed(seed)
    m = SlotTracker(SimpleNamespace(d_slot=D, n_max_slots=N)).cuda()
    if decisive:
        with torch.no_grad():
            w0, w1, w2 = (m.match_mlp[i].weight for i in (0, 2, 4))
            w0.mul_(0.02)[:, 2 * D:].add_(torch.eye(D, device="cuda"))
            w1.mul_(0.02).add_(1.0 / D)
            w2.mul_(0.02).sub_(decisive / D)
    return m


def _clips(B, T, N, D, seed, dead, dup=False):
    g = torch.Generator().manual_seed(seed)
    s = torch.randn(B, 1, N, D, generator=g) + 0.02 * torch.randn(B, T, N, D, generator=g)
    if dup:
        s[:, :, 1] = s[:, :, 0]                    # two equal slots: an exact tie in every frame
    live = (torch.rand(B, 1, N, generator=g) >= dead).float().expand(B, T, N)
    if dead and T > 4:
        live = live.clone()
        live[:, T // 2:, 0] = 1 - live[:, T // 2:, 0]   # a slot dies (or appears) half way
    perm = torch.rand(B, T, N, generator=g).argsort(-1)
    return (s.expand(B, T, N, D).gather(2, perm[..., None].expand(B, T, N, D)).contiguous().cuda(),
            live.gather(2, perm).contiguous().cuda())


@pytest.mark.parametrize("B,T,N,D,dead,decisive,dup", [
    (3, 9, 16, 64, 0.0, 8.0, False),     # every match a permutation
    (4, 12, 32, 64, 0.2, 8.0, False),    # dead slots: flat rows and columns, ties among them
    (2, 7, 31, 64, 0.5, 8.0, True),      # padding, half dead, an exact tie
    (3, 8, 32, 64, 0.2, 0.3, False),     # close decisions
    (3, 8, 32, 64, 0.2, 0.0, False),     # untrained weights: matches that are no permutations
    (2, 5, 70, 64, 0.1, 8.0, False),
    (1, 4, 128, 64, 0.1, 8.0, False),    # most slots
    (2, 3, 8, 64, 0.1, 8.0, False),      # too short for matching ahead
    (3, 6, 16, 64, 1.0, 8.0, False),     # every slot dead
])
def test_equals_the_loop(B, T, N, D, dead, decisive, dup):
    from hclsm_amd.kernels.slot_tracker import TrackerWeights, track_sequence
    m = _tracker(D, N, decisive, N + T)
    slots, alive = _clips(B, T, N, D, B + N, dead, dup)
    W = TrackerWeights.from_module(m, torch.float32)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    rep = cus // B + 1
    with torch.no_grad():
        few = track_sequence(slots, alive, W, with_hidden=False)
        many = track_sequence(slots.repeat(rep, 1, 1, 1), alive.repeat(rep, 1, 1), W, with_hidden=False)
    for k, v in few.items():
        if v is not None:
            assert torch.equal(v, many[k][:B]), k
            assert torch.equal(v, many[k][-B:]), k


def test_nan_slots_take_the_loop():
    from hclsm_amd.kernels.slot_tracker import TrackerWeights, track_sequence
    m = _tracker(64, 16, 8.0, 1)
    slots, alive = _clips(2, 8, 16, 64, 5, 0.2)
    slots[0, 3, 4] = float("nan")
    W = TrackerWeights.from_module(m, torch.float32)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    few = track_sequence(slots, alive, W, with_hidden=False)
    many = track_sequence(slots.repeat(cus, 1, 1, 1), alive.repeat(cus, 1, 1), W, with_hidden=False)
    for k, v in few.items():
        if v is not None:
            assert torch.equal(v.nan_to_num(7.0), many[k][:2].nan_to_num(7.0)), k
