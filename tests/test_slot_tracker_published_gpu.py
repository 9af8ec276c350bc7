"""What the workgroups beside the tracking loop publish: a frame pair whose decisions are far apart (worked out in float64
from the same cost block) has a match for every row, one with a close decision has none, and the published matches,
composed through the previous order, are the loop's own wherever its rows are the pair's in another order."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from test_slot_tracker_ahead_gpu import _clips, _tracker

pytestmark = pytest.mark.gpu

READY, FLAT, IDX = 1 << 30, 1 << 29, 0xffff
FIRST = 3                       # the first frame matched beside the loop


def _run(slots, alive, W, n_iters=20, temperature=0.05):
    """track_sequence with a workspace of its own: (perm, cost blocks (B, T-1, N, N), published words (B, T, N))."""
    from hclsm_amd import _lib
    B, T, N, D = slots.shape
    L, code = _lib.lib(), _lib.dtype_code(W.dtype)
    size = int(L.hclsm_slot_track_sequence_workspace(B, T, N, D, 0, code))
    ws = torch.zeros(size, dtype=torch.uint8, device="cuda")
    tracked, alive_out = torch.empty_like(slots), torch.empty_like(alive)
    perm = torch.empty(B, T, N, dtype=torch.int64, device="cuda")
    matched = torch.empty(B, T, N, device="cuda")
    _lib.check(L.hclsm_slot_track_sequence(
        _lib.ptr(slots), _lib.ptr(alive), _lib.ptr(tracked), _lib.ptr(alive_out), _lib.ptr(perm), _lib.ptr(matched), None,
        B, T, N, D, n_iters, temperature, W.ptrs, code, _lib.ptr(ws), size, _lib.stream_of(slots)), "track_sequence")
    up = lambda n: (n + 255) // 256 * 256
    R = B * T * N
    c0 = up(R * D * 4) + up(R * 2 * D * 4)                  # after the clamped slots and their projections
    cost = ws[c0:c0 + B * (T - 1) * N * N * 4].view(torch.float32).view(B, T - 1, N, N)
    words = ws[size - up(R * 4):][:R * 4].view(torch.int32).view(B, T, N)        # the last region
    return perm.cpu(), cost.cpu().numpy(), words.cpu().numpy()


def _decide(cost, n_iters=20, temperature=0.05):
    """True / False where the pair has to be published / must not be, None where it is within the rounding of either."""
    flat = np.clip(cost, -1e4, 1e4) == 1e4
    fr, fc = flat.all(1), flat.all(0)
    la = -np.clip(cost.astype(np.float64), -1e4, 1e4) / temperature
    lse = lambda a, axis: (m := a.max(axis, keepdims=True)) + np.log(np.exp(a - m).sum(axis, keepdims=True))
    sure = True
    for it in range(n_iters):
        la = la - lse(la, 1)
        la = la - lse(la, 0)
        if it + 1 in (5, n_iters):
            best = la.argmax(1)
            other = ~np.eye(len(la), dtype=bool)[best] & ~(fc[best][:, None] & fc[None])
            gap = (la.max(1) - np.where(other, la, -np.inf).max(1)).min()
            conf = np.abs(np.exp(la.max(1)) - 0.3).min()
            if gap > 0.2 and conf > 0.05:
                if np.bincount(best[~fr], minlength=1).max(initial=0) > 1:
                    return False
            elif gap < 0.05:
                return False
            else:
                sure = False
    return True if sure else None


def _check(perm, cost, words, n_iters=20):
    """Returns how many pairs were published and how many were not."""
    B, T, N = perm.shape
    perm = perm.numpy()
    counts = [0, 0]
    for b in range(B):
        assert not words[b, :FIRST].any()
        for t in range(FIRST, T):
            w = words[b, t]
            ready = (w & READY) != 0
            assert ready.all() or not ready.any()          # a whole pair or nothing of it
            want = _decide(cost[b, t - 1], n_iters)
            assert want is None or want == bool(ready.all()), (b, t, want)
            counts[int(not ready.all())] += 1
            if ready.all():
                live = (w & FLAT) == 0
                if (np.bincount(perm[b, t - 1], minlength=N)[live] == 1).all():
                    assert np.array_equal(w[perm[b, t - 1]] & IDX, perm[b, t]), (b, t)
    return counts


@pytest.mark.parametrize("B,T,N,D,dead,decisive,dup,some", [
    (3, 40, 16, 64, 0.0, 8.0, False, (True, False)),     # every match a permutation
    (2, 33, 32, 64, 0.2, 8.0, False, (True, None)),      # dead slots: several waves look at the flat columns
    (4, 12, 31, 64, 0.5, 8.0, False, (True, None)),      # half dead, padding
    (2, 7, 31, 64, 0.0, 8.0, True, (False, True)),       # an exact tie among live slots decides nothing
    (3, 8, 32, 64, 0.2, 0.0, False, (False, True)),      # untrained weights
    (2, 6, 70, 64, 0.1, 8.0, False, (True, None)),
    (1, 5, 128, 64, 0.1, 8.0, False, (True, None)),      # most slots
    (3, 6, 16, 64, 1.0, 8.0, False, (True, False)),      # every slot dead: flat throughout
])
def test_published_pairs(B, T, N, D, dead, decisive, dup, some):
    from hclsm_amd.kernels.slot_tracker import TrackerWeights
    m = _tracker(D, N, decisive, N + T)
    slots, alive = _clips(B, T, N, D, B + N, dead, dup)
    done, left = _check(*_run(slots, alive, TrackerWeights.from_module(m, torch.float32)))
    for have, want in ((done, some[0]), (left, some[1])):
        assert want is None or want == (have > 0), (done, left)


@pytest.mark.parametrize("temperature,n_iters,beside", [
    (0.05, 20, True), (0.039, 20, True), (1.0, 20, None), (0.05, 1024, None), (0.038, 20, False), (0.001, 20, False),
    (0.05, 1025, False)])
def test_only_where_the_order_of_the_rows_cannot_matter(temperature, n_iters, beside):
    """The first column step rounds to one unit of 2e4 / temperature.  Where two such units reach the margin of the
    published matches (0.1 in log units), or rounding can add up over the rounds, the loop does every step."""
    from hclsm_amd.kernels.slot_tracker import TrackerWeights
    m = _tracker(64, 32, 8.0, 7)
    slots, alive = _clips(2, 9, 32, 64, 3, 0.2)
    W = TrackerWeights.from_module(m, torch.float32)
    perm, cost, words = _run(slots, alive, W, n_iters, temperature)
    if beside is not None:
        assert bool((words & READY).any()) == beside
    perm2, _, _ = _run(slots.repeat(200, 1, 1, 1), alive.repeat(200, 1, 1), W, n_iters, temperature)   # loops alone
    assert torch.equal(perm, perm2[:2])
