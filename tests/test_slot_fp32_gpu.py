"""The fp32 slot-attention forward at the edges of its 16-wide blocks (tokens, slots, columns) and where a width does
not allow four-element loads, against the numpy oracle."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import slot_attention as osa
from oracle.ssm_scan import normwise_rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,M,N,d,hidden,d_in", [
    (1, 1, 1, 16, 16, 16),       # smallest
    (2, 15, 17, 48, 64, 32),     # one below / above a block
    (3, 33, 16, 64, 20, 36),     # hidden and d_in not multiples of 16
    (2, 196, 65, 80, 160, 20),   # five slot blocks, the last of one slot
    (1, 257, 128, 32, 48, 64),   # most slots, past 256 tokens
    (40, 64, 12, 192, 384, 48),  # enough rows for the wide linear kernels
])
@pytest.mark.parametrize("renorm", [False, True])
def test_forward_matches_oracle(B, M, N, d, hidden, d_in, renorm):
    from hclsm_amd.kernels import slot_iteration as si
    g = torch.Generator().manual_seed(B + M + N + d)
    r = lambda *s: torch.randn(*s, generator=g)
    w = dict(w_q=r(d, d) / d ** 0.5, w_k=r(d, d_in) / d_in ** 0.5, w_v=r(d, d_in) / d_in ** 0.5,
             w_ih=r(3 * d, d) / d ** 0.5, w_hh=r(3 * d, d) / d ** 0.5, w1=r(hidden, d) / d ** 0.5,
             w2=r(d, hidden) / hidden ** 0.5, b_ih=0.1 * r(3 * d), b_hh=0.1 * r(3 * d), b1=0.1 * r(hidden),
             b2=0.1 * r(d), ln_pre_w=1 + 0.1 * r(d), ln_pre_b=0.1 * r(d), ln_mlp_w=1 + 0.1 * r(d),
             ln_mlp_b=0.1 * r(d), ln_in_w=1 + 0.1 * r(d_in), ln_in_b=0.1 * r(d_in))
    tokens, slots0 = r(B, M, d_in), r(B, N, d)
    mode = si.CONFIG2_MODE if renorm else si.REFERENCE_MODE
    W = si.SlotWeights.from_dict(w, torch.float32, "cuda")
    got = si.slot_attention_forward(tokens.cuda(), slots0.cuda(), W, 2, mode)
    ref = osa.slot_attention_forward(tokens.double().numpy(), slots0.double().numpy(),
                                     {n: t.double().numpy() for n, t in w.items()}, 2, logit_clamp=mode.logit_clamp,
                                     renorm_eps=mode.renorm_eps, slot_clamp=mode.slot_clamp)
    assert normwise_rel_err(got.double().cpu().numpy(), np.asarray(ref)) <= 1e-5   # fp32 sums, two iterations
