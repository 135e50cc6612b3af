"""The many-token router's tiles (16, 32 and 64 tokens, chunks in one run or split over four groups of
threads) give the few-token router's bits: ids, weights and scores, at the sizes around each choice."""
from __future__ import annotations

import pytest
import torch

from helpers import SEED

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t,d,e,order", [(160, 4096, 384, "ascending"), (161, 5120, 384, "rank"),
                                         (337, 4096, 384, "ascending"), (673, 5120, 384, "rank"),
                                         (1000, 4096, 384, "ascending"), (1100, 1024, 65, "rank"),
                                         (65, 512, 1000, "ascending"), (2337, 512, 384, "rank"),
                                         (500, 512, 384, "rank"), (6001, 512, 384, "ascending"),
                                         (60, 5120, 1024, "rank")])
def test_tiles_give_the_same_bits(cuda, t, d, e, order):
    from cachalot_amd import synth
    from cachalot_amd.router import route_topk_rows

    w, b = synth.router_weights(SEED, 0, e, d, cuda)
    x = synth.activations(SEED, 5200 + t, t, d, cuda)
    kw = dict(topk=6, score_fn="sqrt_softplus" if order == "ascending" else "sigmoid", order=order)
    idx, wt, sc = route_topk_rows(x, w, b, **kw)
    for t0 in range(0, t, 7):                    # seven tokens: the few-token kernel
        i7, w7, s7 = route_topk_rows(x[t0:t0 + 7], w, b, **kw)
        assert torch.equal(idx[t0:t0 + 7], i7)
        assert torch.equal(wt[t0:t0 + 7].view(torch.int32), w7.view(torch.int32))
        assert torch.equal(sc[t0:t0 + 7].view(torch.int32), s7.view(torch.int32))
