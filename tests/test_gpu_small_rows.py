"""Grouped experts with few rows per expert (small_rows_mx.hip: the weight stream of batched decode,
drafted tokens and short prompts) against the oracle, every bank kind: experts of 1 .. 17 rows around
the 4- and 8-row tile edges, an expert without a slot, dropped ids, K with partial chunks and groups,
weight slices past F."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from helpers import SEED, make_store
from oracle import synth as osynth
from oracle.bf16 import bf16_bits_to_f32
from test_gpu_workloads import _bf16, _f32, _grouped_check, _np

pytestmark = pytest.mark.gpu

# rows per expert: 1, and one below, at and above the 4- and 8-row tiles, two tiles and more
COUNTS = {0: 1, 3: 3, 4: 4, 9: 5, 11: 7, 12: 8, 20: 9, 31: 17}
LOST = 7                                    # five rows of an expert that is not resident

CASES = [(kind, 2048, 1856) for kind in ("fp4", (2, 128, "bfloat16"), (2, 64, "float16"), (2, 32, "bfloat16"),
                                         (3, 128, "bfloat16"), (3, 64, "float16"), (3, 32, "float16"),
                                         (4, 128, "float16"), (4, 64, "bfloat16"), (4, 32, "bfloat16"))]
CASES += [("fp4", 5120, 2304), ((2, 128, "float16"), 4096, 2880), ((3, 64, "float16"), 4096, 2880)]


@pytest.mark.parametrize("kind,d,f", CASES)
def test_few_rows_per_expert(cuda, kind, d, f, monkeypatch):
    from cachalot_amd.moe_prefill import grouped_experts
    from cachalot_amd.storage.index import affine_format, fp4_format

    monkeypatch.setenv("CACHALOT_AFFINE_VALU", "0")
    monkeypatch.setenv("CACHALOT_PREFILL_BF16", "0")
    fmt = fp4_format(d, f) if kind == "fp4" else affine_format(d, f, bits=kind[0], group_size=kind[1],
                                                               scale_dtype=kind[2])
    E, t, k = 32, 32, 2
    routes = [e for e, n in COUNTS.items() for _ in range(n)] + [LOST] * 5 + [-1, E, 1 << 20, -7, E + 3]
    idx = np.asarray(routes, np.int32).reshape(k, t).T.copy()      # 64 routes: two per expert slot (2-bit: 1.5 to 8)
    rng = np.random.default_rng(d + f)
    idx = idx[rng.permutation(t)]
    w = rng.dirichlet(np.ones(k), size=t).astype(np.float32)
    store = make_store(fmt, n_layers=1, n_experts=E)
    table = store.layer_table(0).clone()
    table[LOST] = -1
    xb = osynth.activations(SEED, 5100, t, d)
    ab = osynth.activations(SEED, 5101, t, d)
    args = (_bf16(xb, cuda), torch.from_numpy(idx).to(cuda), torch.from_numpy(w).to(cuda), store.pool, table)
    kw = dict(addend=_bf16(ab, cuda), want_routed=True, want_terms=True)
    routed, out, y = grouped_experts(*args, **kw)
    gone = (idx < 0) | (idx >= E) | (idx == LOST)
    yf = _f32(y)
    assert not yf[gone].any()
    _grouped_check(f"few rows {kind} D={d} F={f}", fmt, 0, bf16_bits_to_f32(xb), np.where(gone, -1, idx), w,
                   _np(routed), _f32(out), yf, E, addend=bf16_bits_to_f32(ab))
    # the same under capture, replayed with other work in between
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        _, gout, _ = grouped_experts(*args, **kw)
    for _ in range(3):
        gout.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(gout, out)
        grouped_experts(*args, **kw)
