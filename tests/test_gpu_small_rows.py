"""Grouped experts with few rows per expert (small_rows.hip: the weight stream of batched decode,
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


def _check_counts(cuda, what, kind, d, f, times=1):
    """The routes of COUNTS (times over), a lost expert and dropped ids against the oracle, eager and captured."""
    from cachalot_amd.moe_prefill import grouped_experts
    from cachalot_amd.storage.index import affine_format, fp4_format

    fmt = fp4_format(d, f) if kind == "fp4" else affine_format(d, f, bits=kind[0], group_size=kind[1],
                                                               scale_dtype=kind[2])
    E, k = 32, 2
    routes = [e for e, n in COUNTS.items() for _ in range(n * times)] + [LOST] * 5 + [-1, E, 1 << 20, -7, E + 3]
    if kind[:2] == (2, 128):
        routes += [17, 18] * 12                                    # 2.75 routes per expert slot (2.5 to 8 here)
    t = len(routes) // k
    idx = np.asarray(routes, np.int32).reshape(k, t).T.copy()      # 64 routes: two per expert slot
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
    _grouped_check(f"{what} {kind} D={d} F={f}", fmt, 0, bf16_bits_to_f32(xb), np.where(gone, -1, idx), w,
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


@pytest.mark.parametrize("kind,d,f", CASES)
def test_few_rows_per_expert(cuda, kind, d, f, monkeypatch):
    monkeypatch.setenv("CACHALOT_AFFINE_VALU", "0")
    monkeypatch.setenv("CACHALOT_PREFILL_BF16", "0")
    _check_counts(cuda, "few rows", kind, d, f)


# K of a few chunks: waves without a macro of their own (3- and 4-bit); FP4 and 2-bit codes, whose
# rings are three macros deep, need K > 1792 in both projections and take the 16-row tiles here
@pytest.mark.parametrize("kind,d,f", [(kind, d, f) for d, f in ((1024, 640), (128, 64))
                                      for kind in ("fp4", (2, 64, "float16"), (2, 32, "bfloat16"),
                                                   (3, 128, "bfloat16"), (3, 64, "float16"), (3, 32, "float16"),
                                                   (4, 128, "float16"), (4, 64, "bfloat16"), (4, 32, "bfloat16"))])
def test_few_rows_short_in_k(cuda, kind, d, f):
    _check_counts(cuda, "few rows, short K", kind, d, f)


# CACHALOT_PREFILL_BF16=1: two rows per expert slot the 16-row tiles, six the 64-row ones (FP4: 128-row)
@pytest.mark.parametrize("times", [1, 3])
@pytest.mark.parametrize("kind", ["fp4", (2, 64, "float16"), (2, 32, "bfloat16"), (3, 128, "bfloat16"),
                                  (3, 64, "float16"), (3, 32, "float16"), (4, 128, "float16"), (4, 64, "bfloat16"),
                                  (4, 32, "bfloat16")])
def test_general_tiles(cuda, kind, times, monkeypatch):
    monkeypatch.setenv("CACHALOT_PREFILL_BF16", "1")
    _check_counts(cuda, f"general tiles x {times}", kind, 1024, 640, times)


KINDS = ["fp4", (2, 128, "bfloat16"), (2, 64, "float16"), (2, 32, "bfloat16"), (3, 128, "bfloat16"),
         (3, 64, "float16"), (3, 32, "float16"), (4, 128, "float16"), (4, 64, "bfloat16"), (4, 32, "bfloat16")]


def _bank(kind, d, f, E):
    from cachalot_amd.storage.index import affine_format, fp4_format

    fmt = fp4_format(d, f) if kind == "fp4" else affine_format(d, f, bits=kind[0], group_size=kind[1],
                                                               scale_dtype=kind[2])
    return fmt, make_store(fmt, n_layers=1, n_experts=E)


def _three_per_expert(rng, E, device):
    """E tokens, three routes each, every expert with three rows (inside every kind's range)."""
    idx = np.stack([rng.permutation(E) for _ in range(3)], axis=1).astype(np.int32)
    w = rng.dirichlet(np.ones(3), size=E).astype(np.float32)
    return torch.from_numpy(idx).to(device), torch.from_numpy(w).to(device)


@pytest.mark.parametrize("kind", KINDS)
def test_a_strong_element_costs_its_neighbours_no_bits(cuda, kind):
    """One element of every 32 is 2^15 times the others, and the codes (and biases) that meet it are
    zero: the same bits as with that element zero, since bf16 operands carry each element by itself."""
    from cachalot_amd.moe_prefill import grouped_experts

    d, f, E = 2048, 1856, 32
    fmt, store = _bank(kind, d, f, E)
    pool = store.pool
    rec = pool.storage.view(pool.n_slots, pool.record_bytes)
    # code 5 of each 32: byte of the 32's run, bits kept
    keep = {"fp4": [(2, 0x0F)], 2: [(1, 0xF3)], 3: [(1, 0x7F), (2, 0xFC)], 4: [(2, 0x0F)]}["fp4" if kind == "fp4" else kind[0]]
    run = 16 if kind == "fp4" else 4 * kind[0]
    for p in ("w1", "w3"):
        o = pool.offsets[f"{p}.weight"]
        codes = rec[:E, o:o + fmt.tensor_bytes(f"{p}.weight")].unflatten(1, (-1, run))
        for byte, bits in keep:
            codes[:, :, byte] &= bits
        if kind != "fp4":
            o = pool.offsets[f"{p}.biases"]
            rec[:E, o:o + fmt.tensor_bytes(f"{p}.biases")] = 0
    torch.cuda.synchronize()
    idx, w = _three_per_expert(np.random.default_rng(5), E, cuda)
    x = _bf16(osynth.activations(SEED, 5110, E, d), cuda)
    strong, none = x.clone(), x.clone()
    strong.view(E, -1, 32)[:, :, 5] = 2.0 ** 15
    none.view(E, -1, 32)[:, :, 5] = 0.0
    y = [grouped_experts(v, idx, w, pool, store.layer_table(0), want_terms=True)[2] for v in (strong, none)]
    assert torch.equal(y[0].view(torch.int16), y[1].view(torch.int16))
    assert y[1].float().abs().max() > 0


@pytest.mark.parametrize("limit", [10.0, 0.0])
@pytest.mark.parametrize("kind", KINDS)
def test_infinities_and_nan_as_on_the_general_path(cuda, kind, limit, monkeypatch):
    """A token with an infinity or a NaN: NaN, infinities and their signs where the 16-row tiles give
    them; every other token keeps its bits."""
    from cachalot_amd.moe_prefill import grouped_experts

    d, f, E = 2048, 1856, 32
    _, store = _bank(kind, d, f, E)
    idx, w = _three_per_expert(np.random.default_rng(6), E, cuda)
    x = _bf16(osynth.activations(SEED, 5111, E, d), cuda)

    def run(v):
        return grouped_experts(v, idx, w, store.pool, store.layer_table(0), swiglu_limit=limit, want_terms=True)[2]

    finite = run(x)
    for bad in (float("inf"), -float("inf"), float("nan")):
        v = x.clone()
        v[3, 100] = bad
        v[9, d - 1] = bad
        y = run(v)
        monkeypatch.setenv("CACHALOT_GROUPED_SMALL", "1")
        want = run(v)
        monkeypatch.delenv("CACHALOT_GROUPED_SMALL")
        for t in (3, 9):
            for cls in (torch.isnan, torch.isposinf, torch.isneginf):
                assert torch.equal(cls(y[t]), cls(want[t])), (kind, bad, cls.__name__)
        rest = [t for t in range(E) if t not in (3, 9)]
        assert torch.equal(y[rest].view(torch.int16), finite[rest].view(torch.int16)), (kind, bad)


@pytest.mark.parametrize("kind", ["fp4", (2, 128, "bfloat16"), (3, 64, "float16")])
def test_activations_off_the_16_byte_grid(cuda, kind):
    from cachalot_amd.moe_prefill import grouped_experts

    d, f, E = 2048, 1856, 32
    _, store = _bank(kind, d, f, E)
    idx, w = _three_per_expert(np.random.default_rng(7), E, cuda)
    x = _bf16(osynth.activations(SEED, 5112, E, d), cuda)
    flat = torch.empty(E * d + 4, dtype=torch.bfloat16, device=cuda)
    off = flat[4:].view(E, d)
    off.copy_(x)
    assert off.data_ptr() % 16 == 8
    y = [grouped_experts(v, idx, w, store.pool, store.layer_table(0), want_terms=True)[2] for v in (x, off)]
    assert torch.equal(y[0].view(torch.int16), y[1].view(torch.int16))


@pytest.mark.parametrize("hot", [2, 5, 32])
@pytest.mark.parametrize("kind,t", [("fp4", 40), ("fp4", 75), ((2, 128, "bfloat16"), 70), ((2, 128, "bfloat16"), 120),
                                    ((2, 32, "bfloat16"), 30), ((3, 32, "float16"), 70), ((4, 32, "bfloat16"), 330)])
def test_concentrated_and_spread_routes(cuda, kind, t, hot):
    """The list of few-row tiles or, for routes on a few experts, of the other kernels' tiles, chosen on
    the device: both against the oracle, and under capture each as the routes of its replay want it."""
    from cachalot_amd.moe_prefill import grouped_experts

    d, f, E, k = 2048, 1856, 32, 2
    fmt, store = _bank(kind, d, f, E)
    rng = np.random.default_rng(hot + t)
    idx = np.stack([rng.permutation(hot)[:k] for _ in range(t)]).astype(np.int32)
    w = rng.dirichlet(np.ones(k), size=t).astype(np.float32)
    xb = osynth.activations(SEED, 5120 + t, t, d)
    args = (_bf16(xb, cuda), torch.from_numpy(idx).to(cuda), torch.from_numpy(w).to(cuda), store.pool,
            store.layer_table(0))
    routed, out, y = grouped_experts(*args, want_routed=True, want_terms=True)
    _grouped_check(f"{kind} {t} tokens on {hot} experts", fmt, 0, bf16_bits_to_f32(xb), idx, w, _np(routed), _f32(out),
                   _f32(y), E)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        _, gout = grouped_experts(*args)
    for n in (hot, 2, 32, hot):
        args[1].copy_(torch.from_numpy(np.stack([rng.permutation(n)[:k] for _ in range(t)]).astype(np.int32)))
        gout.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(gout, grouped_experts(*args)[1])


@pytest.mark.parametrize("kind", ["fp4", (3, 64, "float16"), (4, 32, "bfloat16")])
def test_several_rounds_of_runs(cuda, kind):
    """A call of more than 2 x 512 x 16 items, dealt in several rounds of runs: a token's terms are the
    bits it gets in a call of few tokens (one round), whatever tiles and runs its rows fall into."""
    from cachalot_amd.moe_prefill import grouped_experts

    d, f, E, t, k = 2048, 2048, 320, 200, 4
    _, store = _bank(kind, d, f, E)
    rng = np.random.default_rng(11)
    idx = torch.from_numpy(np.stack([rng.permutation(E)[:k] for _ in range(t)]).astype(np.int32)).to(cuda)
    w = torch.from_numpy(rng.dirichlet(np.ones(k), size=t).astype(np.float32)).to(cuda)
    x = _bf16(osynth.activations(SEED, 5130, t, d), cuda)

    def run(a, b):
        return grouped_experts(x[a:b], idx[a:b], w[a:b], store.pool, store.layer_table(0), want_terms=True)[2]

    whole = run(0, t)
    parts = torch.cat([run(a, a + 8) for a in range(0, t, 8)])
    assert torch.equal(whole.view(torch.int16), parts.view(torch.int16))
