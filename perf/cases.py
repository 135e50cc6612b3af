"""The work this framework is used for, as measurable cases.

A case is one pass through a public entry point over a fully resident expert bank:

* ``tokens == 1``: ``moe_layer_forward`` for one token through ``layers`` MoE layers, each
  with an activation of its own (attention sits between the MoE layers of a model, so no
  layer reads another's output here);
* ``tokens > 1``: ``moe_prefill_grouped`` over that many rows (batched decode, verification
  of drafted tokens, prefill chunks);
* ``bank == "shared"``: ``shared_expert_forward_batched``, the FP8 shared expert alone.

``captured`` passes replay a HIP graph of the same calls, recorded once, which is how a
decode loop runs them; the others call the entry point eagerly.  The banks, routers and
activations have the distributions of a model's: E2M1 codes with E8M0 block scales,
min/max-fitted affine groups (bias near -s (2^bits - 1) / 2), normalised activations with a
few strong channels, a router with a small bias, or one skewed so that the experts' loads
follow a Zipf law, as text of one kind gives.
"""
from __future__ import annotations

import math

import torch

from cachalot_amd.cache.resident_store import ResidentExpertStore
from cachalot_amd.moe_layer import moe_layer_forward
from cachalot_amd.moe_prefill import moe_prefill_grouped
from cachalot_amd.shared_expert import shared_expert_forward_batched
from cachalot_amd.storage.index import affine_format, fp4_format

LIMIT = 10.0

# bank name -> (bits, group, scale dtype); bits 0: FP4 E2M1 / E8M0
BANKS = {
    "fp4": (0, 32, ""),
    "q2_f16": (2, 128, "float16"),
    "q2_bf16": (2, 128, "bfloat16"),
    "oq3e": (3, 64, "float16"),
    "a3_g128": (3, 128, "bfloat16"),
    "a4_g64": (4, 64, "float16"),
    "a4_g128": (4, 128, "bfloat16"),
}


def _case(name, bank, tokens, *, d=4096, f=2880, experts=384, topk=6, layers=1, shared=False, captured=False,
          score="sigmoid", order="ascending", zipf=False):
    case = dict(bank=bank, tokens=tokens, d=d, f=f, experts=experts, topk=topk, layers=layers, shared=shared,
                captured=captured, score=score, order=order, zipf=zipf)
    return dict(name=name, **case) if name else case


def listed():
    return [
        # the smallest call: one token, one layer, called eagerly (a program's first tokens, a test)
        _case("call_q2", "q2_bf16", 1),
        # one token through part of a decoder's stack of 2-bit layers, the headline workload
        _case("decode_q2", "q2_f16", 1, layers=8, captured=True),
        # the shipped FP4 checkpoint with its FP8 shared expert, the whole MoE layer of a decode step
        _case("decode_fp4_shared", "fp4", 1, layers=4, shared=True, captured=True, score="sqrt_softplus"),
        # the 3-bit bank at the other layer shape (5120 x 2304)
        _case("decode_oq3e", "oq3e", 1, d=5120, f=2304, layers=6, captured=True),
        # sixteen sequences decoded together over the 2-bit bank
        _case("batch16_q2", "q2_f16", 16, layers=2, captured=True),
        # a batch over the FP4 bank: a few routes per expert
        _case("batch24_fp4", "fp4", 24, layers=2),
        # an odd number of drafted tokens verified over the 3-bit bank
        _case("verify7_oq3e", "oq3e", 7, layers=2),
        # a short ragged prompt, 2-bit bank at 5120 x 2304, with the shared expert
        _case("chunk301_q2_shared", "q2_bf16", 301, d=5120, f=2304, shared=True, score="sqrt_softplus"),
        # a ragged prompt over FP4 with the shared expert
        _case("chunk1000_fp4_shared", "fp4", 1000, shared=True, score="sqrt_softplus"),
        # a prefill chunk over the 3-bit bank
        _case("prefill2048_oq3e", "oq3e", 2048, order="rank"),
        # the full prefill chunk over FP4 with skewed expert loads
        _case("prefill4096_fp4", "fp4", 4096, zipf=True),
        # the shared expert's own GEMMs over a prefill chunk
        _case("shared4096", "shared", 4096),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    what = rng.choice(["decode", "decode", "batch", "batch", "rows", "rows", "rows", "shared"])
    d, f, experts = rng.choice([(4096, 2880, 384), (4096, 2880, 384), (5120, 2304, 384), (5120, 2304, 256),
                                (1024, 640, 64)])
    if what == "shared":
        return _case("", "shared", _log_int(rng, 2, 4096), d=d, f=f, experts=0, topk=0)
    bank = rng.choice(["fp4", "fp4", "q2_f16", "q2_bf16", "oq3e", "oq3e", rng.choice(["a3_g128", "a4_g64", "a4_g128"])])
    common = dict(d=d, f=f, experts=experts, topk=rng.choice([4, 6, 6, 6, 8]), shared=rng.random() < 0.3,
                  score=rng.choice(["sigmoid", "sqrt_softplus"]), order=rng.choice(["ascending", "ascending", "rank"]))
    if what == "decode":
        return _case("", bank, 1, layers=rng.randint(4, 6), captured=rng.random() < 0.8, **common)
    if what == "batch":
        return _case("", bank, _log_int(rng, 2, 64), layers=2, captured=rng.random() < 0.5, **common)
    # the affine banks past 2 bits stay at half the chunk: more work per row
    return _case("", bank, _log_int(rng, 48, 3000 if BANKS[bank][0] in (0, 2) else 2000), zipf=rng.random() < 0.4,
                 **common)


# ------------------------------------------------------------------ inputs ---
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) & 0x7FFFFFFFFFFF)
    return g


def _format(case):
    bits, group, dt = BANKS[case["bank"]]
    if bits == 0:
        return fp4_format(case["d"], case["f"])
    return affine_format(case["d"], case["f"], bits=bits, group_size=group, scale_dtype=dt)


def _random_bytes(n, g):
    words = torch.empty((n + 7) // 8, dtype=torch.int64, device="cuda")
    words.random_(-(2 ** 63), 2 ** 63 - 1, generator=g)
    return words.view(torch.uint8)[:n]


def _expert_tensors(case, fmt, n, g):
    """The stacked tensors of one layer's n experts: name -> uint8 [n, bytes]."""
    bits, group, dt = BANKS[case["bank"]]
    out = {}
    for proj, k in (("w1", case["d"]), ("w2", case["f"]), ("w3", case["d"])):
        name = f"{proj}.weight"
        rows = fmt.shapes[name][0]
        w = _random_bytes(n * fmt.tensor_bytes(name), g).view(n, rows, -1)
        if bits:
            w[:, :, k * bits // 8:] = 0            # the padding of a partial last group
        out[name] = w.view(n, -1)
        if bits == 0:
            out[f"{proj}.scale"] = torch.randint(118, 122, (n, fmt.tensor_bytes(f"{proj}.scale")), device="cuda",
                                                 dtype=torch.uint8, generator=g)
            continue
        groups = fmt.shapes[f"{proj}.scales"][1]
        top = {2: 0.05, 3: 0.024, 4: 0.012}[bits]
        s = torch.rand(n, rows * groups, device="cuda", generator=g).mul_(0.9 * top).add_(0.1 * top)
        b = torch.randn(n, rows * groups, device="cuda", generator=g).mul_(0.2).add_(1.0).mul_(s)
        b.mul_(-0.5 * (2 ** bits - 1))
        tt = getattr(torch, dt)
        out[f"{proj}.scales"] = s.to(tt).view(torch.uint8)
        out[f"{proj}.biases"] = b.to(tt).view(torch.uint8)
    return out


def _activations(case, g):
    t, d = case["tokens"], case["d"]
    x = torch.randn(case["layers"], t, d, device="cuda", generator=g)
    gain = torch.ones(d, device="cuda")
    gain[torch.randint(0, d, (d // 64,), device="cuda", generator=g)] = 6.0
    return (x * gain).to(torch.bfloat16)


def _gates(case, g):
    e, d = case["experts"], case["d"]
    out = []
    for _ in range(case["layers"]):
        w = (torch.randn(e, d, device="cuda", generator=g) * 0.02).to(torch.bfloat16)
        b = torch.randn(e, device="cuda", generator=g) * 0.01
        if case["zipf"]:
            rank = torch.randperm(e, device="cuda", generator=g).float()
            b = b + 0.5 * (rank + 1.0) ** -1.1
        out.append((w, b))
    return out


def _shared_sets(case, g):
    """One FP8 shared expert per layer: E4M3 weights, E8M0 scales per 32 x 32 block."""
    d, f = case["d"], case["f"]
    sets = []
    for _ in range(case["layers"]):
        s = {}
        for p, n, k in (("w1", f, d), ("w3", f, d), ("w2", d, f)):
            s[p] = torch.randn(n, k, device="cuda", generator=g).to(torch.float8_e4m3fn).view(torch.uint8)
            s[p + "_scales"] = torch.randint(120, 123, ((n + 31) // 32, k // 32), device="cuda", dtype=torch.uint8,
                                             generator=g)
        sets.append(s)
    return sets


def _calls(case, state):
    """The pass: every layer's call, in order."""
    out = []
    for la in range(case["layers"]):
        w, b = state["gates"][la]
        shared = {f"shared_{n}": t for n, t in state["shared"][la].items()} if case["shared"] else {}
        kw = dict(layer_id=la, gate_weight=w, gate_bias=b, expert_index=None, expert_store=state["store"],
                  topk=case["topk"], score_fn=case["score"], order=case["order"], swiglu_limit=LIMIT, **shared)
        if case["tokens"] == 1:
            y, route = moe_layer_forward(state["x"][la][0], **kw)
        else:
            y, route = moe_prefill_grouped(state["x"][la], **kw)
        out.append((y, route.indices, route.weights, route.scores))
    return out


def prepare(case, seed):
    g = _gen(seed)
    state = {"case": case, "x": _activations(case, g)}
    if case["bank"] == "shared":
        state["shared"] = _shared_sets(case, g)
        return state
    fmt, e, layers = _format(case), case["experts"], case["layers"]
    state["gates"] = _gates(case, g)
    state["shared"] = _shared_sets(case, g) if case["shared"] else None
    store = ResidentExpertStore(fmt=fmt, n_slots=layers * e, n_layers=layers, n_experts=e, transient_slots=1,
                                device="cuda")
    store.preload([(la, i) for la in range(layers) for i in range(e)], lambda key, slot: None)
    pool = store.pool
    records = pool.storage.view(pool.n_slots, pool.record_bytes)
    for la in range(layers):                       # slot of (layer, expert) = layer * e + expert
        for name, t in _expert_tensors(case, fmt, e, g).items():
            records[la * e:(la + 1) * e, pool.offsets[name]:pool.offsets[name] + t.shape[1]] = t
    store.track_slots()
    state["store"] = store
    if case["captured"]:
        _calls(case, state)                        # workspaces exist before the capture
        torch.cuda.synchronize()
        state["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(state["graph"]):
            state["out"] = _calls(case, state)
    return state


def run(state):
    case = state["case"]
    if case["bank"] == "shared":
        return shared_expert_forward_batched(state["x"][0], **state["shared"][0], swiglu_limit=LIMIT)
    if case["captured"]:
        state["graph"].replay()
        return state["out"]
    return _calls(case, state)


# -------------------------------------------------------------- properties ---
def _touched(case):
    """Distinct experts a layer's routes reach (uniform routing; a skewed chunk still reaches nearly all)."""
    e = case["experts"]
    return e * (1.0 - (1.0 - case["topk"] / e) ** case["tokens"])


def work(case):
    t, d, f, e, k = case["tokens"], case["d"], case["f"], case["experts"], case["topk"]
    shared_b, shared_f = 3 * d * f + 3 * (d // 32) * ((f + 31) // 32), 6.0 * t * d * f
    io = 2 * t * d * 2
    if case["bank"] == "shared":
        return {"bytes": shared_b + io, "flops": shared_f}
    expert = _format(case).algorithmic_bytes
    b = _touched(case) * expert + e * d * 2 + e * 4 + io + t * (e * 4 + k * 8)
    fl = 6.0 * t * k * d * f + 2.0 * t * e * d
    if case["shared"]:
        b, fl = b + shared_b, fl + shared_f
    return {"bytes": case["layers"] * b, "flops": case["layers"] * fl}


def tolerance(case):
    # against 64-bit sums without the bf16 points: outputs 1.7e-3 (shared expert, FP4 decode) to
    # 3.9e-3 off over all banks and sizes; two 32-bit orders differ by the flips of those roundings
    return {"rel": 1e-2, "max": 0.1}


# ------------------------------------------------------------------- exact ---
_E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0, -0.0, -0.5, -1.0, -1.5, -2.0, -3.0, -4.0, -6.0)


def _dense(case, fmt, tens, i, proj, k):
    """Expert i's matrix as float64 [rows, k]."""
    bits, group, dt = BANKS[case["bank"]]
    rows = fmt.shapes[f"{proj}.weight"][0]
    raw = tens[f"{proj}.weight"][i].view(rows, -1)
    if bits == 0:
        table = torch.tensor(_E2M1, dtype=torch.float64, device="cuda")
        q = torch.stack([table[(raw & 15).long()], table[(raw >> 4).long()]], -1).view(rows, k // 32, 32)
        s = torch.exp2(tens[f"{proj}.scale"][i].view(rows, -1).double() - 127.0)
        return (q * s[:, :, None]).view(rows, k)
    shifts = torch.arange(8, device="cuda")
    if bits == 3:                                  # eight codes in three bytes, low bits first
        b3 = raw.view(rows, -1, 3).long()
        word = b3[..., 0] | (b3[..., 1] << 8) | (b3[..., 2] << 16)
        q = (word[..., None] >> (3 * shifts)) & 7
    else:
        q = (raw.long()[..., None] >> (bits * shifts[:8 // bits])) & (2 ** bits - 1)
    q = q.reshape(rows, -1, group).double()
    s = tens[f"{proj}.scales"][i].view(getattr(torch, dt)).view(rows, -1).double()
    b = tens[f"{proj}.biases"][i].view(getattr(torch, dt)).view(rows, -1).double()
    return (q * s[:, :, None] + b[:, :, None]).view(rows, -1)[:, :k]


def _swiglu(g, u):
    return torch.nn.functional.silu(g.clamp(max=LIMIT)) * u.clamp(-LIMIT, LIMIT)


def _act_quant(v):
    """Blocks of 32: the smallest power of two that takes the block into E4M3's range, E4M3 rounding."""
    blocks = v.double().view(v.shape[0], -1, 32)
    amax = blocks.abs().amax(-1, keepdim=True).clamp(min=1e-4)
    s = torch.exp2(torch.ceil(torch.log2(amax / 448.0)))
    return ((blocks / s).float().to(torch.float8_e4m3fn).double() * s).view(v.shape)


def _shared_exact(case, s, x):
    def dense(p):
        w = s[p].view(torch.float8_e4m3fn).double()
        sc = torch.exp2(s[p + "_scales"].double() - 127.0)
        return w * sc.repeat_interleave(32, 0)[:w.shape[0]].repeat_interleave(32, 1)

    q = _act_quant(x)
    h = _swiglu((q @ dense("w1").t()).to(torch.bfloat16).double(), (q @ dense("w3").t()).to(torch.bfloat16).double())
    return _act_quant(h.to(torch.bfloat16)) @ dense("w2").t()


def exact(case, seed):
    g = _gen(seed)
    xs = _activations(case, g)
    if case["bank"] == "shared":
        return _shared_exact(case, _shared_sets(case, g)[0], xs[0])
    fmt, e, k = _format(case), case["experts"], case["topk"]
    gates = _gates(case, g)
    shared = _shared_sets(case, g) if case["shared"] else None
    out = []
    for la in range(case["layers"]):
        tens = _expert_tensors(case, fmt, e, g)
        x = xs[la].double()
        w, b = gates[la]
        z = x @ w.double().t()
        scores = torch.sigmoid(z) if case["score"] == "sigmoid" else torch.nn.functional.softplus(z).sqrt()
        idx = torch.topk(scores + b.double(), k, dim=-1).indices          # largest first
        if case["order"] == "ascending":
            idx = idx.flip(-1)
        wt = torch.gather(scores, 1, idx)
        wt = wt / wt.sum(-1, keepdim=True) * 1.5
        y = torch.zeros_like(x)
        for i in torch.unique(idx).tolist():
            t, slot = torch.nonzero(idx == i, as_tuple=True)
            xi = x[t]
            h = _swiglu(xi @ _dense(case, fmt, tens, i, "w1", case["d"]).t(),
                        xi @ _dense(case, fmt, tens, i, "w3", case["d"]).t()) * wt[t, slot][:, None]
            y.index_add_(0, t, h @ _dense(case, fmt, tens, i, "w2", case["f"]).t())
        if shared is not None:
            y = y + _shared_exact(case, shared[la], xs[la])
        parts = (y, None, wt, scores)
        out.append(tuple(p if p is None or case["tokens"] > 1 else p[0] for p in parts))
    return out
