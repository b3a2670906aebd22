"""The work whose speed is kept track of, case by case.

A case is one call, or one short sequence of calls, that a serving engine makes
through the package's public entry points: attention over a paged KV cache
(plan prepared, ``Plan.run``), the per-token operators around it (``norm``,
``norm_rope_append``, ``silu_mul``), and a decode step replayed from a HIP
graph after a prepare.  Sequence lengths come from the case alone (its
``lens_seed``); page tables and tensor contents come from the seed.
"""

import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "flashengine.cpp_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import feattn  # noqa: E402
from feattn import workloads as W  # noqa: E402

DIM = 128
EPS = 1e-6
THETA = 1e6
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}


def _attention(name, hq, hkv, seqs=0, rows=1, ctx=(0, 0), chunks=0, tokens=0, prefix=(0, 0), causal=True,
               dtype="bf16", lse=False, lens_seed=1):
    """`seqs` sequences with `rows` new tokens each over ctx[0]..ctx[1] cached
    ones, and `chunks` prompt chunks of `tokens` new tokens together, each
    over prefix[0]..prefix[1] cached ones."""
    return {"name": name, "kind": "attention", "hq": hq, "hkv": hkv, "seqs": seqs, "rows": rows, "ctx_lo": ctx[0],
            "ctx_hi": ctx[1], "chunks": chunks, "tokens": tokens, "prefix_lo": prefix[0], "prefix_hi": prefix[1],
            "causal": causal, "dtype": dtype, "lse": lse, "lens_seed": lens_seed}


def _norm(name, rows, width, residual=True, dtype="bf16"):
    return {"name": name, "kind": "norm", "rows": rows, "width": width, "residual": residual, "dtype": dtype}


def _append(name, rows, hq, hkv, dtype="bf16"):
    return {"name": name, "kind": "append", "rows": rows, "hq": hq, "hkv": hkv, "dtype": dtype}


def _silu(name, rows, width, dtype="bf16"):
    return {"name": name, "kind": "silu", "rows": rows, "width": width, "dtype": dtype}


def _step(name, hq, hkv, seqs, ctx, hidden, inner, layers, dtype="bf16", lens_seed=1):
    return {"name": name, "kind": "step", "hq": hq, "hkv": hkv, "seqs": seqs, "ctx_lo": ctx[0], "ctx_hi": ctx[1],
            "hidden": hidden, "inner": inner, "layers": layers, "dtype": dtype, "lens_seed": lens_seed}


def listed():
    return [
        # A few short conversations on a small model: one attention call of a
        # decode step, bound by launches and latency.
        _attention("decode_small", 16, 8, seqs=4, ctx=(511, 511)),
        # A full decode batch of an 8B-class model, ragged contexts: the
        # headline call, bound by the KV bytes.  With the log-sum-exp output.
        _attention("decode_8b", 32, 8, seqs=64, ctx=(511, 4095), lse=True, lens_seed=2),
        # Verification of 4 draft tokens + 1 per sequence, float16, five query
        # heads per kv head: several rows per sequence, ragged contexts.
        _attention("verify_f16", 40, 8, seqs=24, rows=5, ctx=(200, 6000), dtype="f16", lens_seed=7),
        # DFlash draft blocks: 16 rows that see each other and a long context.
        _attention("dflash_blocks", 32, 8, seqs=32, rows=16, ctx=(2048, 16384), causal=False, lens_seed=5),
        # The prefill budget of an 8B-class model filled by chunks of eight
        # prompts, some of them over a cached prefix.
        _attention("prefill_8b", 32, 8, chunks=8, tokens=8192, prefix=(0, 2048), lens_seed=3),
        # One user's prompt of odd length on a small model, nothing cached:
        # time to the first token.
        _attention("prefill_prompt", 16, 8, chunks=1, tokens=777, dtype="f16"),
        # One chunk of a long document: 2048 new tokens over 30000 cached.
        _attention("prefill_long", 32, 4, chunks=1, tokens=2048, prefix=(30000, 30000)),
        # A mixed step: 256 decoding sequences and 2 prompt chunks, eight
        # query heads per kv head.
        _attention("mixed_30b", 32, 4, seqs=256, ctx=(1023, 8191), chunks=2, tokens=2048, prefix=(4096, 4096),
                   lens_seed=4),
        # The norm before a layer's projections at the prefill budget, the
        # residual added and written.
        _norm("norm_prefill", 8192, 4096),
        # q/k norm, RoPE and the paged append of the same tokens.
        _append("append_prefill", 8192, 32, 8),
        # The gated activation of the same tokens.
        _silu("silu_prefill", 8192, 12288),
        # A decode step of a small batch as an engine runs it: prepare, then
        # the layers' own kernels replayed from a captured graph.
        _step("graph_step", 32, 8, seqs=12, ctx=(100, 2047), hidden=4096, inner=12288, layers=4, lens_seed=11),
    ]


_HEADS = [(16, 8), (32, 8), (32, 4), (40, 8)]


def _log_int(rng, lo, hi):
    """An integer of [lo, hi], spread evenly over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "verify", "block", "prefill", "prefill", "mixed", "norm", "append", "silu",
                       "step"])
    hq, hkv = rng.choice(_HEADS)
    dtype = rng.choice(["bf16", "bf16", "f16"])
    ls = rng.randrange(1, 1 << 20)
    if kind in ("decode", "verify", "block"):
        most = {"decode": 500000, "verify": 250000, "block": 300000}[kind]  # cached tokens of the batch
        hi = _log_int(rng, 16, 32768)
        seqs = min(_log_int(rng, 1, 256 if kind == "decode" else 64), max(1, most // hi))
        rows = {"decode": 1, "verify": rng.randint(2, 8), "block": rng.choice([8, 16, 16])}[kind]
        c = _attention("", hq, hkv, seqs=seqs, rows=rows, ctx=(rng.randint(1, hi), hi), causal=kind != "block",
                       dtype=dtype, lse=rng.random() < 0.3, lens_seed=ls)
    elif kind == "prefill":
        tokens = _log_int(rng, 64, 8192)
        chunks = min(rng.randint(1, 8), max(1, tokens // 64))
        prefix = min(rng.choice([0, _log_int(rng, 16, 30000)]), (2048 * 30000 * 32 // hq) // tokens)
        c = _attention("", hq, hkv, chunks=chunks, tokens=tokens, prefix=(rng.randint(0, prefix), prefix),
                       dtype=dtype, lens_seed=ls)
    elif kind == "mixed":
        hi = _log_int(rng, 64, 8191)
        tokens = _log_int(rng, 64, 2048)
        prefix = _log_int(rng, 16, 4096)
        c = _attention("", hq, hkv, seqs=min(_log_int(rng, 2, 256), max(2, 500000 // hi)), ctx=(rng.randint(1, hi), hi),
                       chunks=rng.randint(1, 2), tokens=tokens, prefix=(rng.randint(0, prefix), prefix), dtype=dtype,
                       lens_seed=ls)
    elif kind == "norm":
        width = rng.choice([128, 1000, 4096, 5120, 8 * rng.randint(16, 1024), rng.randint(100, 6000)])
        c = _norm("", _log_int(rng, 1, 8192), width, rng.random() < 0.7, dtype)
    elif kind == "append":
        c = _append("", _log_int(rng, 1, 8192), hq, hkv, dtype)
    elif kind == "silu":
        width = rng.choice([3072, 12288, 8 * rng.randint(16, 1536), rng.randint(100, 6000)])
        c = _silu("", _log_int(rng, 1, 8192), width, dtype)
    else:
        hi = _log_int(rng, 32, 4095)
        c = _step("", hq, hkv, rng.randint(1, 24), (rng.randint(1, hi), hi), 128 * rng.randint(8, 40),
                  128 * rng.randint(16, 100), rng.randint(2, 4), dtype, ls)
    del c["name"]
    return c


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------

def _lens(case):
    """(cached tokens, new tokens) of every sequence: from the case alone."""
    r = np.random.default_rng(case["lens_seed"])
    starts = r.integers(case["ctx_lo"], case["ctx_hi"] + 1, size=case["seqs"]).tolist()
    rows = [case.get("rows", 1)] * case["seqs"]
    n = case.get("chunks", 0)
    if n:
        starts += r.integers(case["prefix_lo"], case["prefix_hi"] + 1, size=n).tolist()
        least = min(64, case["tokens"] // n)
        rows += [least + int(e) for e in r.multinomial(case["tokens"] - least * n, np.full(n, 1.0 / n))]
    return starts, rows


def _randn(shape, gen, dtype, scale=1.0):
    x = torch.randn(shape, generator=gen, device="cuda", dtype=dtype)
    return x.mul_(scale) if scale != 1.0 else x


def _weight(n, gen, dtype):
    return (1 + 0.1 * torch.randn(n, generator=gen, device="cuda")).to(dtype)


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _batch(case, seed):
    starts, rows = _lens(case)
    return W.make_batch(case["hq"], case["hkv"], starts, rows, seed=int(seed) % (1 << 30), extra_pages=1)


def _meta(b):
    """The CSR arrays as C arrays, as a caller that prepares every step holds them."""
    return [feattn._i32(x) for x in (b.qo, b.kv, b.pages, b.last)]


def prepare(case, seed):
    """Random normal activations (a norm stands before q and k, so their
    elements are of order one in earnest too), pages in random order."""
    kind, dt = case["kind"], DTYPES[case["dtype"]]
    gen = _gen(seed)
    bf16 = dt == torch.bfloat16
    st = {"case": dict(case), "bf16": bf16}
    if kind == "attention":
        b = _batch(case, seed)
        shape = (b.blocks + 1, b.page, b.hkv, DIM)
        st.update(kc=_randn(shape, gen, dt), vc=_randn(shape, gen, dt), q=_randn((b.rows, b.hq, DIM), gen, dt))
        st["out"] = torch.empty_like(st["q"])
        st["lse"] = torch.empty(b.rows, b.hq, device="cuda") if case["lse"] else None
        st["plan"] = feattn.Plan(b.hq, b.hkv, DIM, b.page, b.batch, b.max_pages(), bf16, b.blocks)
        st["plan"].prepare(*_meta(b), b.batch, b.rows)
        st["batch"] = b
    elif kind == "norm":
        shape = (case["rows"], case["width"])
        st.update(x=_randn(shape, gen, dt), w=_weight(case["width"], gen, dt))
        st["res"] = _randn(shape, gen, dt, 3.0) if case["residual"] else None
        st["out"] = torch.empty_like(st["x"])
        st["new_res"] = torch.empty_like(st["x"]) if case["residual"] else None
    elif kind == "append":
        rows, heads = case["rows"], case["hq"] + 2 * case["hkv"]
        pages = (rows + 15) // 16 + 1
        g = torch.Generator().manual_seed(int(seed))
        slots = torch.randperm(pages, generator=g)[:, None] * 16 + torch.arange(16)[None]  # tokens fill pages in turn
        st.update(qkv=_randn((rows, heads * DIM), gen, dt, 2.0), qw=_weight(DIM, gen, dt), kw=_weight(DIM, gen, dt),
                  kc=_randn((pages, 16, case["hkv"], DIM), gen, dt), vc=_randn((pages, 16, case["hkv"], DIM), gen, dt),
                  q=torch.empty((rows, case["hq"], DIM), device="cuda", dtype=dt),
                  slots=slots.reshape(-1)[:rows].cuda(), cache_slots=pages * 16,
                  pos=(torch.arange(rows) % 4096 + int(torch.randint(0, 4096, (), generator=g))).cuda(),
                  table=_table(8192))
    elif kind == "silu":
        st["gu"] = _randn((case["rows"], 2 * case["width"]), gen, dt, 2.0)
        st["out"] = torch.empty((case["rows"], case["width"]), device="cuda", dtype=dt)
    else:
        _prepare_step(st, case, seed, gen, dt)
    return st


def _table(max_pos):
    t = torch.empty(max_pos, DIM, device="cuda")
    feattn.rope_table(t, max_pos, DIM, THETA)
    return t


def _prepare_step(st, case, seed, gen, dt):
    b = _batch(case, seed)
    rows, hq, hkv, hidden, inner = b.rows, b.hq, b.hkv, case["hidden"], case["inner"]
    st.update(batch=b, meta=_meta(b), table=_table(8192), pos=torch.from_numpy(b.positions).cuda(),
              slots=torch.from_numpy(b.slots).cuda(), layers=[])
    for _ in range(case["layers"]):
        # What the projections between the kernels write stands in buffers of
        # its own: hidden states, q | k | v heads, gate | up.
        shape = (b.blocks + 1, b.page, hkv, DIM)
        st["layers"].append({
            "x": _randn((rows, hidden), gen, dt), "res": _randn((rows, hidden), gen, dt, 3.0),
            "w1": _weight(hidden, gen, dt), "w2": _weight(hidden, gen, dt), "qw": _weight(DIM, gen, dt),
            "kw": _weight(DIM, gen, dt), "qkv": _randn((rows, (hq + 2 * hkv) * DIM), gen, dt, 2.0),
            "y": _randn((rows, hidden), gen, dt), "gu": _randn((rows, 2 * inner), gen, dt, 2.0),
            "kc": _randn(shape, gen, dt), "vc": _randn(shape, gen, dt),
            **{k: torch.empty((rows, hidden), device="cuda", dtype=dt) for k in ("h1", "r1", "h2", "r2")},
            "q": torch.empty((rows, hq, DIM), device="cuda", dtype=dt),
            "att": torch.empty((rows, hq, DIM), device="cuda", dtype=dt),
            "act": torch.empty((rows, inner), device="cuda", dtype=dt)})
    st["plan"] = feattn.Plan(hq, hkv, DIM, b.page, b.batch, b.max_pages(), st["bf16"], b.blocks)
    st["plan"].prepare(*st["meta"], b.batch, rows, graph=True)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        _layers(st)
    torch.cuda.current_stream().wait_stream(side)
    st["graph"] = torch.cuda.CUDAGraph()
    with torch.cuda.graph(st["graph"]):
        _layers(st)


def _layers(st):
    b, bf16 = st["batch"], st["bf16"]
    hidden, inner = st["case"]["hidden"], st["case"]["inner"]
    for l in st["layers"]:
        feattn.norm(l["x"], l["w1"], l["h1"], b.rows, hidden, EPS, bf16, residual=l["res"], new_residual=l["r1"])
        feattn.norm_rope_append(l["qkv"], l["qkv"].shape[1], l["qw"], l["kw"], EPS, l["q"], l["kc"], l["vc"],
                                st["pos"], st["slots"], st["table"], b.rows, b.hq, b.hkv, bf16, 8192, b.cache_slots)
        st["plan"].run(l["q"], l["kc"], l["vc"], l["att"], causal=True)
        feattn.norm(l["y"], l["w2"], l["h2"], b.rows, hidden, EPS, bf16, residual=l["r1"], new_residual=l["r2"])
        feattn.silu_mul(l["gu"], l["act"], b.rows, inner, bf16)


_STEP_OUT = ("h1", "r1", "q", "kc", "vc", "att", "h2", "r2", "act")


def run(st):
    c = st["case"]
    kind, bf16 = c["kind"], st["bf16"]
    if kind == "attention":
        st["plan"].run(st["q"], st["kc"], st["vc"], st["out"], causal=c["causal"], lse=st["lse"])
        return [st["out"]] if st["lse"] is None else [st["out"], st["lse"]]
    if kind == "norm":
        feattn.norm(st["x"], st["w"], st["out"], c["rows"], c["width"], EPS, bf16, residual=st["res"],
                    new_residual=st["new_res"])
        return [st["out"]] if st["res"] is None else [st["out"], st["new_res"]]
    if kind == "append":
        feattn.norm_rope_append(st["qkv"], st["qkv"].shape[1], st["qw"], st["kw"], EPS, st["q"], st["kc"], st["vc"],
                                st["pos"], st["slots"], st["table"], c["rows"], c["hq"], c["hkv"], bf16, 8192,
                                st["cache_slots"])
        return [st["q"], st["kc"], st["vc"]]
    if kind == "silu":
        feattn.silu_mul(st["gu"], st["out"], c["rows"], c["width"], bf16)
        return [st["out"]]
    b = st["batch"]
    st["plan"].prepare(*st["meta"], b.batch, b.rows, graph=True)
    st["graph"].replay()
    return [[l[k] for k in _STEP_OUT] for l in st["layers"]]


# ---------------------------------------------------------------------------
# What a pass cannot do without, and how far results may be apart
# ---------------------------------------------------------------------------

def _attention_work(case):
    starts, rows = _lens(case)
    pairs = sum(n * s + (n * (n + 1) // 2 if case.get("causal", True) else n * n) for s, n in zip(starts, rows))
    new = sum(rows)
    nbytes = sum(s + n for s, n in zip(starts, rows)) * W.kv_bytes_per_token(case["hkv"])
    nbytes += 2 * new * case["hq"] * DIM * 2 + 4 * sum(math.ceil((s + n) / 16) for s, n in zip(starts, rows))
    if case.get("lse"):
        nbytes += 4 * new * case["hq"]
    return nbytes, 4 * case["hq"] * DIM * pairs


def _norm_work(rows, width, residual):
    return 2 * (rows * width * (4 if residual else 2) + width), 4 * rows * width


def _append_work(rows, hq, hkv):
    heads = hq + 2 * hkv
    return rows * (2 * heads * DIM * 2 + 16 + 4 * DIM), 10 * rows * (hq + hkv) * DIM


def work(case):
    kind = case["kind"]
    if kind == "attention":
        parts = [_attention_work(case)]
    elif kind == "norm":
        parts = [_norm_work(case["rows"], case["width"], case["residual"])]
    elif kind == "append":
        parts = [_append_work(case["rows"], case["hq"], case["hkv"])]
    elif kind == "silu":
        parts = [(6 * case["rows"] * case["width"], 4 * case["rows"] * case["width"])]
    else:
        n = case["seqs"]
        parts = [_norm_work(n, case["hidden"], True)] * 2 + [_append_work(n, case["hq"], case["hkv"]),
                                                             _attention_work(case),
                                                             (6 * n * case["inner"], 4 * n * case["inner"])]
        parts = parts * case["layers"]
    return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}


def tolerance(case):
    if case["kind"] in ("norm", "append"):
        return "exact"  # the order of every sum and rounding is part of their contract
    # 16-bit probabilities, split partials and outputs: each rounds by up to
    # 2^-9 (bfloat16) or 2^-12 (float16) of the value.
    return {"rel": 1e-2 if case["dtype"] == "bf16" else 2e-3}


# ---------------------------------------------------------------------------
# The same results in 64 bits, from torch alone
# ---------------------------------------------------------------------------

def _rms64(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _rope64(x, pos, table):
    t = table.double()[pos][:, None]
    c, s = t[..., :DIM // 2], t[..., DIM // 2:]
    a, b = x[..., :DIM // 2], x[..., DIM // 2:]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _attention64(b, q, kc, vc, causal):
    out = torch.empty(q.shape, device=q.device, dtype=torch.float64)
    lse = torch.empty(q.shape[:2], device=q.device, dtype=torch.float64)
    group = b.hq // b.hkv
    flat_k, flat_v = kc.reshape(-1, b.hkv, DIM), vc.reshape(-1, b.hkv, DIM)
    for i in range(b.batch):
        n, rows = b.lens[i], b.qlens[i]
        pages = torch.tensor(b.pages[b.kv[i]:b.kv[i + 1]], device=q.device)
        at = (pages[:, None] * b.page + torch.arange(b.page, device=q.device)[None]).reshape(-1)[:n]
        k = flat_k[at].double().permute(1, 2, 0).contiguous()
        v = flat_v[at].double().permute(1, 0, 2).contiguous()
        step = max(1, min(rows, (1 << 28) // (n * b.hq)))
        for r0 in range(0, rows, step):
            r1 = min(rows, r0 + step)
            lo = b.qo[i] + r0
            x = q[lo:lo + r1 - r0].double().view(r1 - r0, b.hkv, group, DIM).permute(1, 0, 2, 3)
            s = torch.matmul(x.reshape(b.hkv, -1, DIM), k).div_(math.sqrt(DIM))
            if causal:
                last = (n - rows + torch.arange(r0, r1, device=q.device)).repeat_interleave(group)
                s.masked_fill_((torch.arange(n, device=q.device)[None] > last[:, None])[None], -math.inf)
            l = torch.logsumexp(s, -1)
            o = torch.matmul(s.sub_(l[..., None]).exp_(), v)
            out[lo:lo + r1 - r0] = o.view(b.hkv, r1 - r0, group, DIM).permute(1, 0, 2, 3).reshape(r1 - r0, b.hq, DIM)
            lse[lo:lo + r1 - r0] = l.view(b.hkv, r1 - r0, group).permute(1, 0, 2).reshape(r1 - r0, b.hq)
    return out, lse


def _append64(qkv, qw, kw, kc, vc, pos, slots, table, hq, hkv):
    h = qkv.double().view(qkv.shape[0], hq + 2 * hkv, DIM)
    kc, vc = kc.double(), vc.double()
    kc.view(-1, hkv, DIM)[slots] = _rope64(_rms64(h[:, hq:hq + hkv], kw), pos, table)
    vc.view(-1, hkv, DIM)[slots] = h[:, hq + hkv:]
    return _rope64(_rms64(h[:, :hq], qw), pos, table), kc, vc


def _silu64(gu):
    g, u = gu.double().chunk(2, -1)
    return g * torch.sigmoid(g) * u


def exact(case, seed):
    st = prepare(case, seed)
    kind = case["kind"]
    if kind == "attention":
        out, lse = _attention64(st["batch"], st["q"], st["kc"], st["vc"], case["causal"])
        return [out, lse] if case["lse"] else [out]
    if kind == "norm":
        v = st["x"].double() if st["res"] is None else st["x"].double() + st["res"].double()
        return [_rms64(v, st["w"])] if st["res"] is None else [_rms64(v, st["w"]), v]
    if kind == "append":
        return list(_append64(st["qkv"], st["qw"], st["kw"], st["kc"], st["vc"], st["pos"], st["slots"], st["table"],
                              case["hq"], case["hkv"]))
    if kind == "silu":
        return [_silu64(st["gu"])]
    b, res = st["batch"], []
    for l in st["layers"]:
        r1 = l["x"].double() + l["res"].double()
        q, kc, vc = _append64(l["qkv"], l["qw"], l["kw"], l["kc"], l["vc"], st["pos"], st["slots"], st["table"], b.hq,
                              b.hkv)
        r2 = l["y"].double() + r1
        res.append([_rms64(r1, l["w1"]), r1, q, kc, vc, _attention64(b, q, kc, vc, True)[0], _rms64(r2, l["w2"]), r2,
                    _silu64(l["gu"])])
    return res
