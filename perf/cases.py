"""Performance cases of the framework: the work that a decode loop has it do.

A case is a dict of plain values.  Its ``kind`` says which public entry points one pass goes
through:

  step       ``step.speculative_step`` over ``layers`` attention layers, one query token each:
             block selection, prediction states and strict repair of one decode token
  batch      one call of ``paged.speculative_step`` / ``speculative_signed_step`` / ``exact``
             over a ragged batch of requests in one page pool
  compose    the same step from the single entry points (select, speculate, repair), with one
             of the repair strategies, over ``layers`` layers
  small      selection shared by every head over blocks of 4 or 8 tokens: indexer, hierarchical
             partials, hierarchical repair (or the hierarchical exact attention)
  bounds     block metadata of a prefilled cache (``bounds.block_bounds``)

Decode loops on this device replay captured graphs, so ``graph`` cases capture their layers
once, when the inputs are made, and a pass is one replay; the others call the entry points
directly.  The host-backed cache is left out: the host link sets its time.

Inputs follow the framework's benchmark configurations: normal queries, keys and values, 5 %
of every KV head's blocks shifted towards its group's mean query, predictions that agree with
the selection at ``overlap``.
"""
import math
import sys
from pathlib import Path

import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "strict-topk-overlap_amd"))

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
DEV = "cuda"


def _case(kind, hq, hkv, d, b, n, k, **more):
    c = dict(kind=kind, hq=hq, hkv=hkv, d=d, b=b, n=n, k=k, sp=k, overlap=0.9, dtype="bf16",
             bounds="keys", layers=1, graph=False)
    c.update(more)
    return c


def listed():
    cs = {
        # one tiny layer called directly: all launch and host latency
        "small_step": _case("step", 4, 4, 64, 32, 64, 8, overlap=0.75, dtype="fp16"),
        # one token through the layers of a small model at 16K context
        "layers_16k": _case("step", 16, 8, 128, 32, 512, 64, layers=12, graph=True),
        # the headline step: 64K context, 32 query heads over 8 KV heads
        "layers_64k": _case("step", 32, 8, 128, 32, 2048, 64, layers=12, graph=True),
        # a long context and eight query heads per KV head, as larger models have
        "layers_250k": _case("step", 64, 8, 128, 32, 7999, 96, sp=100, overlap=0.8,
                             dtype="fp16", layers=4, graph=True),
        # a serving batch of ragged requests, strict speculative step
        "batch_saved": _case("batch", 32, 8, 128, 32, 2048, 64, requests=24, min_blocks=40,
                             op="saved", eps=0.0),
        # the ragged signed batch: 8K to 128K tokens, low-mass wrong blocks may stay
        "batch_signed": _case("batch", 32, 8, 128, 32, 4096, 64, requests=16, min_blocks=256,
                              overlap=0.75, op="hybrid", eps=0.01),
        # the same kind of batch without a prediction (exact sparse attention)
        "batch_exact": _case("batch", 16, 8, 128, 32, 1501, 48, requests=31, min_blocks=100,
                             op="exact", eps=0.0),
        # the drop-in composition: float32 bounds, separate calls, one miss list per head
        "compose_saved": _case("compose", 32, 8, 128, 32, 1500, 64, bounds="fp32", layers=8,
                               graph=True, mode="saved", repair="gqa_saved", tau=0.0, eps=0.0,
                               ids=32),
        # expanded KV heads, compact prediction, the split repair
        "compose_split": _case("compose", 32, 32, 128, 32, 1024, 64, overlap=0.8, dtype="fp16",
                               bounds="fp32", layers=4, graph=True, mode="compact",
                               repair="split", tau=0.03, eps=0.0, ids=64),
        # one request's hybrid prediction and the one-kernel repair
        "compose_fused": _case("compose", 16, 8, 128, 32, 777, 48, overlap=0.75, bounds="fp32",
                               layers=8, graph=True, mode="hybrid", repair="fused", tau=0.05,
                               eps=0.01, ids=32),
        # 4-token blocks, 12 query heads per KV head, one selection for all heads
        "small_blocks": _case("small", 48, 4, 128, 4, 8192, 2048, overlap=0.8, layers=2,
                              graph=True, op="repair", ihq=4),
        # block metadata after a prefill of 250K tokens
        "bounds_250k": _case("bounds", 8, 8, 128, 32, 7813, 64),
    }
    return [dict(c, name=name) for name, c in cs.items()]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ones' ranges, at most as large as the largest of them."""
    c = _draw(rng)
    most = 0.95 * max(work(x)["bytes"] for x in listed())
    while work(c)["bytes"] > most:
        size = next(x for x in ("layers", "requests", "n") if c.get(x, 1) > 1)
        c[size] -= -(-c[size] // 8)
    return c


def _draw(rng):
    kind = rng.choice(["step", "step", "step", "batch", "batch", "batch", "compose", "compose",
                       "compose", "small", "bounds"])
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    d = rng.choice([64, 128, 128, 128, 256])
    overlap = round(rng.uniform(0.5, 1.0), 3)
    heads = rng.choice([(4, 4), (8, 8), (16, 8), (32, 8), (40, 8), (64, 8), (16, 2), (24, 4),
                        (48, 16)])
    if kind == "small":
        hq, hkv = rng.choice([(48, 4), (24, 2), (32, 4), (16, 4), (64, 8)])
        n = _log(rng, 1024, 8192)
        return _case("small", hq, hkv, rng.choice([64, 128, 128]), rng.choice([4, 4, 8]), n,
                     rng.randint(n // 8, n // 4), overlap=overlap, dtype=dtype, layers=2,
                     graph=True, op=rng.choice(["repair", "repair", "exact"]),
                     ihq=rng.choice([2, 4, 8]))
    if kind == "bounds":
        return _case("bounds", heads[1], heads[1], d, rng.choice([16, 32, 64]),
                     _log(rng, 256, 65536 // heads[1] * 128 // d), 64, dtype=dtype,
                     bounds=rng.choice(["keys", "fp32"]))
    if kind == "compose":
        hq, hkv = rng.choice([(4, 4), (16, 16), (32, 32), (16, 8), (32, 8), (64, 8)])
        n = _log(rng, 64, 2048)
        k = rng.randint(8, min(96, n // 2))
        mode, repair = rng.choice([("saved", "gqa_saved"), ("saved", "gqa_union"),
                                   ("saved", "light"), ("saved", "split"), ("saved", "fused"),
                                   ("hybrid", "split"), ("hybrid", "fused"),
                                   ("hybrid", "signed"), ("hybrid", "signed_fused"),
                                   ("compact", "split"), ("compact", "fused"),
                                   ("compact", "signed_fused")])
        eps = rng.choice([0.0, 0.01]) if repair in ("fused", "signed", "signed_fused") and \
            mode != "saved" else 0.0
        return _case("compose", hq, hkv, rng.choice([64, 128, 128, 128]), 32, n, k,
                     overlap=overlap, dtype=dtype, bounds="fp32", layers=rng.choice([1, 2, 4]),
                     graph=True, mode=mode, repair=repair,
                     tau=round(rng.uniform(0.02, 0.2), 3) if mode != "saved" else 0.0, eps=eps,
                     ids=rng.choice([32, 32, 64]))
    hq, hkv = heads
    if kind == "batch":
        op = rng.choice(["saved", "saved", "union", "hybrid", "exact"])
        requests = _log(rng, 2, 32)
        n = _log(rng, 128, max(256, min(4096, 49152 * 128 // (requests * hkv * d))))
        return _case("batch", hq, hkv, d, 32, n, rng.randint(16, 64), requests=requests,
                     min_blocks=rng.randint(24, 96), overlap=overlap, dtype=dtype, op=op,
                     bounds=rng.choice(["keys", "keys", "fp32"]),
                     eps=rng.choice([0.0, 0.01]) if op == "hybrid" else 0.0)
    n = _log(rng, 48, 8192)
    k = rng.randint(8, min(128, n // 2))
    layers = max(1, min(12, 16384 * 8 * 128 // (n * hkv * d)))
    return _case("step", hq, hkv, d, rng.choice([16, 32, 32, 32, 64]), n, k,
                 sp=max(4, min(n // 2, 128, k + rng.choice([0, 0, 0, -3, 5]))), overlap=overlap,
                 dtype=dtype, bounds=rng.choice(["keys", "keys", "fp32"]), layers=layers,
                 graph=rng.random() < 0.8)


# ------------------------------------------------------------------ inputs
def _gen(seed, salt=0):
    return torch.Generator(device=DEV).manual_seed(int(seed) * 1009 + salt)


def _randn(gen, shape, dtype):
    return torch.randn(shape, generator=gen, device=DEV, dtype=dtype)


def _hot(k, q, gen, hkv):
    """Shift 5 % of every KV head's blocks of k [Hkv, N, B, D] towards its mean query."""
    qm = q.float().view(hkv, -1, q.shape[-1]).mean(1)
    qhat = (1.5 * qm / qm.norm(dim=-1, keepdim=True)).to(k.dtype)
    n = k.shape[1]
    nhot = max(1, round(0.05 * n))
    for h in range(hkv):
        idx = torch.randperm(n, generator=gen, device=DEV)[:nhot]
        k[h, idx] += qhat[h]


def _scores(q, lo, hi, dtype):
    """Bound scores [Hq, N] of q [Hq, D] on lo, hi [Hkv, N, D] in ``dtype``."""
    hkv = lo.shape[0]
    qg = q.to(dtype).view(hkv, -1, q.shape[-1])
    s = torch.matmul(qg.clamp(min=0), hi.to(dtype).transpose(1, 2).contiguous())
    s += torch.matmul(qg.clamp(max=0), lo.to(dtype).transpose(1, 2).contiguous())
    return s.reshape(q.shape[0], -1)


def _predict(scores, k, sp, overlap, gen):
    """int32 [H, SP]: the top k with a share of 1 - overlap replaced by other blocks, in random
    order; -1 where a row has fewer than SP blocks to name."""
    h, n = scores.shape
    k = min(k, n)
    sel = scores.topk(k, dim=1).indices
    noise = torch.rand((h, n), generator=gen, device=DEV)
    noise.scatter_(1, sel, -1.0)
    replace = min(round((1.0 - overlap) * k), n - k)
    more = min(max(0, sp - k), n - k - replace)
    free = noise.topk(replace + more, dim=1).indices
    mix = torch.rand((h, k), generator=gen, device=DEV).argsort(1)
    row = torch.cat((sel.gather(1, mix)[:, :k - replace], free), 1)
    mix = torch.rand(row.shape, generator=gen, device=DEV).argsort(1)
    row = row.gather(1, mix)[:, :sp]
    out = torch.full((h, sp), -1, dtype=torch.int32, device=DEV)
    out[:, :row.shape[1]] = row.to(torch.int32)
    return out


def _layer(c, seed, layer):
    gen = _gen(seed, 17 * layer + 1)
    dt = DTYPES[c["dtype"]]
    q = _randn(gen, (c["hq"], c["d"]), dt)
    k = _randn(gen, (c["hkv"], c["n"], c["b"], c["d"]), dt)
    v = _randn(gen, k.shape, dt)
    _hot(k, q, gen, c["hkv"])
    lo, hi = k.amin(2), k.amax(2)
    if c["bounds"] == "fp32":
        lo, hi = lo.float(), hi.float()
    p = _predict(_scores(q, lo, hi, torch.float32), c["k"], c["sp"], c["overlap"], gen)
    if c.get("ids") == 64:
        p = p.long()
    return q, k, v, lo, hi, p


def _lengths(c):
    """Blocks per request, spread over [min_blocks, n] on a log scale, none a round number."""
    r, lo, hi = c["requests"], min(c["min_blocks"], c["n"]), c["n"]
    return [max(lo, min(hi, round(lo * (hi / lo) ** (i / max(1, r - 1))))) for i in range(r)]


def _batch(c, seed):
    gen = _gen(seed, 5)
    dt = DTYPES[c["dtype"]]
    hq, hkv, b, d = c["hq"], c["hkv"], c["b"], c["d"]
    counts = _lengths(c)
    mix = torch.randperm(len(counts), generator=gen, device=DEV).tolist()
    counts = [counts[i] for i in mix]
    total = hkv * sum(counts)
    kp = _randn(gen, (total, b, d), dt)
    vp = _randn(gen, (total, b, d), dt)
    q = _randn(gen, (len(counts), hq, d), dt)
    order = torch.randperm(total, generator=gen, device=DEV)
    table = torch.full((len(counts), hkv, c["n"]), -1, dtype=torch.int32, device=DEV)
    part = torch.randint(1, b + 1, (len(counts),), generator=gen, device=DEV)
    base = 0
    for r, n in enumerate(counts):
        pages = order[base:base + hkv * n].view(hkv, n)
        base += hkv * n
        table[r, :, :n] = pages.to(torch.int32)
        qm = q[r].float().view(hkv, -1, d).mean(1)
        qhat = (1.5 * qm / qm.norm(dim=-1, keepdim=True)).to(dt)
        hot = pages[:, torch.randperm(n, generator=gen, device=DEV)[:max(1, round(0.05 * n))]]
        kp[hot.flatten()] += qhat.repeat_interleave(hot.shape[1], 0)[:, None]
    lo, hi = kp.amin(1), kp.amax(1)
    live = torch.arange(b, device=DEV)[None, :, None] < part.repeat_interleave(hkv)[:, None, None]
    last = torch.cat([table[r, :, n - 1] for r, n in enumerate(counts)]).long()
    lo[last] = torch.where(live, kp[last], math.inf).amin(1)
    hi[last] = torch.where(live, kp[last], -math.inf).amax(1)
    if c["bounds"] == "fp32":
        lo, hi = lo.float(), hi.float()
    nb = torch.tensor(counts, dtype=torch.int32, device=DEV)
    nt = ((nb.long() - 1) * b + part).to(torch.int32)
    p = torch.empty((len(counts), hq, c["sp"]), dtype=torch.int32, device=DEV)
    for r, n in enumerate(counts):
        pages = table[r, :, :n].long()
        p[r] = _predict(_scores(q[r], lo[pages], hi[pages], torch.float32), c["k"], c["sp"],
                        c["overlap"], gen)
    return q, kp, vp, lo, hi, table, nb, nt, p, counts


def _small(c, seed, layer):
    gen = _gen(seed, 31 * layer + 3)
    dt = DTYPES[c["dtype"]]
    q = _randn(gen, (c["hq"], c["d"]), dt)
    k = _randn(gen, (c["hkv"], c["n"], c["b"], c["d"]), dt)
    v = _randn(gen, k.shape, dt)
    iq = _randn(gen, (c["ihq"], 128), dt)
    ik = _randn(gen, (c["n"], 128), dt)
    s = torch.matmul(iq.float(), ik.float().t()).clamp(min=0).sum(0, keepdim=True)
    p = _predict(s, c["k"], c["sp"], c["overlap"], gen).expand(c["hq"], -1).contiguous()
    return q, k, v, iq, ik, p


def _captured(fn):
    fn()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = fn()
    return graph, out


def prepare(case, seed):
    c = case
    if c["kind"] == "batch":
        from strict_topk.paged import PagedKV
        q, kp, vp, lo, hi, table, nb, nt, p, _ = _batch(c, seed)
        state = dict(case=c, q=q, p=p, kv=PagedKV(kp, vp, lo, hi, table, nb, nt))
    elif c["kind"] == "bounds":
        gen = _gen(seed, 9)
        state = dict(case=c, k=_randn(gen, (c["hkv"], c["n"], c["b"], c["d"]),
                                      DTYPES[c["dtype"]]))
    else:
        make = _small if c["kind"] == "small" else _layer
        state = dict(case=c, layers=[make(c, seed, i) for i in range(c["layers"])])
    if c["graph"]:
        state["graph"], state["out"] = _captured(lambda: _pass(state))
    return state


# ------------------------------------------------------------------ one pass
def _state(s):
    return [s.m, s.l, s.u]


def _result(r):
    return [x for x in (r.output, r.fallback, r.remaining, r.approximate_heads) if x is not None]


def _compose(c, q, k, v, lo, hi, p):
    from strict_topk import fused, gqa, gqa_light, kernels, selector, signed_fused, signed_repair
    if c["hq"] == c["hkv"]:
        sel = selector.select_blocks(q, lo, hi, c["k"])
    else:
        sel = gqa.select_blocks(q, lo, hi, c["k"])
    name = c["repair"]
    if name in ("gqa_saved", "gqa_union", "light"):
        st = gqa.partials(q, k, v, p)
        fn = {"gqa_saved": gqa.repair_saved, "gqa_union": gqa.repair_union,
              "light": gqa_light.repair_saved_light}[name]
        return [sel, fn(q, k, v, sel, p, st)] + _state(st)
    pred = kernels.speculate(q, k, v, p, c["mode"], c["tau"], keep_mass=True)
    if name == "split":
        res = kernels.repair(q, k, v, sel, p, pred)
    else:
        fn = {"fused": fused.repair_fused, "signed": signed_repair.repair_signed,
              "signed_fused": signed_fused.repair_signed_fused}[name]
        res = fn(q, k, v, sel, p, pred, max_extra_mass=c["eps"])
    return [sel] + _result(res) + _state(pred.state)


def _pass(state):
    c = state["case"]
    kind = c["kind"]
    if kind == "step":
        from strict_topk import step
        outs = []
        for q, k, v, lo, hi, p in state["layers"]:
            r = step.speculative_step(q, k, v, lo, hi, p, c["k"])
            outs.append([r.selected, r.output] + _state(r.state))
        return outs
    if kind == "compose":
        return [_compose(c, *layer) for layer in state["layers"]]
    if kind == "small":
        from strict_topk import gqa_hierarchical, indexer
        outs = []
        for q, k, v, iq, ik, p in state["layers"]:
            sel = indexer.select_shared(iq, ik, c["k"], c["hq"])
            if c["op"] == "exact":
                outs.append([sel, gqa_hierarchical.exact(q, k, v, sel)])
            else:
                st = gqa_hierarchical.partials(q, k, v, p)
                out = gqa_hierarchical.repair_saved_shared(q, k, v, sel, p, st)
                outs.append([sel, out] + _state(st))
        return outs
    if kind == "bounds":
        from strict_topk import bounds
        k = state["k"]
        return list(bounds.block_bounds(k, torch.float32 if c["bounds"] == "fp32" else k.dtype))
    from strict_topk import paged
    q, kv, p = state["q"], state["kv"], state["p"]
    if c["op"] == "exact":
        return list(paged.exact(q, kv, c["k"]))
    if c["op"] == "hybrid":
        r = paged.speculative_signed_step(q, kv, p, c["k"], "hybrid", 0.2,
                                          max_extra_mass=c["eps"])
        return [r.selected] + _result(r.result) + _state(r.state)
    r = paged.speculative_step(q, kv, p, c["k"], union=c["op"] == "union")
    return [r.selected, r.output] + _state(r.state)


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    return _pass(state)


# ------------------------------------------------------------------ work and tolerance
def _unique(n, k, g):
    """Blocks that g query heads of one KV head name between them, k each: the picks fall on
    about a fifth of the blocks (the hot ones, then those with the widest bounds)."""
    k = min(n, k)
    pool = min(n, 0.2 * n + k)
    return min(n, pool * (1.0 - (1.0 - k / pool) ** g))


def work(case):
    c = case
    hq, hkv, d, b, n, k, sp = (c[x] for x in ("hq", "hkv", "d", "b", "n", "k", "sp"))
    g = hq // hkv
    tile = 2 * b * d * 2
    eb = 4 if c["bounds"] == "fp32" else 2
    if c["kind"] == "bounds":
        size = hkv * n * d
        return {"bytes": size * b * 2 + 2 * size * eb, "flops": 2 * size * b}
    if c["kind"] == "small":
        sel = hkv * k * tile + n * 128 * 2 + hq * k * 4
        flops = 2 * c["ihq"] * n * 128 + 4 * hq * k * b * d
        if c["op"] == "exact":
            return {"bytes": c["layers"] * (sel + hq * d * 6), "flops": c["layers"] * flops}
        miss = (1.0 - c["overlap"]) * k
        spec = hkv * (sp + miss) * tile + n * 128 * 2 + hq * (k + sp) * 4
        spec += hq * (sp + (k - miss)) * (d + 2) * 4
        return {"bytes": c["layers"] * (spec + hq * d * 6),
                "flops": c["layers"] * (2 * c["ihq"] * n * 128 + 4 * hq * (sp + miss) * b * d)}

    def one(n):
        kk, ss = min(k, n), min(sp, n)
        miss = min((1.0 - c["overlap"]) * kk, n - kk)
        byt = 2 * hkv * n * d * eb + hq * d * 6 + hq * (k + sp) * 4
        flops = 2 * hq * n * d
        if c.get("op") == "exact":
            return byt + hkv * _unique(n, kk, g) * tile, flops + 4 * hq * kk * b * d
        tiles = _unique(n, ss, g) + min(g * miss, n)
        byt += hkv * min(tiles, 2 * n) * tile + hq * sp * (d + 2) * 4 + hq * (kk - miss) * (d + 2) * 4
        return byt, flops + 4 * hq * (ss + miss) * b * d

    if c["kind"] == "batch":
        parts = [one(n) for n in _lengths(c)]
    else:
        parts = [one(n)] * c["layers"]
    return {"bytes": sum(x for x, _ in parts), "flops": sum(x for _, x in parts)}


def tolerance(case):
    if case["kind"] == "bounds":
        return "exact"
    # 32-bit states and sums over 16-bit inputs, 3e-6 off the 64-bit values at most; IDs and
    # flags are whole numbers and agree
    return {"rel": 1e-5, "max": 1e-4}


# ------------------------------------------------------------------ exact values
def _states64(q, kt, vt, live=None):
    """m, l [H, S], u [H, S, D] of q [H, D] on gathered tiles kt, vt [H, S, B, D]; ``live``
    [H, S, B]: tokens that hold data."""
    q, d = q.double(), q.shape[-1]
    m, l, u = [], [], []
    for h in range(q.shape[0]):
        s = (kt[h].double() * q[h]).sum(-1) / math.sqrt(d)
        if live is not None:
            s = s.masked_fill(~live[h], -math.inf)
        mh = s.amax(-1)
        w = torch.where(s == -math.inf, 0.0, torch.exp(s - mh[:, None].clamp(min=-1e300)))
        vv = vt[h].double()
        if live is not None:
            vv = torch.where(live[h][:, :, None], vv, 0.0)
        m.append(mh)
        l.append(w.sum(-1))
        u.append((w[:, :, None] * vv).sum(1))
    return torch.stack(m), torch.stack(l), torch.stack(u)


def _merge64(m, l, u):
    top = m.amax(1, keepdim=True)
    a = torch.exp(m - top)
    return (a[:, :, None] * u).sum(1) / (a * l).sum(1)[:, None]


def _select64(scores, k):
    kk = min(k, scores.shape[1])
    ids = scores.topk(kk, dim=1).indices.sort(1).values.to(torch.int32)
    out = torch.full((scores.shape[0], k), -1, dtype=torch.int32, device=DEV)
    out[:, :kk] = ids
    return out


def _hit(p, sel):
    return ((p[:, :, None] == sel[:, None, :]) & (p[:, :, None] >= 0)).any(2)


def _signed64(c, tau, states_p, states_a, sel, p, first):
    """output, fallback (no value), remaining, extra-mass decisions of a hybrid or compact
    prediction: the strict attention over the selected blocks, or with the wrong low blocks
    kept where their share of the mass is at most eps."""
    m, l, _ = states_p
    mass = torch.exp(m - m.amax(1, keepdim=True)) * l
    high = mass >= tau * mass.sum(1, keepdim=True)
    hit = _hit(p, sel)
    low_hit = (hit & ~high).any(1)
    low = (mass * ~high).sum(1)
    wrong = (mass * (~hit & ~high & (p >= 0))).sum(1)
    some = (~hit & ~high & (p >= 0)).any(1) & low_hit
    share = wrong / (low + (mass * (hit & high)).sum(1)).clamp(min=1e-300)
    skip = some & (share <= c["eps"]) if c["eps"] > 0 else torch.zeros_like(some)
    keep = skip[:, None] & ~hit & ~high & (p >= 0)
    am, al, au = states_a
    pm, pl, pu = states_p
    out = _merge64(torch.cat((am, torch.where(keep, pm, -math.inf)), 1), torch.cat((al, pl), 1),
                   torch.cat((au, pu), 1))
    rem = torch.where(low_hit & ~skip, (low - wrong) / low.clamp(min=1e-300), 1.0)
    return first + [out, None, rem] + ([None] if c["eps"] > 0 else []), high


def _attend(q, k, v, ids, g, tokens=None):
    """States of every listed block, k, v [Hkv, N, B, D]; -1 gives the empty state."""
    kvh = torch.arange(q.shape[0], device=DEV) // g
    safe = ids.long().clamp(min=0)
    live = None
    if tokens is not None or bool((ids < 0).any()):
        pos = safe[:, :, None] * k.shape[2] + torch.arange(k.shape[2], device=DEV)
        live = (ids >= 0)[:, :, None] & (pos < (1 << 62 if tokens is None else tokens))
    ms, ls, us = [], [], []
    for h in range(q.shape[0]):
        m, l, u = _states64(q[h:h + 1], k[kvh[h], safe[h]][None], v[kvh[h], safe[h]][None],
                            None if live is None else live[h:h + 1])
        ms.append(m)
        ls.append(l)
        us.append(u)
    return torch.cat(ms), torch.cat(ls), torch.cat(us)


def _exact_layer(c, q, k, v, lo, hi, p, tokens=None):
    """The outputs of one step on dense blocks, as ``_pass`` lays them out."""
    g = c["hq"] // c["hkv"]
    sel = _select64(_scores(q, lo, hi, torch.float64), c["k"])
    sa = _attend(q, k, v, sel, g, tokens)
    if c.get("op") == "exact":
        return [sel, _merge64(*sa)]
    sp = _attend(q, k, v, p, g, tokens)
    how = c.get("op") or c.get("repair") or "saved"
    if how in ("saved", "gqa_saved", "light", "union", "gqa_union"):
        if how in ("union", "gqa_union"):
            wrong = ~_hit(p, sel)
            out = _merge64(torch.cat((sa[0], torch.where(wrong, sp[0], -math.inf)), 1),
                           torch.cat((sa[1], sp[1]), 1), torch.cat((sa[2], sp[2]), 1))
        else:
            out = _merge64(*sa)
        return [sel, out] + list(sp)
    mode = c.get("mode", "hybrid")
    if mode == "saved":
        ones = torch.ones(c["hq"], dtype=torch.float64, device=DEV)
        return [sel, _merge64(*sa), None, ones] + ([None] if c["eps"] > 0 else []) + list(sp)
    got, high = _signed64(c, c.get("tau", 0.2), sp, sa, sel, p, [sel])
    if mode == "compact":
        s = c["sp"]
        cap = s if c["tau"] <= 1 / s else min(s, int(1 / c["tau"]) + 1)
        at = torch.where(high, torch.arange(s, device=DEV), s).sort(1).values[:, :cap]
        on = at < s
        at = at.clamp(max=s - 1)
        sp = (torch.where(on, sp[0].gather(1, at), -math.inf),
              torch.where(on, sp[1].gather(1, at), 0.0),
              torch.where(on[:, :, None],
                          sp[2].gather(1, at[:, :, None].expand(-1, -1, c["d"])), 0.0))
    return got + list(sp)


def exact(case, seed):
    c = case
    if c["kind"] == "bounds":
        k = prepare(dict(c, graph=False), seed)["k"]
        return [k.amin(2).double(), k.amax(2).double()]
    if c["kind"] in ("step", "compose"):
        return [_exact_layer(c, *_layer(c, seed, i)) for i in range(c["layers"])]
    if c["kind"] == "small":
        outs = []
        for i in range(c["layers"]):
            q, k, v, iq, ik, p = _small(c, seed, i)
            g = c["hq"] // c["hkv"]
            s = torch.matmul(iq.double(), ik.double().t()).clamp(min=0).sum(0, keepdim=True)
            sel = _select64(s, c["k"]).expand(c["hq"], -1)
            out = _merge64(*_attend(q, k, v, sel, g))
            outs.append([sel, out] + (list(_attend(q, k, v, p, g)) if c["op"] == "repair" else []))
        return outs
    q, kp, vp, lo, hi, table, nb, nt, p, counts = _batch(c, seed)
    rows = []
    for r, n in enumerate(counts):
        pages = table[r, :, :n].long()
        rows.append(_exact_layer(c, q[r], kp[pages], vp[pages], lo[pages], hi[pages], p[r],
                                 int(nt[r])))
    return [None if col[0] is None else torch.stack(col) for col in zip(*rows)]
