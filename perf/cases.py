"""Timed cases of the quotient-filter library: what its users' programs call
it for, through the Python binding, from the smallest calls to the largest
tables.

A case is a dict of plain values.  kind:
  build    one bulk build of a table from `fill` * 2^q keys (the NoDup rule
           drops repeated fingerprints);
  lookup   one membership call of n keys, half of them stored (answers:
           slots);
  count    one counting query of n keys (RSQF);
  window   one step of a sliding window over a resident filter: the oldest n
           keys are deleted, n new ones inserted (the fill stays where it is);
  batch    many small SQFs built by one call and probed by another;
  serve    a backlog of lookup / insert / delete requests over resident
           RSQFs through the serving loop (every inserted batch is deleted
           again, so the loop ends in the state it began with).

Keys are uniform random 32-bit words, as the hashes meet them.  Mutating
passes return the whole table (its device bytes) beside their answers.
"""
import random

import torch

import gpuquotientfilters_amd as G

DEV = "cuda"


def listed():
    return [
        # a membership check of one request's keys: launch latency
        {"name": "sqf_lookup_small", "kind": "lookup", "filter": "sqf", "q": 20, "r": 5, "fill": 0.75, "n": 1000},
        # the headline table probed by a large batch
        {"name": "sqf_lookup_large", "kind": "lookup", "filter": "sqf", "q": 26, "r": 5, "fill": 0.8, "n": 1 << 24},
        # one small filter of many (one per sorted run of a store), 2-byte slots
        {"name": "sqf_build_small", "kind": "build", "filter": "sqf", "q": 17, "r": 13, "fill": 0.75, "nodup": False},
        # the headline bulk build
        {"name": "sqf_build_large", "kind": "build", "filter": "sqf", "q": 26, "r": 5, "fill": 0.8, "nodup": True},
        # deduplication of a stream by small steps
        {"name": "sqf_window_small", "kind": "window", "filter": "sqf", "q": 24, "r": 5, "fill": 0.7, "n": 10007},
        # the same by large steps on the headline table
        {"name": "sqf_window_large", "kind": "window", "filter": "sqf", "q": 26, "r": 5, "fill": 0.75, "n": 1 << 20},
        # packed slot widths
        {"name": "sqf_window_packed", "kind": "window", "filter": "sqf", "q": 22, "r": 9, "fill": 0.7, "n": 50021},
        # the RSQF's headline bulk build (wide fingerprints)
        {"name": "rsqf_build_large", "kind": "build", "filter": "rsqf", "q": 26, "r": 8, "fill": 0.9, "nodup": False},
        # the same table probed by a large batch
        {"name": "rsqf_lookup_large", "kind": "lookup", "filter": "rsqf", "q": 26, "r": 8, "fill": 0.9, "n": 1 << 24},
        # the RSQF's incremental step
        {"name": "rsqf_window_large", "kind": "window", "filter": "rsqf", "q": 26, "r": 8, "fill": 0.8, "n": 1 << 18},
        # resident filters behind a request queue
        {"name": "rsqf_serve", "kind": "serve", "filters": 4, "qlo": 21, "qhi": 24, "r": 8, "fill": 0.5, "requests": 300,
         "nmax": 1 << 17},
        # one call for many small filters
        {"name": "sqf_batch", "kind": "batch", "filters": 48, "qlo": 12, "qhi": 20, "r": 5, "nodup": False},
    ]


def _logint(rng, lo, hi):
    """An integer spread over the logarithm of [lo, hi], usually odd."""
    v = int(round(lo * (hi / lo) ** rng.random()))
    return max(lo, min(hi, v if rng.random() < 0.2 else v | 1))


def draw(rng):
    kind = rng.choices(("build", "lookup", "window", "count", "batch", "serve"), (5, 5, 8, 1, 1, 1))[0]
    if kind == "batch":
        lo = rng.randint(10, 14)
        return {"kind": "batch", "filters": rng.randint(8, 48), "qlo": lo, "qhi": rng.randint(lo + 2, 20),
                "r": 5, "nodup": rng.random() < 0.5}
    if kind == "serve":
        lo = rng.randint(18, 22)
        return {"kind": "serve", "filters": rng.randint(2, 6), "qlo": lo, "qhi": rng.randint(lo + 1, 24), "r": 8,
                "fill": round(rng.uniform(0.4, 0.7), 3), "requests": rng.randint(60, 300),
                "nmax": 1 << rng.randint(12, 17)}
    f = "rsqf" if kind == "count" else rng.choice(("sqf", "rsqf"))
    if f == "sqf":
        r = rng.choice((5, 5, 5, 5, 13, 9, 7))
        q = rng.randint(12, min(26 if r == 5 else 24, 32 - r))
        fill = round(rng.uniform(0.3, 0.8), 3)
    else:
        r = rng.choice((8, 8, 8, 5, 13))
        q = rng.randint(14, 26 if r == 8 else 25)
        fill = round(rng.uniform(0.4, 0.85), 3)
    c = {"kind": kind, "filter": f, "q": q, "r": r, "fill": fill}
    if kind == "build":
        c["nodup"] = f == "sqf" and rng.random() < 0.5
    elif kind == "window":
        c["n"] = _logint(rng, 64, min(1 << 20, (1 << q) // 32))
    else:
        c["n"] = _logint(rng, 64, 1 << (24 if kind == "lookup" else 22))
    return c


class _Bytes:
    """Device bytes of `owner` as torch.as_tensor takes them (no copy)."""

    def __init__(self, owner, ptr, n):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (int(n),), "typestr": "|u1", "data": (int(ptr), False), "version": 2}


def _table(f):
    if isinstance(f, G.RSQF):
        p, n = f.h.blocks, G.lib().gqf_rsqf_table_bytes(f.q, f.r)
    else:
        p, n = f.h.table, G.lib().gqf_sqf_table_bytes(f.q, f.r)
    t = torch.as_tensor(_Bytes(f, p, n), device=DEV)
    t.owner = f  # the filter frees its table: it lives as long as the tensor
    return t


def _keys(gen, n):
    return torch.randint(-(1 << 31), 1 << 31, (n,), dtype=torch.int32, device=DEV, generator=gen)


def _probe(gen, stored, n):
    """n keys, about half of them stored."""
    pick = stored[torch.randint(0, len(stored), (n,), device=DEV, generator=gen)]
    return torch.where(torch.rand(n, device=DEV, generator=gen) < 0.5, pick, _keys(gen, n))


def _new(case, q):
    return (G.RSQF if case["filter"] == "rsqf" else G.SQF)(q, case["r"])


def _count(fill, q):
    return int(fill * (1 << q))


def prepare(case, seed):
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed)
    kind = case["kind"]
    if kind == "batch":
        return _prepare_batch(case, gen)
    if kind == "serve":
        return _prepare_serve(case, gen, seed)
    q, n = case["q"], _count(case["fill"], case["q"])
    f = _new(case, q)
    s = {"kind": kind, "f": f, "table": _table(f), "nodup": case.get("nodup", False), "rsqf": case["filter"] == "rsqf"}
    keys = _keys(gen, n)
    if kind == "build":
        s["keys"] = keys
        return s
    f.bulk_build(keys)
    m = case["n"]
    if kind == "window":
        s["old"], s["new"] = keys[:m].clone(), _keys(gen, m)
    else:
        s["probe"] = _probe(gen, keys, m)
        s["out"] = torch.empty(m, dtype=torch.int32, device=DEV)
    torch.cuda.synchronize()
    return s


def _prepare_batch(case, gen):
    rng = random.Random(case["filters"] * 1000 + case["qhi"])  # the same shapes for every seed
    qs = [rng.randint(case["qlo"], case["qhi"]) for _ in range(case["filters"])]
    nk = [_count(rng.uniform(0.3, 0.8), q) for q in qs]
    npr = [int(2 ** rng.uniform(8, 16)) for _ in qs]
    koff, poff = [0], [0]
    for a, b in zip(nk, npr):
        koff.append(koff[-1] + a)
        poff.append(poff[-1] + b)
    pool = _keys(gen, 4 * koff[-1])
    keys = pool[torch.randint(0, len(pool), (koff[-1],), device=DEV, generator=gen)]  # some repeat
    probe = torch.empty(poff[-1], dtype=torch.int32, device=DEV)
    for i in range(len(qs)):
        probe[poff[i]:poff[i + 1]] = _probe(gen, keys[koff[i]:koff[i + 1]], npr[i])
    out = torch.empty(poff[-1], dtype=torch.int32, device=DEV)
    fs = [G.SQF(q, case["r"]) for q in qs]
    torch.cuda.synchronize()
    b = G.SQFBatch(fs, keys, koff, probe, poff, out, no_dup=case["nodup"])
    return {"kind": "batch", "batch": b, "filters": fs, "tables": [_table(f) for f in fs], "out": out}


def _prepare_serve(case, gen, seed):
    shape = random.Random(case["requests"] * 1000 + case["qhi"])  # filters, kinds and sizes: the same for every seed
    qs = [shape.randint(case["qlo"], case["qhi"]) for _ in range(case["filters"])]
    fs = []
    stored = []
    for q in qs:
        f = G.RSQF(q, case["r"])
        keys = _keys(gen, _count(case["fill"], q))
        f.bulk_build(keys)
        fs.append(f)
        stored.append(keys)
    plan = []  # (filter, op, n, offset of an insert's keys for its delete)
    open_ = [[] for _ in qs]
    off = 0
    for _ in range(case["requests"]):
        i = shape.randrange(len(qs))
        u = shape.random()
        n = _logint(shape, 64, min(case["nmax"], (1 << qs[i]) // 64))
        if u < 0.7:
            plan.append((i, G.OP_LOOKUP, n, off))
            off += n
        elif u < 0.85 or not open_[i]:
            plan.append((i, G.OP_INSERT, n, off))
            open_[i].append((n, off))
            off += n
        else:
            m, at = open_[i].pop(0)
            plan.append((i, G.OP_DELETE, m, at))
    for i, o in enumerate(open_):
        plan += [(i, G.OP_DELETE, m, at) for m, at in o]
    keys = _keys(gen, off)
    out = torch.zeros(off, dtype=torch.int32, device=DEV)
    for i, op, n, at in plan:
        if op == G.OP_LOOKUP:
            keys[at:at + n] = _probe(gen, stored[i], n)
    reqs = (G.Request * len(plan))()
    for r, (i, op, n, at) in zip(reqs, plan):
        r.filter, r.op, r.n, r.arrive_us = i, op, n, 0.0
        r.d_keys, r.d_out = keys.data_ptr() + 4 * at, out.data_ptr() + 4 * at
    torch.cuda.synchronize()
    return {"kind": "serve", "filters": fs, "tables": [_table(f) for f in fs], "reqs": reqs, "keys": keys, "out": out}


def run(s):
    kind = s["kind"]
    if kind == "build":
        if s["rsqf"]:
            s["f"].bulk_build(s["keys"])
        else:
            s["f"].bulk_build(s["keys"], NoDuplicates=s["nodup"])
        return s["table"]
    if kind == "lookup":
        s["f"].lookup(s["probe"], s["out"])
        return s["out"]
    if kind == "count":
        s["f"].count(s["probe"], s["out"])
        return s["out"]
    if kind == "window":
        s["f"].delete(s["old"])
        s["f"].insert(s["new"])
        s["old"], s["new"] = s["new"], s["old"]
        return s["table"]
    if kind == "batch":
        s["batch"].build()
        s["batch"].lookup()
        return [s["out"], s["tables"]]
    G.serve(s["filters"], s["reqs"])
    return [s["out"], s["tables"]]


def _table_bytes(case, q):
    if case.get("filter", "rsqf" if case["kind"] == "serve" else "sqf") == "rsqf":
        return ((1 << q) // 64 + 1) * (17 + 8 * case["r"])  # a reference block: 17 + 8 r bytes
    return int(1.1 * (1 << q) * (case["r"] + 3) / 8)


def _touched(n, table):
    """Table bytes n random accesses touch: a 64-byte sector each, the table at most."""
    return min(64 * n, table)


def work(case):
    kind = case["kind"]
    if kind == "batch":
        rng = random.Random(case["filters"] * 1000 + case["qhi"])
        qs = [rng.randint(case["qlo"], case["qhi"]) for _ in range(case["filters"])]
        nk = [_count(rng.uniform(0.3, 0.8), q) for q in qs]
        npr = [int(2 ** rng.uniform(8, 16)) for _ in qs]
        t = [_table_bytes(case, q) for q in qs]
        return {"bytes": 4 * sum(nk) + sum(t) + sum(8 * m + _touched(m, x) for m, x in zip(npr, t)), "flops": 0}
    if kind == "serve":
        # per request its keys (and answers), and the sectors it reads (and writes back)
        shape = random.Random(case["requests"] * 1000 + case["qhi"])
        qs = [shape.randint(case["qlo"], case["qhi"]) for _ in range(case["filters"])]
        b = 0
        for _ in range(case["requests"]):
            i = shape.randrange(len(qs))
            u = shape.random()
            n = _logint(shape, 64, min(case["nmax"], (1 << qs[i]) // 64))
            t = _touched(n, _table_bytes(case, qs[i]))
            b += 8 * n + t if u < 0.7 else 4 * n + 2 * t
        return {"bytes": b, "flops": 0}
    t = _table_bytes(case, case["q"])
    if kind == "build":
        return {"bytes": 4 * _count(case["fill"], case["q"]) + t, "flops": 0}
    n = case["n"]
    if kind == "window":
        return {"bytes": 2 * (4 * n + 2 * _touched(n, t)), "flops": 0}
    return {"bytes": 8 * n + _touched(n, t), "flops": 0}
