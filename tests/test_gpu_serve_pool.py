"""Serving runs one after another and side by side: workers (streams, contexts,
gather buffers) pass from run to run, and the answers and tables stay those of
single calls; runs with a tight budget start with nothing; gqf_stream_trim
gives the idle ones back."""
import ctypes as C
import threading

import pytest
import torch

import gpuquotientfilters_amd as G
from gpu_helpers import require_gpu, say

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    require_gpu()


def make(seed, qs=(14, 16, 18)):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    rnd = lambda n: torch.randint(-(1 << 31), 1 << 31, (n,), dtype=torch.int32, device="cuda", generator=gen)
    fs, refs, plan = [], [], []
    for i, q in enumerate(qs):
        k = rnd((1 << q) // 2)
        for out in (fs, refs):
            f = G.RSQF(q, 8)
            f.bulk_build(k)
            out.append(f)
        new = rnd((1 << q) // 50)
        plan += [(i, G.OP_LOOKUP, k[: 300 + 7 * i].clone()), (i, G.OP_INSERT, new), (i, G.OP_LOOKUP, new.clone()),
                 (i, G.OP_LOOKUP, rnd(511)), (i, G.OP_DELETE, new)]
    return fs, refs, plan


def serve(fs, plan, **kw):
    outs = [torch.full((len(k),), -7, dtype=torch.int32, device="cuda") for _, _, k in plan]
    reqs = (G.Request * len(plan))()
    for r, (i, op, k), o in zip(reqs, plan, outs):
        r.filter, r.op, r.n, r.arrive_us, r.d_keys, r.d_out = i, op, len(k), 0.0, k.data_ptr(), o.data_ptr()
    torch.cuda.synchronize()
    G.serve(fs, reqs, **kw)
    assert all(r.status == G.OK for r in reqs)
    return outs


def check(fs, refs, plan, **kw):
    outs = serve(fs, plan, **kw)
    for (i, op, k), o in zip(plan, outs):
        if op == G.OP_LOOKUP:
            want = torch.empty_like(o)
            refs[i].lookup(k, want)
            assert torch.equal(o, want)
        elif op == G.OP_INSERT:
            refs[i].insert(k)
        else:
            refs[i].delete(k)
    for f, r in zip(fs, refs):
        assert (f.dump() == r.dump()).all()


def test_runs_in_turn_and_the_pool_given_back():
    fs, refs, plan = make(1)
    resident = sum(G.lib().gqf_rsqf_table_bytes(f.q, f.r) for f in fs)
    for i, kw in enumerate([{}, {}, {"hbm_budget": resident + (8 << 20)}, {"coalesce": False}, {}]):
        say("serve pool, run", i)
        check(fs, refs, plan, **kw)
        if i == 1:
            free0 = torch.cuda.mem_get_info()[0]
            assert G.lib().gqf_stream_trim(None) == G.OK
            assert torch.cuda.mem_get_info()[0] >= free0


def test_runs_side_by_side():
    sets = [make(10 + t, (13 + t, 15, 17)) for t in range(3)]
    errors = []

    def go(t):
        try:
            for _ in range(4):
                check(*sets[t])
        except BaseException as e:  # noqa: BLE001 (reported by the main thread)
            errors.append(e)

    say("serve pool, side by side")
    ts = [threading.Thread(target=go, args=(t,)) for t in range(3)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert not errors, errors
