"""Forms that other tests compare by their results only, on streams of their
own, so that no earlier call of the process decides which one runs: sorts
through one region per segment, and localized RSQF updates of tables that the
reference's own insert wrote."""
import numpy as np
import pytest

import gpuquotientfilters_amd as G
import oracle as O
from conftest import golden
from gpu_helpers import dev, require_gpu, rsqf_lookup, say, sqf_canon
from test_gpu_local import _kernels

pytestmark = pytest.mark.gpu
PARTITION = ("k_rs_upsweep", "k_rs_rowscan", "k_rs_downsweep", "k_rs_segbase")


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    require_gpu()


@pytest.fixture
def stream():
    s = G.Stream()
    yield s
    s.destroy()


def has(names, *kernels):
    return any(k in x for x in names for k in kernels)


@pytest.mark.parametrize("kind,r,n", [("sqf", 5, 16385), ("sqf", 5, 131073), ("sqf", 5, 524289), ("rsqf", 13, 16385),
                                      ("rsqf", 13, 131073)])
def test_sorts_through_regions(stream, kind, r, n):
    """Uniform keys twice (both turns of the counters), then more keys of one
    segment than its region holds: that call and the next four go by the
    counted partition."""
    q = 20
    say("sort through regions", kind, r, n)
    f = (G.SQF if kind == "sqf" else G.RSQF)(q, r)
    uniform = O.mt19937(n, n)
    many = 4 * (n // 256) + 600
    pool = O.mt19937(n + 1, 300 * many)
    top = O.fingerprints(pool, q, r).astype(np.uint64) >> np.uint64(q + r - 8)
    crowded = uniform.copy()
    crowded[:many] = pool[top == 3][:many]
    for i, (keys, place, count) in enumerate([(uniform, True, False), (uniform[::-1].copy(), True, False),
                                              (crowded, True, True), (uniform, False, True)]):
        d = dev(keys)
        G.synchronize()
        if kind == "sqf":
            want = sqf_canon(keys, q, r, True)
            names = _kernels(lambda: f.bulk_build(d, NoDuplicates=True, stream=stream))
            assert (f.table_bytes() == want).all()
        else:
            st, want = O.rsqf_canon(O.fingerprints(keys, q, r), q, r)
            assert st == O.OK
            names = _kernels(lambda: f.bulk_build(d, stream=stream))
            assert (f.dump() == want).all()
        assert has(names, "k_rs_place") == place and has(names, *PARTITION) == count, (i, names)


@pytest.mark.parametrize("table", ["table_random", "table_ascending"])
def test_localized_rsqf_updates_of_reference_tables(stream, table):
    """History-dependent layouts, with holes: one batch in and half of it out,
    beside the rebuilds (a delete of more keys, the others not stored)."""
    name = "rsqf_r5_q12_a0.9.npz"
    g = golden(name)
    q, r = int(g["q"]), int(g["r"])
    say("localized rsqf on reference table", name, table)
    keys = O.mt19937(84, 20)
    f = G.RSQF(q, r)
    f.load(g[table])
    f.insertGPU(dev(keys))
    probe = O.mt19937(85, 1 << 13)
    absent = probe[rsqf_lookup(f, probe) == G.NOT_FOUND][:400]
    assert len(absent) == 400
    out, ran = [], []
    for path, gone in ((G.INSERT_AUTO, keys[::2]), (G.INSERT_REBUILD, np.concatenate([keys[::2], absent]))):
        G.set_rsqf_insert_path(path)
        try:
            f = G.RSQF(q, r)
            f.load(g[table])
            a, b = dev(keys), dev(gone)
            G.synchronize()
            ran.append(_kernels(lambda: f.insertGPU(a, stream=stream)))
            first = f.dump()
            ran.append(_kernels(lambda: f.deleteGPU(b, stream=stream)))
            out.append((first, f.dump()))
        finally:
            G.set_rsqf_insert_path(G.INSERT_AUTO)
    assert (out[0][0] == out[1][0]).all() and (out[0][1] == out[1][1]).all()
    assert (out[0][0] != out[0][1]).any()
    assert [has(x, "k_rl_apply") for x in ran] == [True, True, False, False]
