"""Bulk builds by runs (more than 256 * 7600 keys, remainders of up to 8
bits, tables that are not sparse), bit for bit against the canonical layout:
both sides of the size rules, every group width, plain, packed and RSQF
tables, fingerprints past 32 bits, repeats kept and dropped, clusters across
group ends, and the key sets that this form hands over to the sort."""
import numpy as np
import pytest

import gpuquotientfilters_amd as G
import oracle as O
from gpu_helpers import dev, require_gpu, say
from test_gpu_local import _kernels, sqf_equal, sqf_table

pytestmark = pytest.mark.gpu
EDGE = 256 * 7600  # the largest batch that is sorted


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    require_gpu()


def _keys(kind, q, r, n):
    """n keys with a share of repeats, runs of many entries and clusters at
    the ends of quotient ranges of 2^12 .. 2^15."""
    keys = O.mt19937(700 + q, n)
    keys[n - n // 16:] = keys[:n // 16]
    cand = O.mt19937(701, 1 << 20)
    fq = O.fingerprints(cand, q, r) >> np.uint64(r)
    if kind == "repeats":
        keys = keys[:900000][np.random.default_rng(9).integers(0, 900000, n)]
    elif kind == "run":  # one run of more than 255 entries
        keys[:256] = cand[0]
    elif kind == "dense":  # more than 255 keys in 32 neighbouring quotients
        near = cand[(fq // 32) == (fq[0] // 32)]
        keys[:300] = np.resize(near, 300)
    elif kind in ("ends", "spill"):  # entries that reach past group ends
        end = cand[(fq % 32768) >= 32768 - 128]
        ef = O.fingerprints(end, q, r) >> np.uint64(r)
        _, one = np.unique(ef // 32, return_index=True)  # a quotient in every 32
        end = end[np.sort(one)][:40]
        if kind == "ends":
            keys[:2800] = np.resize(np.repeat(end, 70), 2800)
        else:  # 4 runs of 200 before one group end
            f = O.fingerprints(cand, q, r) >> np.uint64(r)
            last = (f[0] | np.uint64(32767)) + np.uint64(1)
            near = cand[(f < last) & (f >= last - np.uint64(256))]
            _, one = np.unique((O.fingerprints(near, q, r) >> np.uint64(r)) // 32, return_index=True)
            near = near[one][-6:]
            keys[:200 * len(near)] = np.repeat(near, 200)
    return keys[np.random.default_rng(q).permutation(n)]


SQF = [(21, 5, EDGE, "", False, False), (21, 5, EDGE + 1, "", True, True), (21, 5, EDGE + 1, "", False, True),
       (21, 6, 1960003, "ends", False, True), (22, 8, 3900001, "", True, True), (22, 5, 3900001, "ends", False, True),
       (23, 7, 7654321, "ends", False, True), (24, 5, 15000001, "", True, True), (24, 5, 2800000, "ends", False, True),
       (24, 5, 2790000, "ends", False, False),
       (20, 5, 2500001, "repeats", True, True), (22, 5, 3000000, "run", False, False), (21, 6, 1950000, "dense", False, False),
       (22, 5, 3900000, "spill", False, False)]


@pytest.mark.parametrize("q,r,n,kind,no_dup,runs", SQF)
def test_sqf_build_by_runs(q, r, n, kind, no_dup, runs):
    say("sqf build by runs", q, r, n, kind, no_dup)
    st = G.Stream()  # a context of its own: no build of it has been handed over yet
    keys = _keys(kind, q, r, n)
    f = G.SQF(q, r)
    d = dev(keys)
    names = _kernels(lambda: f.bulk_build(d, NoDuplicates=no_dup, stream=st))
    fps = O.fingerprints(keys, q, r)
    sqf_equal(f, sqf_table(fps, q, r, no_dup))
    assert any("k_rb_write" in x for x in names) == (not runs)
    assert any("k_db_sqf" in x for x in names) == (n > EDGE and 6 * n >= 1 << q)
    st.destroy()


RSQF = [(21, 5, EDGE + 1, ""), (21, 1, EDGE + 5, ""), (22, 8, 3900001, "ends"), (23, 7, 7654321, ""),
        (25, 8, EDGE + 77, "ends"), (26, 8, (1 << 21) + 3, ""), (26, 8, (1 << 21) - 1, ""), (22, 5, 3000000, "run"), (22, 5, 3900000, "spill")]


@pytest.mark.parametrize("q,r,n,kind", RSQF)
def test_rsqf_build_by_runs(q, r, n, kind):
    say("rsqf build by runs", q, r, n, kind)
    st = G.Stream()
    keys = _keys(kind, q, r, n)
    f = G.RSQF(q, r)
    d = dev(keys)
    names = _kernels(lambda: f.bulk_build(d, stream=st))
    ok, want = O.rsqf_canon(O.fingerprints(keys, q, r), q, r)
    assert ok == O.OK
    got = f.dump()
    assert (got == want).all(), np.flatnonzero(got != want)[:8]
    assert any("k_rr_write" in x for x in names) == (kind in ("run", "spill") or 32 * n < 1 << q)
    st.destroy()


@pytest.mark.parametrize("cls", ["SQF", "RSQF"])
def test_build_by_runs_capacity(cls):
    """Keys that do not fit leave the table as it was."""
    q, r = 20, 8
    say("build by runs capacity", cls)
    f = getattr(G, cls)(q, r)
    f.bulk_build(dev(O.mt19937(720, 700000)))
    dump = f.table_bytes if cls == "SQF" else f.dump
    before = np.array(dump(), copy=True)
    with pytest.raises(G.CapacityError):
        f.bulk_build(dev(O.mt19937(721, EDGE + 1000)))
    assert (dump() == before).all()
