"""Small batches whose longest region would take its lane longer than the
general path takes the table: copies of one key, and keys crowded in the long
clusters of full tables, are handed over; ordinary batches of the same sizes
are not.  The tables are the canonical ones either way."""
import numpy as np
import pytest

import gpuquotientfilters_amd as G
import oracle as O
from gpu_helpers import dev, require_gpu, say
from test_gpu_local import _kernels, delete_multiset, insert_set, rsqf_equal, rsqf_table, sqf_equal, sqf_table

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    require_gpu()


def handed(names):
    assert any("l_apply" in x for x in names)  # k_sl_apply, k_rl_apply
    return any(w in x for x in names for w in ("k_rb_write", "k_wm_write", "k_rr_write"))


# table, fill, batch: (kind, n), whether inserts and deletes are handed over
RSQF = [(20, 8, 0.9, "copies", 60, True, True), (20, 8, 0.5, "copies", 60, True, True), (18, 16, 0.7, "copies", 63, True, True),
        (20, 8, 0.75, "uniform", 1000, False, False), (20, 8, 0.5, "copies", 2, False, False),
        (22, 5, 0.8, "sixteen", 1000, True, True), (22, 8, 0.85, "uniform", 4000, False, False)]


@pytest.mark.parametrize("q,r,fill,kind,n,ins,dele", RSQF)
def test_rsqf(q, r, fill, kind, n, ins, dele):
    say("local budget, rsqf", q, r, fill, kind, n)
    keys = O.mt19937(600 + q, O.key_count(fill, q))
    b = O.mt19937(601 + q, n)
    if kind == "copies":
        b[:] = b[0]
    elif kind == "sixteen":
        b = b[np.arange(n) % 16]
    f = G.RSQF(q, r)
    f.bulk_build(dev(keys))
    fps, bf = O.fingerprints(keys, q, r), O.fingerprints(b, q, r)
    st = G.Stream()  # a context of its own: no batch of it has been handed over yet
    names = _kernels(lambda: f.insert(dev(b), stream=st))
    rsqf_equal(f, rsqf_table(np.concatenate([fps, bf]), q, r))
    assert handed(names) == ins
    names = _kernels(lambda: f.deleteGPU(dev(b), stream=st))
    rsqf_equal(f, rsqf_table(fps, q, r))
    assert handed(names) == dele
    st.destroy()


SQF = [(22, 5, 0.9, 30011, True, True), (20, 5, 0.9, 10007, True, True), (18, 13, 0.9, 1500, True, True),
       (22, 5, 0.75, 10007, False, False), (20, 5, 0.5, 3001, False, False)]


@pytest.mark.parametrize("q,r,fill,n,ins,dele", SQF)
def test_sqf(q, r, fill, n, ins, dele):
    say("local budget, sqf", q, r, fill, n)
    keys = O.mt19937(610 + q, O.key_count(fill, q))
    b = O.mt19937(611 + q, n)
    f = G.SQF(q, r)
    f.bulk_build(dev(keys))
    fps, bf = np.unique(O.fingerprints(keys, q, r)), O.fingerprints(b, q, r)
    st = G.Stream()
    names = _kernels(lambda: f.insert(dev(b), stream=st))
    fps = np.unique(insert_set(fps, bf))
    sqf_equal(f, sqf_table(fps, q, r))
    assert handed(names) == ins
    names = _kernels(lambda: f.superclusterDeletes(dev(b), stream=st))
    sqf_equal(f, sqf_table(delete_multiset(fps, bf), q, r))
    assert handed(names) == dele
    st.destroy()
