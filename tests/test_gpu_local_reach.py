"""Localized inserts whose region runs from one window into the next: up to 64
keys that the first has no room for, and the keys of the second that it takes
with it, where the second has few empty slots in its first blocks.  Every key
has to be there, wherever the call's rules draw the line."""
import numpy as np
import pytest

import gpuquotientfilters_amd as G
import oracle as O
from gpu_helpers import dev, require_gpu, say
from test_gpu_local import _kernels, insert_set, rsqf_equal, rsqf_table, sqf_equal, sqf_table

pytestmark = pytest.mark.gpu

Q, W0 = 20, 5 * 4096  # more windows than batch keys; the window that overflows
HALO = 45 * 64        # slots of the next window that a region may reach (RSQF)


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    require_gpu()


def key_of_quotient(q, r, lo, hi):
    """A key for every quotient of [lo, hi)."""
    keys = O.mt19937(7, 1 << 24)
    fq = (O.fingerprints(keys, q, r) >> np.uint64(r)).astype(np.int64)
    sel = np.flatnonzero((fq >= lo) & (fq < hi))
    u, first = np.unique(fq[sel], return_index=True)
    assert len(u) == hi - lo
    return keys[sel[first]]


def crowded(r, empties, x, c):
    """Stored keys and a batch: slot W0 + 4095 and, in the next window's first
    HALO slots, all but `empties` are taken; x copies of the former's key and c
    keys past the 22nd of those empty slots."""
    lo, nxt = W0 + 4095, W0 + 4096
    key = key_of_quotient(Q, r, lo, nxt + HALO)
    s = np.arange(HALO)
    gap = HALO // empties
    stored = np.concatenate([key[:1], key[1:][(s % gap != 0) | (s // gap >= empties)]])
    batch = np.concatenate([np.repeat(key[:1], x), key[1 + 1000:1 + 1000 + 40 * c:40]])
    return stored, batch


@pytest.mark.parametrize("x,c,empties", [(x, c, e) for e in (64, 72) for x, c in [
    (64, 0), (63, 1), (63, 2), (64, 1), (64, 7), (60, 20), (65, 1), (40, 3)]] + [
    (8, 0, 8), (7, 1, 8), (8, 1, 8), (7, 2, 8), (1, 0, 1), (9, 1, 10), (9, 2, 10), (6, 2, 8), (6, 3, 8)])
def test_rsqf_insert_across_a_window(x, c, empties):
    r = 8
    say("rsqf insert across a window", x, c, empties)
    st = G.Stream()
    stored, batch = crowded(r, empties, x, c)
    f = G.RSQF(Q, r)
    f.bulk_build(dev(stored))
    names = _kernels(lambda: f.insert(dev(batch), stream=st))
    fps = np.concatenate([O.fingerprints(stored, Q, r), O.fingerprints(batch, Q, r)])
    rsqf_equal(f, rsqf_table(fps, Q, r))
    if x < 10:  # (more copies of a key than that take the general path in a table of this size)
        assert any("k_rl_apply" in k for k in names) and any("k_wm_write" in k for k in names) == (x + c > empties)
    # what is left in place after the same keys are deleted again
    f.deleteGPU(dev(batch), stream=st)
    left = np.sort(fps)
    at = np.searchsorted(left, np.sort(O.fingerprints(batch, Q, r)), side="left")
    keep = np.ones(len(left), bool)
    for a in at:
        while not keep[a]:
            a += 1
        keep[a] = False
    rsqf_equal(f, rsqf_table(left[keep], Q, r))
    st.destroy()


@pytest.mark.parametrize("x,c", [(64, 0), (63, 2), (64, 20), (30, 20)])
def test_sqf_insert_across_a_window(x, c):
    """The SQF stores a fingerprint once: x different remainders at the quotient."""
    r = 8  # packed slots
    say("sqf insert across a window", x, c)
    st = G.Stream()
    keys = O.mt19937(9, 1 << 24)
    fp = O.fingerprints(keys, Q, r)
    fq = (fp >> np.uint64(r)).astype(np.int64)
    lo = W0 + 4095
    sel = np.flatnonzero((fq >= lo) & (fq < lo + 1 + HALO))
    _, first = np.unique(fq[sel], return_index=True)
    key = keys[sel[first]]
    near = np.flatnonzero((fq > lo - 30) & (fq <= lo))  # about 16 keys a quotient
    s = np.arange(HALO)
    stored = np.concatenate([keys[near[-40:]], key[1:][(s % 45 != 0) | (s // 45 >= 64)]])
    batch = np.concatenate([keys[near[:x]], key[1 + 1000:1 + 1000 + 40 * c:40]])
    f = G.SQF(Q, r)
    f.bulk_build(dev(stored))
    f.insert(dev(batch), stream=st)
    fps = np.unique(insert_set(np.unique(O.fingerprints(stored, Q, r)), O.fingerprints(batch, Q, r)))
    sqf_equal(f, sqf_table(fps, Q, r))
    st.destroy()


@pytest.mark.parametrize("past,local", [(20, True), (690, True), (760, False), (1500, False)])
@pytest.mark.parametrize("q,r", [(20, 5), (17, 13)])
def test_sqf_clusters_past_a_window(q, r, past, local):
    """A cluster of shifted entries from a window's end to `past` slots into the
    next: updates in it are localized while the slots are held, handed over
    beyond that; updates before it are localized in any case."""
    say("sqf cluster past a window", q, r, past)
    lo = W0 + 4096 - 20
    pool = O.mt19937(11, 1 << 25)
    fp = O.fingerprints(pool, q, r)
    fq = (fp >> np.uint64(r)).astype(np.int64)
    sel = np.flatnonzero((fq >= lo) & (fq < W0 + 4096 + past))
    _, first = np.unique(fq[sel], return_index=True)
    key = pool[sel[first]]
    assert len(key) == 20 + past
    own = pool[fq == lo]
    own = own[np.unique(O.fingerprints(own, q, r), return_index=True)[1]][:4]  # shift the others by 3
    alone = pool[np.flatnonzero(fq == W0 + 100)[:1]]
    f = G.SQF(q, r)
    f.bulk_build(dev(np.concatenate([own, key[1:], alone])))
    fps = np.unique(O.fingerprints(np.concatenate([own, key[1:], alone]), q, r))
    inside = pool[np.flatnonzero((fq == lo + 5) & ~np.isin(fp, fps))[:1]]
    for batch, is_local in ((inside, local), (pool[np.flatnonzero(fq == W0 + 50)[:1]], True)):
        st = G.Stream()  # a context of its own: no batch of it has been handed over yet
        names = _kernels(lambda: f.insert(dev(batch), stream=st))
        fps = np.unique(insert_set(fps, O.fingerprints(batch, q, r)))
        sqf_equal(f, sqf_table(fps, q, r))
        assert any("k_rb_write" in x for x in names) == (not is_local)
        st.destroy()
    for batch, is_local in ((key[6:7], local), (alone, True), (inside, local)):
        st = G.Stream()
        names = _kernels(lambda: f.delete(dev(batch), stream=st))
        fps = fps[~np.isin(fps, O.fingerprints(batch, q, r))]
        sqf_equal(f, sqf_table(fps, q, r))
        assert any("k_rb_write" in x for x in names) == (not is_local)
        st.destroy()
