"""Localized inserts and deletes of small batches (the table's 4096-slot
windows updated in place) against the oracle's end state, bit for bit: slot
widths, fills up to long clusters that cross windows, batch sizes around one
wave's keys, hot keys, keys at window and table ends, and batches that the
localized form hands over to the general path."""
import numpy as np
import pytest

import gpuquotientfilters_amd as G
import oracle as O
from gpu_helpers import dev, require_gpu, say

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    require_gpu()


def _kernels(fn):
    G.synchronize()
    G.profile_reset()
    G.profile_enable(True)
    try:
        fn()
        G.synchronize()
    finally:
        G.profile_enable(False)
    names = set(G.profile_stats())
    G.profile_reset()
    return names


def sqf_table(fps, q, r, no_dup=False):
    """The canonical table of a multiset of fingerprints, as the filter holds it."""
    st, t = O.sqf_canon(np.sort(fps), q, r, no_dup)
    assert st == O.OK
    if (r + 3) % 8:
        return O.sqf_pack(O.sqf_decode(t, q, r), q, r).view(np.uint8)
    return t


def sqf_equal(f, want):
    got = f.table_bytes()
    n = min(len(got), len(want))
    assert (got[:n] == want[:n]).all(), np.flatnonzero(got[:n] != want[:n])[:8]


def insert_set(fps, batch):
    """The insert rule: a batch fingerprint that is stored, or came before, is dropped."""
    return np.concatenate([fps, np.setdiff1d(batch, fps)])


def delete_multiset(fps, batch):
    v, c = np.unique(fps, return_counts=True)
    d, dc = np.unique(batch, return_counts=True)
    at = np.searchsorted(v, d)
    ok = (at < len(v)) & (v[np.minimum(at, len(v) - 1)] == d)
    c = c.copy()
    c[at[ok]] -= np.minimum(c[at[ok]], dc[ok])
    return np.repeat(v, c)


CASES = [(13, 5, 0.5, False), (16, 5, 0.75, False), (18, 5, 0.85, True), (16, 13, 0.9, False), (15, 9, 0.8, False),
         (17, 6, 0.7, True), (20, 5, 0.3, False), (12, 13, 0.6, True)]


@pytest.mark.parametrize("q,r,alpha,dup", CASES)
def test_sqf_local_insert(q, r, alpha, dup):
    say("sqf local insert", q, r, alpha, dup)
    st = G.Stream()  # a context of its own: no batch of it has been handed over yet
    keys = O.mt19937(300 + q, O.key_count(alpha, q))
    if dup:
        keys = np.concatenate([keys[:-50], keys[:50]])
    f = G.SQF(q, r)
    f.bulk_build(dev(keys), NoDuplicates=not dup)
    fps = O.fingerprints(keys, q, r)
    if not dup:
        fps = np.unique(fps)
    S = G.SQF.num_slots(q)
    pool = O.mt19937(301 + q, S)
    at = 0
    local = 0
    for n in [1, 2, 63, 64, 65, 1000, S // 400 + 1, S // 64, S // 33]:
        n = min(n, S // 32, int(0.95 * S) - len(fps))
        if n <= 0:
            break
        b = np.concatenate([pool[at:at + n - n // 4], keys[at:at + n // 4]])
        at += n
        names = _kernels(lambda: f.insert(dev(b), stream=st))
        local += any("k_sl_apply" in x for x in names) and not any("k_rb_write" in x for x in names)
        fps = insert_set(fps, O.fingerprints(b, q, r))
        sqf_equal(f, sqf_table(fps, q, r))
    assert local >= 2  # the localized form ran, and alone
    st.destroy()


def test_sqf_local_insert_hot_and_edges():
    """Hot keys (more than a wave of copies: handed over), keys in the first
    and last slots, clusters across window ends."""
    q, r = 16, 5
    say("sqf local insert edges", q, r)
    cand = O.mt19937(310, 1 << 19)
    fq = O.fingerprints(cand, q, r) >> np.uint64(r)
    edge = cand[(fq % 4096 >= 4056) | (fq % 4096 < 8)]
    ends = cand[(fq < 3) | (fq >= (1 << q) - 3)]
    base = np.concatenate([O.mt19937(311, O.key_count(0.6, q)), edge[:1500]])
    f = G.SQF(q, r)
    f.bulk_build(dev(base))
    fps = np.unique(O.fingerprints(base, q, r))
    for b in [edge[1500:2700], ends[:40], np.full(30, cand[0]), np.full(900, cand[1]), edge[2700:3400],
              np.concatenate([np.full(500, cand[2]), edge[3400:3500]])]:
        f.insert(dev(b))
        fps = insert_set(fps, O.fingerprints(b, q, r))
        sqf_equal(f, sqf_table(fps, q, r))


@pytest.mark.parametrize("q,r,alpha,dup", CASES)
def test_sqf_local_delete(q, r, alpha, dup):
    """Stored keys, keys that are not stored, repeated keys, several copies."""
    say("sqf local delete", q, r, alpha, dup)
    st = G.Stream()
    keys = O.mt19937(320 + q, O.key_count(alpha, q))
    if dup:
        keys = np.concatenate([keys[:-50], keys[:25], keys[:25]])
    f = G.SQF(q, r)
    f.bulk_build(dev(keys), NoDuplicates=not dup)
    fps = O.fingerprints(keys, q, r)
    if not dup:
        fps = np.unique(fps)
    S = G.SQF.num_slots(q)
    other = O.mt19937(321 + q, S)
    at = local = 0
    for n in [1, 2, 63, 64, 65, 1000, S // 400 + 1, S // 82]:
        n = min(n, S // 82)
        if n <= 0:
            break
        b = np.concatenate([keys[at:at + n - n // 3], keys[at:at + n // 6], other[at:at + n // 6]])
        at += n
        names = _kernels(lambda: f.superclusterDeletes(dev(b), stream=st))
        local += any("k_sl_apply" in x for x in names) and not any("k_rb_write" in x for x in names)
        fps = delete_multiset(fps, O.fingerprints(b, q, r))
        sqf_equal(f, sqf_table(fps, q, r))
    assert local >= 2
    st.destroy()


def test_sqf_local_delete_hot_and_edges():
    q, r = 16, 5
    say("sqf local delete edges", q, r)
    cand = O.mt19937(330, 1 << 19)
    fq = O.fingerprints(cand, q, r) >> np.uint64(r)
    edge = cand[(fq % 4096 >= 4056) | (fq % 4096 < 8)]
    ends = cand[(fq < 3) | (fq >= (1 << q) - 3)]
    base = np.concatenate([O.mt19937(331, O.key_count(0.6, q)), edge[:2500], ends[:30], np.full(90, cand[5])])
    f = G.SQF(q, r)
    f.bulk_build(dev(base), NoDuplicates=False)
    fps = O.fingerprints(base, q, r)
    for b in [edge[:800], ends[:40], np.full(30, cand[5]), np.full(70, cand[5]), edge[800:1600], base[:800],
              edge[1600:2400]]:
        f.superclusterDeletes(dev(b))
        fps = delete_multiset(fps, O.fingerprints(b, q, r))
        sqf_equal(f, sqf_table(fps, q, r))


# ---------------------------------------------------------------- RSQF
RCASES = [(13, 8, 0.5), (16, 8, 0.8), (18, 8, 0.9), (16, 16, 0.9), (17, 5, 0.85), (16, 11, 0.8), (20, 13, 0.5),
          (15, 1, 0.5), (25, 8, 0.1)]


def rsqf_table(fps, q, r):
    st, t = O.rsqf_canon(np.sort(fps), q, r)
    assert st == O.OK
    return t


def rsqf_equal(f, want):
    got = f.dump()
    assert (got == want).all(), np.flatnonzero(got != want)[:8]


@pytest.mark.parametrize("q,r,alpha", RCASES)
def test_rsqf_local_insert(q, r, alpha):
    say("rsqf local insert", q, r, alpha)
    st = G.Stream()
    keys = O.mt19937(340 + q + r, O.key_count(alpha, q))
    f = G.RSQF(q, r)
    f.bulk_build(dev(keys))
    fps = O.fingerprints(keys, q, r)
    S = 1 << q
    pool = O.mt19937(341 + q, S)
    at = local = 0
    for n in [1, 2, 63, 64, 65, 1000, S // 400 + 1, S // 82]:
        n = min(n, S // 82)
        b = np.concatenate([pool[at:at + n - n // 4], keys[at:at + n // 4]])
        at += n
        if len(b) == 0:
            continue
        out = G.DeviceArray.empty(len(b))
        names = _kernels(lambda: f.insert(dev(b), out, stream=st))
        ran = any("k_rl_apply" in x for x in names)
        alone = not any("k_wm_write" in x or "k_rr_write" in x for x in names)
        local += ran and alone
        fps = np.concatenate([fps, O.fingerprints(b, q, r)])
        want = rsqf_table(fps, q, r)
        rsqf_equal(f, want)
        assert (out.to_host() == O.rsqf_lookup_keys(want, q, r, b)).all()
    assert local >= 2
    st.destroy()


def test_rsqf_local_insert_hot_and_edges():
    q, r = 16, 8
    say("rsqf local insert edges", q, r)
    cand = O.mt19937(350, 1 << 19)
    fq = O.fingerprints(cand, q, r) >> np.uint64(r)
    edge = cand[((fq % 4096 >= 4056) | (fq % 4096 < 8)) & (fq < (1 << q) - 64)]  # the last block overflows
    ends = cand[(fq < 3) | (fq >= (1 << q) - 3)]
    base = np.concatenate([O.mt19937(351, O.key_count(0.6, q)), edge[:1500]])
    f = G.RSQF(q, r)
    f.bulk_build(dev(base))
    fps = O.fingerprints(base, q, r)
    # (30 copies: one region; 70 and 300: a wave of copies and more, handed over)
    for b in [edge[1500:2200], ends[:40], np.full(30, cand[0]), np.full(70, cand[1]), np.full(300, cand[1]),
              edge[2200:2900], np.concatenate([np.full(40, cand[1]), edge[2900:3000]])]:
        f.insert(dev(b))
        fps = np.concatenate([fps, O.fingerprints(b, q, r)])
        rsqf_equal(f, rsqf_table(fps, q, r))


@pytest.mark.parametrize("q,r,alpha", RCASES)
def test_rsqf_local_delete(q, r, alpha):
    """Stored keys, keys that are not stored, repeated keys, several copies."""
    say("rsqf local delete", q, r, alpha)
    st = G.Stream()
    keys = O.mt19937(360 + q + r, O.key_count(alpha, q))
    keys = np.concatenate([keys[:-50], keys[:25], keys[:25]])
    f = G.RSQF(q, r)
    f.bulk_build(dev(keys))
    fps = O.fingerprints(keys, q, r)
    S = 1 << q
    other = O.mt19937(361 + q, S)
    at = local = 0
    for n in [1, 2, 63, 64, 65, 1000, S // 400 + 1, S // 82]:
        n = min(n, S // 82)
        b = np.concatenate([keys[at:at + n - n // 3], keys[at:at + n // 6], other[at:at + n // 6]])
        at += n
        if len(b) == 0:
            continue
        names = _kernels(lambda: f.deleteGPU(dev(b), stream=st))
        local += any("k_rl_apply" in x for x in names) and not any("k_rr_write" in x for x in names)
        fps = delete_multiset(fps, O.fingerprints(b, q, r))
        rsqf_equal(f, rsqf_table(fps, q, r))
    assert local >= 2
    st.destroy()


def test_rsqf_local_delete_hot_and_edges():
    q, r = 16, 8
    say("rsqf local delete edges", q, r)
    cand = O.mt19937(370, 1 << 19)
    fq = O.fingerprints(cand, q, r) >> np.uint64(r)
    edge = cand[((fq % 4096 >= 4056) | (fq % 4096 < 8)) & (fq < (1 << q) - 64)]
    ends = cand[(fq < 3) | (fq >= (1 << q) - 3)]
    base = np.concatenate([O.mt19937(371, O.key_count(0.6, q)), edge[:2500], ends[:30], np.full(90, cand[5])])
    f = G.RSQF(q, r)
    f.bulk_build(dev(base))
    fps = O.fingerprints(base, q, r)
    for b in [edge[:700], ends[:40], np.full(30, cand[5]), np.full(70, cand[5]), edge[700:1400], base[:700],
              edge[1400:2100]]:
        f.deleteGPU(dev(b))
        fps = delete_multiset(fps, O.fingerprints(b, q, r))
        rsqf_equal(f, rsqf_table(fps, q, r))
