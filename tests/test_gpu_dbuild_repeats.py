"""Builds by runs of keys with many copies: repeats kept and dropped, runs of
lengths around those that a lane, a wave in one round and a wave in several
sort, of one value and of several, in every number of quotients per thread,
and in both forms (a stream expects many copies until a build has shown few).
Bit for bit against the canonical layout."""
import numpy as np
import pytest

import gpuquotientfilters_amd as G
import oracle as O
from gpu_helpers import dev, require_gpu, say
from test_gpu_local import _kernels, rsqf_equal, rsqf_table, sqf_equal, sqf_table

pytestmark = pytest.mark.gpu
LENGTHS = [2, 5, 8, 9, 23, 24, 25, 26, 63, 64, 65, 127, 128, 129]
LONG = [191, 192, 193, 200, 210]  # where few other keys lie near (255 per 32 quotients)


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    require_gpu()


def with_runs(keys, q, r, seed):
    """keys, the first of them replaced by runs of LENGTHS (and LONG) entries, of
    up to six values each, at quotients far from each other."""
    lengths = LENGTHS + (LONG if len(keys) < (1 << q) // 3 else [])
    pool = O.mt19937(740, 1 << 23)
    fq = (O.fingerprints(pool, q, r) >> np.uint64(r)).astype(np.int64)
    rng = np.random.default_rng(seed)
    at = 0
    for i in range(4 * len(lengths)):
        n = lengths[i % len(lengths)]
        quotient = fq[rng.integers(0, len(fq))]
        own = pool[fq == quotient][:1 if i % 3 == 0 else 6]
        keys[at:at + n] = own[rng.integers(0, len(own), n)]
        at += n
    return rng.permutation(keys)


CASES = [(20, 5, 2000003, 8, True), (21, 5, 1960001, 4, True), (21, 8, 1960001, 1.5, True), (22, 5, 2100001, 32, True),
         (22, 5, 3500003, 4, True), (22, 8, 2500001, 8, False), (23, 5, 3000001, 2, True), (24, 5, 4000001, 8, True),
         (24, 7, 4000001, 12, False), (24, 5, 5000001, 1, True)]


@pytest.mark.parametrize("q,r,n,copies,no_dup", CASES)
def test_sqf_repeats(q, r, n, copies, no_dup):
    say("sqf build of repeats", q, r, n, copies, no_dup)
    st = G.Stream()
    few = O.mt19937(741, n)
    pool = few[:int(n / copies)]
    keys = few if copies == 1 else pool[np.random.default_rng(5).integers(0, len(pool), n)]
    if q >= 22:  # (more than 255 keys per 32 quotients otherwise)
        keys = with_runs(keys.copy(), q, r, q)
    f = G.SQF(q, r)
    d = dev(keys)
    want = sqf_table(O.fingerprints(keys, q, r), q, r, no_dup)
    for form in ("many", "few"):
        names = _kernels(lambda: f.bulk_build(d, NoDuplicates=no_dup, stream=st))
        assert any("k_db_sqf" in x for x in names) and not any("k_rb_write" in x for x in names)
        sqf_equal(f, want)
        if q < 22:
            break
        f.bulk_build(dev(few), NoDuplicates=no_dup, stream=st)  # shows few
    st.destroy()


@pytest.mark.parametrize("q,r,n,copies", [(22, 8, 2100001, 32), (22, 5, 3000001, 4), (23, 8, 3000001, 8), (25, 8, 3000001, 32)])
def test_rsqf_repeats(q, r, n, copies):
    say("rsqf build of repeats", q, r, n, copies)
    st = G.Stream()
    few = O.mt19937(742, n)
    pool = few[:int(n / copies)]
    keys = with_runs(pool[np.random.default_rng(5).integers(0, len(pool), n)], q, r, q)
    f = G.RSQF(q, r)
    d = dev(keys)
    want = rsqf_table(O.fingerprints(keys, q, r), q, r)
    for form in ("many", "few"):
        names = _kernels(lambda: f.bulk_build(d, stream=st))
        assert any("k_db_rsqf" in x for x in names) and not any("k_rr_write" in x for x in names)
        rsqf_equal(f, want)
        f.bulk_build(dev(few), stream=st)
    st.destroy()


def test_dropped_repeats_take_no_longer():
    """The runs of keys that are copied 32 times: up to four times as long as
    those of single keys (ten times with each repeat dropped by itself)."""
    q, r, n = 22, 5, 2100001
    say("build of repeats, time")
    st = G.Stream()
    f = G.SQF(q, r)
    few = O.mt19937(743, n)
    pool = few[:n // 32]
    many = pool[np.random.default_rng(5).integers(0, len(pool), n)]

    def runs_ms(k):
        d = dev(k)
        f.bulk_build(d, stream=st)
        best = 1e9
        for _ in range(5):
            G.synchronize()
            G.profile_reset()
            G.profile_enable(True)
            f.bulk_build(d, stream=st)
            G.synchronize()
            G.profile_enable(False)
            best = min(best, sum(v[1] for k, v in G.profile_stats().items() if "k_db_runs" in k))
        G.profile_reset()
        return best

    a, b = runs_ms(few), runs_ms(many)
    say("few, many", a, b)
    assert b < 4 * a
    st.destroy()
