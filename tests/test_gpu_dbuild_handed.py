"""Builds by runs that are handed over: the work that is left when the
partition has seen that the keys do not fit is not done."""
import numpy as np
import pytest

import gpuquotientfilters_amd as G
import oracle as O
from gpu_helpers import dev, require_gpu, say
from test_gpu_local import rsqf_equal, rsqf_table, sqf_equal, sqf_table

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    require_gpu()


def runs_ms(fn):
    G.synchronize()
    G.profile_reset()
    G.profile_enable(True)
    try:
        fn()
        G.synchronize()
    finally:
        G.profile_enable(False)
    stats = G.profile_stats()
    G.profile_reset()
    ms = [v[1] for k, v in stats.items() if "k_db_runs" in k]
    assert len(ms) == 1
    return ms[0]


@pytest.mark.parametrize("cls,no_dup", [("SQF", True), ("SQF", False), ("RSQF", False)])
def test_runs_of_a_build_that_the_partition_hands_over(cls, no_dup):
    q, r, n = 22, 5, 3700000
    say("build handed over by the partition", cls, no_dup)
    keys = O.mt19937(730, n)
    near = O.mt19937(731, 1 << 24)
    near = near[O.fingerprints(near, q, r) >> np.uint64(r + 14) == 3]  # one group's quotients
    assert len(near) > 40000
    crowded = keys.copy()
    crowded[1000:1000 + 40000] = near[:40000]
    f = getattr(G, cls)(q, r)
    kw = {"NoDuplicates": no_dup} if cls == "SQF" else {}

    def build(k):
        st = G.Stream()  # a context of its own: no build of it has been handed over yet
        d = dev(k)
        f.bulk_build(dev(k[:1000]), stream=st, **kw)
        ms = runs_ms(lambda: f.bulk_build(d, stream=st, **kw))
        st.destroy()
        return ms

    build(keys)
    whole, handed = build(keys), build(crowded)
    fps = O.fingerprints(crowded, q, r)
    if cls == "SQF":
        sqf_equal(f, sqf_table(fps, q, r, no_dup))
    else:
        rsqf_equal(f, rsqf_table(fps, q, r))
    say("whole, handed", whole, handed)
    assert handed < whole / 2
