"""The window scan of localized updates at both sides of its one-workgroup
form (8192 windows) and at its smallest, SQF and RSQF, insert and delete, bit
for bit; batches whose windows hand them over leave the table to the general
path."""
import numpy as np
import pytest

import gpuquotientfilters_amd as G
import oracle as O
from gpu_helpers import dev, require_gpu, say
from test_gpu_local import _kernels, insert_set, sqf_equal, sqf_table

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    require_gpu()


def _rsqf_equal(f, fps, q, r):
    ok, want = O.rsqf_canon(np.sort(fps), q, r)
    assert ok == O.OK
    got = f.dump()
    assert (got == want).all(), np.flatnonzero(got != want)[:8]


# windows: 2 (SQF 1), 257, 4097, 8193
@pytest.mark.parametrize("q", [12, 20, 24, 25])
@pytest.mark.parametrize("cls", ["SQF", "RSQF"])
@pytest.mark.parametrize("hot", [False, True])
def test_local_scan_sizes(q, cls, hot):
    r = 6 if q == 25 else 8 if cls == "RSQF" else 5
    n = min(120000, O.key_count(0.4, q))
    say("local scan", cls, q, r, hot)
    st = G.Stream()  # a context of its own: no batch of it has been handed over yet
    keys = O.mt19937(950 + q, n)
    b = O.mt19937(951 + q, max(8, n // 60))
    if hot:
        b[: len(b) // 2] = b[0] if cls == "RSQF" else b[: len(b) // 2]
        b = np.concatenate([b, np.repeat(b[-1:], 600)])[: max(8, (1 << q) // 90)]
    f = getattr(G, cls)(q, r)
    f.bulk_build(dev(keys))
    names = _kernels(lambda: f.insert(dev(b), stream=st))
    assert any("_plan" in x for x in names)
    fps, bf = O.fingerprints(keys, q, r), O.fingerprints(b, q, r)
    if cls == "SQF":
        fps = insert_set(np.unique(fps), bf)
        sqf_equal(f, sqf_table(fps, q, r))
    else:
        fps = np.concatenate([fps, bf])
        _rsqf_equal(f, fps, q, r)
    gone = keys[: max(8, n // 70)]
    gone = gone[np.unique(O.fingerprints(gone, q, r), return_index=True)[1]]
    names = _kernels(lambda: f.delete(dev(gone), stream=st))
    assert any("_plan" in x for x in names)
    v, c = np.unique(fps, return_counts=True)
    at = np.searchsorted(v, O.fingerprints(gone, q, r))
    np.subtract.at(c, at, 1)
    fps = np.repeat(v, c)
    if cls == "SQF":
        sqf_equal(f, sqf_table(fps, q, r))
    else:
        _rsqf_equal(f, fps, q, r)
    st.destroy()
