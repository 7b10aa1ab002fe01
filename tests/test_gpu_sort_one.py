"""The one-workgroup sort (up to 16384 keys), seen through builds, bit for
bit: the edges of its tile and of a thread's share, ranges of fewer bits than
the bucket index, full 32-bit ranges, and buckets crowded by copies of a key
or by neighbouring fingerprints."""
import numpy as np
import pytest

import gpuquotientfilters_amd as G
import oracle as O
from gpu_helpers import dev, require_gpu, say
from test_gpu_local import _kernels, sqf_equal, sqf_table

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    require_gpu()


@pytest.mark.parametrize("q,r,n,copies", [
    (10, 5, 1, 0), (10, 5, 2, 0), (8, 5, 200, 0), (16, 5, 1023, 0), (16, 13, 4095, 0), (16, 5, 4097, 33),
    (17, 13, 16383, 0), (17, 13, 16384, 0), (19, 13, 16384, 34), (16, 5, 12000, 9000), (14, 13, 8193, 32),
    (17, 13, 16385, 0),
])
def test_build_by_the_one_workgroup_sort(q, r, n, copies):
    say("one-workgroup sort", q, r, n, copies)
    keys = O.mt19937(800 + n, n)
    keys[:copies] = keys[n - 1]
    keys = keys[np.random.default_rng(n).permutation(n)]
    f = G.SQF(q, r)
    d = dev(keys)
    names = _kernels(lambda: f.bulk_build(d, NoDuplicates=False))
    sqf_equal(f, sqf_table(O.fingerprints(keys, q, r), q, r))
    assert any("k_rs_one" in x for x in names) == (n <= 16384)
