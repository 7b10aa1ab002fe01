"""Sorts through one region per segment (k_rs_place): bulk builds whose sorts
take it, at the sizes where the tile changes, uniform and skewed keys in turn
on one stream (a full region hands the keys to the counted partition, and the
counters of both turns have to be clean), against the oracle's tables."""
import numpy as np
import pytest

import gpuquotientfilters_amd as G
import oracle as O
from gpu_helpers import dev, require_gpu, say, sqf_canon

pytestmark = pytest.mark.gpu
SIZES = [16385, 65536, 131072, 131073, 262145, 524289, 1048577, 256 * 7600]


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    require_gpu()


@pytest.mark.parametrize("n", SIZES)
def test_sqf_builds(n):
    q, r = max(16, int(n * 1.3).bit_length()), 5
    say("place sort, sqf", n, q)
    f = G.SQF(q, r)
    for seed in (1, 2, 3):
        k = O.mt19937(seed, n)
        f.bulk_build(dev(k), NoDuplicates=seed == 2)
        assert (f.table_bytes() == sqf_canon(k, q, r, seed == 2)).all()


@pytest.mark.parametrize("n", SIZES[:3] + SIZES[4:6])
def test_rsqf_wide_builds(n):
    q, r = 20, 13
    say("place sort, rsqf", n)
    f = G.RSQF(q, r)
    for seed in (1, 2):
        k = O.mt19937(seed, n)
        f.bulk_build(dev(k))
        st, want = O.rsqf_canon(O.fingerprints(k, q, r), q, r)
        assert st == O.OK and (f.dump() == want).all()


def test_skewed_and_uniform_keys_in_turn():
    q, r, n = 19, 5, 200001
    f = G.SQF(q, r)
    uniform = O.mt19937(9, n)
    hot = uniform.copy()
    hot[: n // 8] = uniform[0]
    small = np.arange(n, dtype=np.uint32)
    for i, k in enumerate([uniform, hot, uniform, small, uniform, uniform, uniform, uniform, uniform, hot, uniform]):
        say("place sort, turn", i)
        st, want = O.sqf_canon(O.fingerprints(k, q, r), q, r, True)
        if st != O.OK:  # (small integers crowd into clusters past the table's end)
            with pytest.raises(G.CapacityError):
                f.bulk_build(dev(k), NoDuplicates=True)
            continue
        f.bulk_build(dev(k), NoDuplicates=True)
        assert (f.table_bytes() == want).all()
