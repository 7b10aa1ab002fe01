"""The one-workgroup sort where many of its keys are alike: sizes around the
powers of two and the largest that the network takes, all keys alike, a few
different ones, and the time beside that of different keys."""
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


@pytest.mark.parametrize("n", [33, 34, 63, 64, 65, 100, 511, 1023, 1024, 1025, 2047, 2049, 4095, 4096, 4097, 9000])
@pytest.mark.parametrize("q,r", [(15, 5), (19, 13)])
def test_crowded_keys(q, r, n):
    say("one-workgroup sort, crowded", q, r, n)
    for distinct in (1, 3, n // 2):
        keys = O.mt19937(810 + n, n)
        keys[:n - n // 4] = keys[np.arange(n - n // 4) % distinct]
        keys = keys[np.random.default_rng(n).permutation(n)]
        f = G.SQF(q, r)
        names = _kernels(lambda: f.bulk_build(dev(keys), NoDuplicates=True))
        assert any("k_rs_one" in x for x in names)
        sqf_equal(f, sqf_table(O.fingerprints(keys, q, r), q, r, True))


def test_crowded_keys_time():
    """Up to three times the time of different keys (five, by counting passes)."""
    q, r, n = 16, 5, 256
    f = G.SQF(q, r)

    def ms(keys):
        d = dev(keys)
        best = 1e9
        for _ in range(6):
            f.bulk_build(d, NoDuplicates=True)
            G.profile_reset()
            G.profile_enable(True)
            f.bulk_build(d, NoDuplicates=True)
            G.synchronize()
            G.profile_enable(False)
            best = min(best, sum(v[1] for k, v in G.profile_stats().items() if "k_rs_one" in k))
        G.profile_reset()
        return best

    different, alike = ms(O.mt19937(820, n)), ms(np.full(n, 12345, np.uint32))
    say("one-workgroup sort, different, alike", different, alike)
    assert alike < 3 * different
