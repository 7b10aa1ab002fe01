"""RSQF inserts whose answers go over their keys (d_out is d_keys): the slots
are those of the keys, whichever form the batch ends up in -- the localized
one, the windows, or the rebuild."""
import numpy as np
import pytest

import gpuquotientfilters_amd as G
import oracle as O
from gpu_helpers import dev, require_gpu, say
from test_gpu_local import _kernels, rsqf_equal, rsqf_table

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    require_gpu()


@pytest.mark.parametrize("form,copies,n", [("k_rl_apply", 3, 500), ("k_wm_write", 300, 500), ("k_rr_write", 9000, 9500)])
@pytest.mark.parametrize("q,r", [(16, 8), (18, 16), (16, 5)])
def test_answers_over_the_keys(form, copies, n, q, r):
    say("insert in place", form, copies, q, r)
    st = G.Stream()
    stored = O.mt19937(400 + q, O.key_count(0.6, q))
    f = G.RSQF(q, r)
    f.bulk_build(dev(stored))
    batch = O.mt19937(401 + q, n)
    batch[:copies] = stored[np.argmin(O.fingerprints(stored, q, r))]  # (room after it for every copy)
    batch = np.random.default_rng(1).permutation(batch)
    d = dev(batch)
    names = _kernels(lambda: f.insert(d, d, stream=st))
    assert any(form in k for k in names), names
    assert form != "k_rl_apply" or not any("k_wm_write" in k for k in names)
    want = rsqf_table(np.concatenate([O.fingerprints(stored, q, r), O.fingerprints(batch, q, r)]), q, r)
    rsqf_equal(f, want)
    assert (d.to_host() == O.rsqf_lookup_keys(want, q, r, batch)).all()
    st.destroy()
