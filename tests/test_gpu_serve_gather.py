"""Coalesced lookups of many requests (more than one launch of the gather
takes; empty, tiny and tile-sized ones) against a lookup of each, and result
buffers that overlap: the later request's results stand."""
import numpy as np
import pytest

import gpuquotientfilters_amd as G
import oracle as O
from gpu_helpers import dev, require_gpu, rsqf_lookup, say

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    require_gpu()


@pytest.mark.parametrize("overlap", [False, True])
def test_coalesced_lookups_gather_and_scatter(overlap):
    say("serve gather", overlap)
    q, r = 14, 8
    keys = O.mt19937(900, O.key_count(0.7, q))
    f = G.RSQF(q, r)
    f.bulk_build(dev(keys))
    sizes = [0, 1, 63, 1023, 1024, 1025, 4096, 17, 0, 2048] * 45
    starts = np.concatenate([[0], np.cumsum(sizes)])
    n = int(starts[-1])
    probe = O.mt19937(901, n)
    probe[::3] = np.resize(keys, len(probe[::3]))
    want = rsqf_lookup(f, probe)
    d, out = dev(probe), dev(np.full(n, 7, np.uint32))
    reqs = (G.Request * len(sizes))()
    for i, k in enumerate(sizes):
        x = reqs[i]
        x.filter, x.op, x.n, x.arrive_us = 0, G.OP_LOOKUP, k, 0.0
        x.d_keys = d.ptr + 4 * int(starts[i])
        x.d_out = out.ptr + (0 if overlap else 4 * int(starts[i]))
    st = G.serve([f], reqs)
    assert all(x.status == 0 for x in reqs) and st.calls < len(sizes) // 4
    got = out.to_host().view(want.dtype)
    if overlap:  # the last request's results, and where it does not reach those of the last longer one
        end = np.zeros(0, want.dtype)
        for i, k in enumerate(sizes):
            end = np.concatenate([want[starts[i]:starts[i + 1]], end[k:]])
        assert (got[:len(end)] == end).all() and (got[len(end):] == 7).all()
    else:
        assert (got == want).all()
