"""Large lookup batches by groups of quotients (gqf_plookup.hpp): the answers
of the whole batch equal those of the same keys in small batches (the direct
walk), and the oracle's on a part of them."""
import numpy as np
import pytest
import torch

import gpuquotientfilters_amd as G
import oracle as O
from gpu_helpers import require_gpu, say

pytestmark = pytest.mark.gpu
N = 1 << 23  # at least the smallest batch that goes by groups


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    require_gpu()


def keys_of(gen, n):
    return torch.randint(-(1 << 31), 1 << 31, (n,), dtype=torch.int32, device="cuda", generator=gen)


def check(f, probe, part=1 << 19, in_place=False):
    n = len(probe)
    want = torch.full((n,), 7, dtype=torch.int32, device="cuda")
    for a in range(0, n, part):
        b = min(n, a + part)
        f.lookup(probe[a:b], want[a:b])
    got = probe if in_place else torch.full((n,), 7, dtype=torch.int32, device="cuda")
    f.lookup(probe, got)
    assert torch.equal(got, want)
    return want


# quotients of one group and of several sizes of it, both ends of the table;
# fills from sparse to clusters and runs longer than what a group loads beside
# its own slots (q = 20: groups of 2^12 quotients)
@pytest.mark.parametrize("kind,q,r,fill,n", [
    ("sqf", 22, 5, 0.75, N), ("sqf", 22, 5, 0.97, N + 5), ("sqf", 24, 5, 0.3, N + 1), ("sqf", 26, 5, 0.8, N + 4096 * 3 + 2),
    ("sqf", 24, 5, 0.93, N + 32767), ("sqf", 20, 5, 0.7, N // 2 + 3), ("rsqf", 24, 8, 0.9, N), ("rsqf", 24, 8, 0.98, N + 3), ("rsqf", 26, 8, 0.9, N + 7),
    ("rsqf", 25, 5, 0.8, N + 1), ("rsqf", 24, 1, 0.5, N), ("rsqf", 25, 7, 0.97, N + 2), ("rsqf", 26, 6, 0.6, 2 * N + 1),
])
def test_equals_the_direct_walk(kind, q, r, fill, n):
    say("large lookup", kind, q, r, fill, n)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(q * 100 + r)
    f = (G.SQF if kind == "sqf" else G.RSQF)(q, r)
    stored = keys_of(gen, int(fill * (1 << q)))
    f.bulk_build(stored)
    probe = torch.where(torch.rand(n, device="cuda", generator=gen) < 0.5,
                        stored[torch.randint(0, len(stored), (n,), device="cuda", generator=gen)], keys_of(gen, n))
    want = check(f, probe)
    if kind == "sqf" and q <= 24 and fill < 0.9:  # (the oracle walks long clusters slot by slot)
        part = probe[-20000:].cpu().numpy().view(np.uint32)
        t = f.table_bytes()
        assert (want[-20000:].cpu().numpy().view(np.uint32) == O.sqf_lookup_keys(t, q, r, part)).all()


@pytest.mark.parametrize("kind,q,r", [("sqf", 24, 5), ("rsqf", 26, 8)])
def test_hot_keys_and_in_place(kind, q, r):
    """A group without room for its keys (every other key the same one), twice
    in a row; and answers written over the keys."""
    say("large lookup, hot keys", kind, q, r)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(3)
    f = (G.SQF if kind == "sqf" else G.RSQF)(q, r)
    stored = keys_of(gen, int(0.7 * (1 << q)))
    f.bulk_build(stored)
    check(f, torch.cat([stored[:N], stored[:1]]).clone(), in_place=True)
    probe = stored[torch.randint(0, len(stored), (N,), device="cuda", generator=gen)]
    probe[::2] = stored[5]
    check(f, probe)
    check(f, probe, in_place=True)
