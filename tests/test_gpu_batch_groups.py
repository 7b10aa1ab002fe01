"""Batched builds by one top-digit pass and LDS group sorts: group sizes around
what LDS holds, filters whose keys crowd one digit (sorted by k_bs_big), and
replays of one graph over changed keys, against the oracle's tables."""
import numpy as np
import pytest
import torch

import gpuquotientfilters_amd as G
import oracle as O
from gpu_helpers import dev, require_gpu, say, sqf_canon

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    require_gpu()


def crowded(n, seed):
    """n keys, seven eighths of them copies of 50 keys whose fingerprints share a digit."""
    k = O.mt19937(seed, 4 * n + 60000)
    fp = O.fingerprints(k, 18, 5) >> 15
    few = k[fp == 200][:50]
    out = k[:n].copy()
    out[n // 8:] = few[np.arange(n - n // 8) % len(few)]
    return out


@pytest.mark.parametrize("r", [5, 13])
def test_group_sizes_and_crowded_digits(r):
    q = 18
    sizes = [0, 1, 2, 4095, 4096, 4097, 8192, 8193, 65537, 180001]
    qs = [q] * len(sizes) + [q, q, 11]
    seeds = range(1, 4)
    mk = lambda s: [O.mt19937(10 * s + i, n) for i, n in enumerate(sizes)] + [
        crowded(20001, s) if s != 2 else O.mt19937(77, 20001), crowded(150000, s + 5), O.mt19937(s + 50, 1200)]
    sets = [mk(s) for s in seeds]
    off = [0]
    for k in sets[0]:
        off.append(off[-1] + len(k))
    d = torch.empty(off[-1], dtype=torch.int32, device="cuda")
    load = lambda ks: d.copy_(torch.from_numpy(np.concatenate(ks).view(np.int32)))
    load([O.mt19937(90 + i, len(k)) for i, k in enumerate(sets[0])])  # (the autotuner sees uniform keys)
    torch.cuda.synchronize()
    fs = [G.SQF(x, r) for x in qs]
    say("batch groups", r, off[-1])
    b = G.SQFBatch(fs, d, off, no_dup=True)
    for s, ks in enumerate(sets + sets[:1]):  # graph replays, eager work between
        say("batch groups, replay", s)
        load(ks)
        torch.cuda.synchronize()
        _, st = b.build(use_graph=s != 1)
        assert st == [G.OK] * len(fs)
        for f, x, k in zip(fs, qs, ks):
            assert (f.table_bytes() == sqf_canon(k, x, r, True)).all()
    b.destroy()
