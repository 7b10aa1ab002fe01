"""Batches refilled in place with keys unlike those they were tuned on: a
batch that sorts groups in LDS hands builds with crowded digits over to the
8-bit passes, keeps to them for a few builds, and comes back; the tables are
the oracle's throughout, by graph and launch by launch."""
import numpy as np
import pytest
import torch

import gpuquotientfilters_amd as G
import oracle as O
from gpu_helpers import require_gpu, say
from test_gpu_local import _kernels

pytestmark = pytest.mark.gpu

QS = [19, 20, 18, 12, 20, 19, 17, 20]


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    require_gpu()


def fill(kind, n, seed):
    k = O.mt19937(seed, n)
    rng = np.random.default_rng(seed)
    if kind == "hot":
        k[:] = k[0]
    elif kind == "half":
        k[rng.random(n) < 0.5] = k[0]
    elif kind == "few":  # crowded buckets, no group past what LDS holds
        hot = k[:400]
        at = rng.random(n) < 0.3
        k[at] = hot[rng.integers(0, 400, at.sum())]
    return k


@pytest.mark.parametrize("no_dup", [True, False])
def test_refilled_batches(no_dup):
    sizes = [int(0.35 * (1 << q)) + 3 for q in QS]
    off = np.concatenate([[0], np.cumsum(sizes)]).tolist()
    d = torch.empty(off[-1], dtype=torch.int32, device="cuda")
    fs = [G.SQF(q, 5) for q in QS]

    def load(kinds, seed):
        ks = [fill(k, n, 100 * seed + i) for i, (k, n) in enumerate(zip(kinds, sizes))]
        d.copy_(torch.from_numpy(np.concatenate(ks).view(np.int32)))
        torch.cuda.synchronize()
        return ks

    def check(b, ks, use_graph):
        st = b.build(use_graph=use_graph)[1]
        for f, q, k, s in zip(fs, QS, ks, st):
            ok, t = O.sqf_canon(O.fingerprints(k, q, 5), q, 5, no_dup)
            assert (s == G.OK) == (ok == O.OK)
            if ok == O.OK:
                assert (f.table_bytes() == t).all()

    uniform = ["uni"] * len(QS)
    load(uniform, 0)
    b = G.SQFBatch(fs, d, off, no_dup=no_dup)
    ks = load(uniform, 1)
    names = _kernels(lambda: check(b, ks, False))
    assert any("k_bs_groups" in x for x in names) and not any("k_bs_upsweep<false>" in x for x in names)
    say("batch refill, crowded buckets", no_dup)
    ks = load(["few"] * len(QS), 2)
    names = _kernels(lambda: check(b, ks, False))
    assert not any("k_bs_upsweep<false>" in x for x in names)
    check(b, ks, True)
    kinds = ["half" if no_dup or q == 12 else "uni" for q in QS]  # (copies past the slots behind them do not fit)
    kinds[1] = "hot" if no_dup else "half"
    say("batch refill, crowded digits", no_dup)
    ks = load(kinds, 3)
    names = _kernels(lambda: check(b, ks, False))
    assert any("k_bs_groups" in x for x in names) and any("k_bs_upsweep<false>" in x for x in names)
    names = _kernels(lambda: check(b, ks, False))
    assert not any("k_bs_groups" in x for x in names) and any("k_bs_upsweep<false>" in x for x in names)
    for i in range(8):  # graphs: the passes, the groups again, handed over, the passes
        say("batch refill, graph", i)
        if i == 4:
            ks = load(kinds, 4)
        check(b, ks, True)
    ks = load(uniform, 5)
    for i in range(12):
        check(b, ks, i % 3 != 0)
    names = _kernels(lambda: check(b, ks, False))
    assert any("k_bs_groups" in x for x in names) and not any("k_bs_upsweep<false>" in x for x in names)
    b.destroy()
