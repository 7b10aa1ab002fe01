"""Large lookup batches on streams of their own, so that no earlier call of the
process decides the form: the groups are really taken where they are meant to
be, keys crowded into one group and tables whose walks are long go to the
direct walk from the next call on, and every answer is the direct walk's."""
import pytest
import torch

import gpuquotientfilters_amd as G
from gpu_helpers import require_gpu, say
from test_gpu_local import _kernels
from test_gpu_plookup import keys_of

pytestmark = pytest.mark.gpu
N = 1 << 22


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    require_gpu()


@pytest.fixture
def stream():
    s = G.Stream()
    yield s
    s.destroy()


def direct(f, probe, part=1 << 19):
    want = torch.empty_like(probe)
    for a in range(0, len(probe), part):
        f.lookup(probe[a:a + part], want[a:a + part])
    return want


def by_groups(f, probe, want, stream, in_place=False):
    """Whether the call goes by groups; its answers are `want`."""
    got = probe if in_place else torch.full_like(probe, 7)
    torch.cuda.synchronize()
    names = _kernels(lambda: f.lookup(probe, got, stream=stream))
    G.synchronize()
    torch.cuda.synchronize()
    assert torch.equal(got, want)
    groups = any("k_pl_gather" in x for x in names)
    assert groups != any("lookup" in x for x in names)
    return groups


def filled(kind, q, r, fill, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    f = (G.SQF if kind == "sqf" else G.RSQF)(q, r)
    stored = keys_of(gen, int(fill * (1 << q)))
    f.bulk_build(stored)
    probe = torch.where(torch.rand(N, device="cuda", generator=gen) < 0.5,
                        stored[torch.randint(0, len(stored), (N,), device="cuda", generator=gen)], keys_of(gen, N))
    return f, stored, probe


# fills up to those where the groups are the faster form, and past them
@pytest.mark.parametrize("kind,q,r,fill,stays", [
    ("sqf", 20, 5, 0.5, True), ("sqf", 20, 5, 0.85, True), ("sqf", 20, 5, 0.95, False), ("sqf", 20, 5, 1.0, False),
    ("sqf", 21, 5, 0.96, False), ("sqf", 22, 5, 0.8, True), ("sqf", 22, 5, 0.96, False), ("sqf", 24, 5, 0.9, True),
    ("sqf", 24, 5, 1.0, False), ("sqf", 26, 5, 0.9, True), ("rsqf", 24, 8, 0.9, True), ("rsqf", 25, 6, 0.95, True),
])
def test_form_by_fill(stream, kind, q, r, fill, stays):
    say("large lookup, form", kind, q, r, fill)
    f, _, probe = filled(kind, q, r, fill, q + r)
    want = direct(f, probe)
    assert by_groups(f, probe, want, stream)
    assert by_groups(f, probe, want, stream) == stays


@pytest.mark.parametrize("kind,q,r", [("sqf", 24, 5), ("rsqf", 26, 8)])
@pytest.mark.parametrize("in_place", [False, True])
def test_one_crowded_group(stream, kind, q, r, in_place):
    """Every other key the same one: its group has no room for them, the rest
    of the batch still goes by groups; in place, the keys left to walk for are
    not yet written over."""
    say("large lookup, crowded group", kind, q, r, in_place)
    f, stored, probe = filled(kind, q, r, 0.7, 5)
    probe[::2] = stored[9]
    want = direct(f, probe)
    assert by_groups(f, probe.clone(), want, stream, in_place)
    assert not by_groups(f, probe.clone(), want, stream, in_place)


@pytest.mark.parametrize("kind,q,r", [("sqf", 24, 5), ("rsqf", 26, 8)])
def test_in_place(stream, kind, q, r):
    say("large lookup, in place", kind, q, r)
    f, _, probe = filled(kind, q, r, 0.7, 6)
    want = direct(f, probe)
    assert by_groups(f, probe, want, stream, True)
