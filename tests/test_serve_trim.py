"""The serving scheduler (gqf_serve_run) with executors whose trim leaves
bytes held: every run ends, and what cannot fit is rejected.  Each run is a
process of its own with a time limit (a scheduler that asks for the same
release again and again never returns).  No GPU."""
import subprocess
import sys

import pytest

from conftest import ROOT

RUN = """
import ctypes as C, sys
sys.path.insert(0, {root!r})
import gpuquotientfilters_amd as G

workers, coalesce, begin, keep, sizes, budget = {args!r}
held = [begin] * workers
reqs = (G.Request * len(sizes))()
for i, (f, n) in enumerate(sizes):
    reqs[i].filter, reqs[i].op, reqs[i].n, reqs[i].d_keys, reqs[i].d_out = f, G.OP_LOOKUP, n, 0x1000, 0x1000
trims = [0] * workers
def grow(u, w, f, op, n, c): return max(0, n - held[w])
def hold(u, w): return held[w]
def trim(u, w):
    trims[w] += 1
    held[w] = min(held[w], keep)
def run(u, w, b, nb):
    held[w] = max(held[w], sum(b[i].contents.n for i in range(nb)))
    return G.OK
ex = G.ServeExecutor(None, G.GROW_FN(grow), G.HELD_FN(hold), G.TRIM_FN(trim), G.RUN_FN(run))
cfg = G.ServeConfig(budget, coalesce, 0, 0)
st = G.ServeStats()
n = max(f for f, _ in sizes) + 1
assert G.lib().gqf_serve_run(n, 0, reqs, len(sizes), C.byref(cfg), C.byref(ex), C.byref(st)) == G.OK
print("statuses", *[r.status for r in reqs], "trims", max(trims))
"""


def go(*args):
    p = subprocess.run([sys.executable, "-c", RUN.format(root=ROOT, args=args)], capture_output=True, text=True,
                       timeout=30)
    assert p.returncode == 0, p.stderr[-2000:]
    return p.stdout


@pytest.mark.parametrize("begin,keep", [(100, 100), (600, 100), (600, 599), (0, 0)])
def test_own_holdings_that_stay(begin, keep):
    """One worker: the second request can never fit and is rejected."""
    out = go(1, 0, begin, keep, [(0, 500), (0, 2000), (0, 400)], 1000)
    words = out.split()
    assert words[1] == "0" and words[2] != "0" and words[3] == "0"
    assert int(words[words.index("trims") + 1]) <= 4


def test_other_workers_holdings_that_stay():
    """Two workers with more than half of the budget each left after a trim:
    the one that comes second is rejected or served, and the run ends."""
    out = go(2, 1, 0, 450, [(0, 500), (1, 700), (1, 300), (0, 500)], 960)
    words = out.split()
    assert words[1] == "0" and words[4] == "0"
    assert int(words[words.index("trims") + 1]) <= 8
