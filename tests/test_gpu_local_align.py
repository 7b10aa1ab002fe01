"""Localized SQF inserts and deletes of small batches in tables that start
off a 16-byte boundary: the localized form runs, and the table is the
canonical one."""
import numpy as np
import pytest
import torch

import gpuquotientfilters_amd as G
import oracle as O
from gpu_helpers import dev, require_gpu, say
from test_gpu_local import _kernels, delete_multiset, insert_set, sqf_equal, sqf_table

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    require_gpu()


@pytest.mark.parametrize("off", [4, 8, 12])
@pytest.mark.parametrize("q,r", [(16, 5), (13, 13), (15, 13), (20, 5)])
def test_tables_off_a_16_byte_boundary(q, r, off):
    say("local, unaligned table", q, r, off)
    st = G.Stream()
    f = G.SQF(q, r)
    own = f.h.table
    bytes_ = G.lib().gqf_sqf_table_bytes(q, r)
    guard = 64
    mem = torch.full((guard + bytes_ + guard,), 0xA5, dtype=torch.uint8, device="cuda")
    assert mem.data_ptr() % 16 == 0
    try:
        f.h.table = mem.data_ptr() + guard + off
        keys = O.mt19937(500 + q, O.key_count(0.75, q))
        f.bulk_build(dev(keys))
        fps = np.unique(O.fingerprints(keys, q, r))
        S = G.SQF.num_slots(q)
        new = O.mt19937(501 + q, S)
        for n in (1, 65, S // 200):
            names = _kernels(lambda: f.insert(dev(new[:n]), stream=st))
            assert any("k_sl_apply" in x for x in names) and not any("k_rb_write" in x for x in names)
            fps = np.unique(insert_set(fps, O.fingerprints(new[:n], q, r)))
            sqf_equal(f, sqf_table(fps, q, r))
            gone = np.concatenate([keys[:n // 2], new[:n - n // 2]])
            names = _kernels(lambda: f.superclusterDeletes(dev(gone), stream=st))
            assert any("k_sl_apply" in x for x in names) and not any("k_rb_write" in x for x in names)
            fps = delete_multiset(fps, O.fingerprints(gone, q, r))
            sqf_equal(f, sqf_table(fps, q, r))
        side = mem.cpu().numpy()
        assert (side[:guard + off] == 0xA5).all() and (side[guard + off + bytes_:] == 0xA5).all()
    finally:
        f.h.table = own
    st.destroy()
