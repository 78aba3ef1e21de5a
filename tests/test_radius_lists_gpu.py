"""Radius query at the edges of its passes: lists around the 64 entries that a
wave sorts itself, query counts around the 4096 of one scan step, a capacity
that cuts a list, both entry points, against the oracle."""
import ctypes as C

import numpy as np
import pytest

from dynoplan_amd import _native as N
from dynoplan_amd import synth
from dynoplan_amd.expander import expander_for

import oracle_lib as O

pytestmark = pytest.mark.gpu

LENGTHS = (0, 1, 2, 3, 4, 5, 31, 32, 33, 63, 64, 65, 66, 128, 500)


@pytest.mark.parametrize("queries,longest", [(1, 64), (1, 500), (15, 64), (15, 500), (4095, 64), (4096, 5), (4097, 65),
                                             (9000, 33)])
def test_lists(need_gpu, queries, longest):
    import torch

    w = synth.unicycle1_small(seed=41)
    rng = np.random.default_rng(queries + longest)
    lengths = [n for n in LENGTHS if n <= longest]
    centre = np.stack([0.5 + 0.6 * np.arange(len(lengths)), np.full(len(lengths), 1.0), np.zeros(len(lengths))], 1)
    vis = np.concatenate([c + np.concatenate([rng.normal(0, 0.01, (n, 2)), np.zeros((n, 1))], 1)
                          for c, n in zip(centre, lengths)])
    w["visited"] = np.ascontiguousarray(vis[rng.permutation(vis.shape[0])])
    q = np.ascontiguousarray(centre[(np.arange(queries) + len(lengths) - 1) % len(lengths)])
    r = 0.2
    want_off, want = O.radius(w.desc, w.visited, q, r)
    assert np.diff(want_off).max() == longest
    with expander_for(w) as ex:
        off, idx = ex.visited_radius(q, r)
        assert np.array_equal(off, want_off) and np.array_equal(idx, want)
        qd = torch.from_numpy(q).cuda()
        od = torch.zeros(queries + 1, dtype=torch.int64, device="cuda")
        total = int(want_off[-1])
        for cap in (total, total + 7, total - 1):
            xd = torch.full((total + 8,), -1, dtype=torch.int64, device="cuda")
            torch.cuda.synchronize()
            rc = ex.lib.dp_visited_radius_noalloc(ex.ctx, C.c_void_p(qd.data_ptr()), queries, r,
                                                  C.c_void_p(od.data_ptr()), C.c_void_p(xd.data_ptr()), cap, None)
            torch.cuda.synchronize()
            got = xd.cpu().numpy()
            assert np.array_equal(od.cpu().numpy(), want_off)
            assert (got[cap:] == -1).all()
            assert rc == (N.DP_OK if cap >= total else N.DP_ERR_CAPACITY)
            # every list that lies below the capacity is whole and ascending
            whole = want_off[np.searchsorted(want_off, min(cap, total), side="right") - 1]
            assert np.array_equal(got[:whole], want[:whole])
