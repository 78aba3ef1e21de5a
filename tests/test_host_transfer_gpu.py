"""Uploads and read-back through pinned staging memory, bit for bit against the
oracle: batches larger than one staging buffer in either direction, output
arrays left out, expansions that alternate between the context's stream and a
caller's, and counters read after every kind of call."""
import ctypes as C

import numpy as np
import pytest

from dynoplan_amd import _native as N
from dynoplan_amd import synth
from dynoplan_amd.expander import expander_for

import oracle_lib as O
from parity_util import assert_parity

pytestmark = pytest.mark.gpu

COUNTS = ("pairs", "bounds", "collide", "free_", "novel", "dup_visited", "dup_batch", "capped", "goal_hits", "checked")
STAGE = 8 << 20  # DP_STAGE_MAX


def workload(prims, nodes, visited=200, seed=3, obstacles=12, world=30.0):
    return synth._planar_workload("", N.SYS_UNICYCLE1, seed, prims, 5, obstacles, world, 12, nodes, visited,
                                  prim_fn=synth.unicycle1_primitives)


@pytest.mark.parametrize("prims,nodes", [(500, 6000), (4, STAGE // 32 + 1)])
def test_larger_than_the_staging_buffer(need_gpu, prims, nodes):
    w = workload(prims, nodes, world=200.0 if nodes > 100000 else 30.0)
    with expander_for(w) as ex:
        c = ex.expand(w.nodes, w.g_parent, w.params)
        gpu = ex.fetch()
        n = c["pairs"]
        assert 58 * n > (STAGE if prims > 4 else 0), "the read-back is meant to go in pieces"
        # one array alone, and a view behind a guard
        fin = np.full((n + 1, 3), 7.0)
        po = N.PairsOut()
        po.capacity, po.final_state = n, fin.ctypes.data_as(C.POINTER(C.c_double))
        N.check(ex.lib.dp_fetch_pairs(ex.ctx, C.byref(po)))
        res = np.full(n + 1, 99, np.int8)
        po = N.PairsOut()
        po.capacity, po.resolution = n, res.ctypes.data_as(C.POINTER(C.c_int8))
        N.check(ex.lib.dp_fetch_pairs(ex.ctx, C.byref(po)))
    ora, co = O.expand(w)
    assert_parity(gpu, ora, "staged")
    assert {k: c[k] for k in COUNTS} == {k: co[k] for k in COUNTS}
    assert np.array_equal(fin[:n], gpu["final_state"], equal_nan=True) and (fin[n] == 7.0).all()
    assert np.array_equal(res[:n], gpu["resolution"]) and res[n] == 99


def test_streams_in_turn(need_gpu):
    import torch

    w = [workload(300, 40, seed=3), workload(300, 40, seed=3)]
    w[1]["nodes"] = np.ascontiguousarray(w[0].nodes[::-1] + 0.01)
    ora = [O.expand(x) for x in w]
    side = torch.cuda.Stream()
    with expander_for(w[0]) as ex:
        for turn in range(6):
            x, (want, cw) = w[turn % 2], ora[turn % 2]
            if turn in (0, 1, 5):
                c = ex.expand(x.nodes, x.g_parent, w[0].params)
            else:
                ex.upload_nodes(x.nodes, x.g_parent)
                ex.expand_async(w[0].params, side.cuda_stream if turn in (2, 4) else None)
                c = ex.counts()
            assert_parity(ex.fetch(), want, f"turn {turn}")
            assert {k: c[k] for k in COUNTS} == {k: cw[k] for k in COUNTS}, turn
