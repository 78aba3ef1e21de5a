"""Allocation-free radius query after NOVEL states were appended and a small
batch was expanded, which leaves them unsorted behind the grid: both entry
points against the oracle, over a tail that grows and a rebuild in between."""
import ctypes as C

import numpy as np
import pytest

from dynoplan_amd import _native as N
from dynoplan_amd import synth
from dynoplan_amd.expander import expander_for

import oracle_lib as O

pytestmark = pytest.mark.gpu


def noalloc(ex, q, r, cap):
    import torch
    n = q.shape[0]
    qd = torch.from_numpy(q).cuda()
    od = torch.full((n + 1,), -7, dtype=torch.int64, device="cuda")
    xd = torch.full((cap,), -7, dtype=torch.int64, device="cuda")
    torch.cuda.synchronize()
    rc = ex.lib.dp_visited_radius_noalloc(ex.ctx, C.c_void_p(qd.data_ptr()), n, float(r), C.c_void_p(od.data_ptr()),
                                          C.c_void_p(xd.data_ptr()), cap, None)
    torch.cuda.synchronize()
    return rc, od.cpu().numpy(), xd.cpu().numpy()


@pytest.mark.parametrize("system", [N.SYS_UNICYCLE1, N.SYS_CAR_TRAILER, N.SYS_QUADROTOR])
def test_appended_states_are_found(need_gpu, system):
    if system == N.SYS_QUADROTOR:
        w = synth.quadrotor(seed=21, P=800, N_nodes=40, n_visited=300, thrust="balanced")
    else:
        fn = {N.SYS_UNICYCLE1: synth.unicycle1_primitives, N.SYS_CAR_TRAILER: synth.car_trailer_primitives}[system]
        w = synth._planar_workload("", system, 21, 800, 5, 20, 8.0, 12, 40, 300, prim_fn=fn)
    r = (1.0 - float(np.float32(w.params.alpha))) * float(np.float32(w.params.delta))
    vis = w.visited
    found = 0
    with expander_for(w) as ex:
        for step in range(10):
            n = w.nodes.shape[0] if step == 6 else 1 + step % 2  # 40 nodes: the grid is built again
            nodes, g = w.nodes[2 * step:][:n] if step != 6 else w.nodes, w.g_parent[:n]
            ex.expand(nodes, g, w.params)
            q = np.ascontiguousarray(np.concatenate([vis[-100:], vis[:50], nodes]))
            want_off, want = O.radius(w.desc, vis, q, r)
            cap = int(want_off[-1]) + 3
            rc, off, idx = noalloc(ex, q, r, cap)
            assert rc == N.DP_OK, (step, ex.lib.dp_last_error())
            assert np.array_equal(off, want_off), step
            assert np.array_equal(idx[: off[-1]], want) and (idx[off[-1]:] == -7).all(), step
            found += int((want >= w.visited.shape[0]).sum())
            if step == 4:
                o2, i2 = ex.visited_radius(q, r)
                assert np.array_equal(o2, want_off) and np.array_equal(i2, want)
            out = ex.fetch()
            ex.visited_append_novel()
            novel = out["final_state"][out["resolution"] == N.R_NOVEL]
            vis = np.concatenate([vis, novel])
            if novel.shape[0]:  # refused until the next expansion or query
                assert noalloc(ex, q, r, cap)[0] == N.DP_ERR_STATE
    assert found > 0
