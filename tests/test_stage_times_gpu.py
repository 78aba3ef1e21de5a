"""Stage times of an expansion that the host completes afterwards (a quadrotor
node past its FP64 window): they are the expansion's own, before and after."""
import copy

import numpy as np
import pytest

from dynoplan_amd import synth
from dynoplan_amd.expander import expander_for

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nodes", [1, 6])  # resolved by one workgroup; by the general path
def test_completed_batch_keeps_its_stage_times(need_gpu, nodes):
    # duplicates of the visited set all around the nodes: no cap in the window
    w = synth.quadrotor(seed=5, P=4000, N_nodes=nodes, n_visited=30000, thrust="balanced")
    rng = np.random.default_rng(0)
    v = np.repeat(w.nodes, 30000, axis=0)
    v[:, 0:3] += rng.normal(0.0, 0.15, (v.shape[0], 3))
    v[:, 3:7] = synth.random_attitudes(rng, v.shape[0])
    v[:, 7:10] += rng.normal(0.0, 0.5, (v.shape[0], 3))
    v[:, 10:13] = rng.normal(0.0, 0.7, (v.shape[0], 3))
    w["visited"] = np.ascontiguousarray(v)
    p = copy.copy(w.params)
    p.limit_branching_factor, p.delta = 20, 1.2
    with expander_for(w) as ex:
        ex.upload_nodes(w.nodes, w.g_parent)
        ex.expand_async(p)
        before = ex.timing(), ex.timing_detail()
        assert ex.counts()["fp64_deferred"] > 0
        assert ex.health()["host_completions"] == 1
        after = ex.timing(), ex.timing_detail()
    print(after)
    assert after == before
    # a total from events, the stages from a 10 ns clock
    for part in after:
        assert all(t >= -1e-4 for t in part.values()), part
