"""dbrrt's choice among more pairs than one chunk of a node's waves, with equal
distances (repeated primitives), and batches whose (node, primitive)
combinations are counted before their arrays are sized, against the oracle."""
import numpy as np
import pytest

from dynoplan_amd import _native as N
from dynoplan_amd import synth
from dynoplan_amd.expander import expander_for

import oracle_lib as O
from parity_util import assert_parity
from test_adopters_gpu import assert_select

pytestmark = pytest.mark.gpu


def workload(nodes, prims, repeat=1):
    w = synth._planar_workload("", N.SYS_UNICYCLE1, 5 + nodes, prims // repeat, 5, 12, 20.0, 40, nodes, 50,
                               prim_fn=synth.unicycle1_primitives)
    if repeat > 1:
        S = w.offsets[-1]
        w["offsets"] = np.concatenate([[0]] + [w.offsets[1:] + k * S for k in range(repeat)]).astype(w.offsets.dtype)
        w["states"] = np.concatenate([w.states] * repeat)
        w["actions"] = np.concatenate([w.actions] * repeat)
    return w


@pytest.mark.parametrize("nodes,prims,repeat", [(1, 30, 1), (3, 640, 1), (7, 5000, 1), (5, 6000, 3), (900, 5000, 1)])
@pytest.mark.parametrize("choose_first", [False, True])
def test_select(need_gpu, nodes, prims, repeat, choose_first):
    w = workload(nodes, prims, repeat)
    rng = np.random.default_rng(prims)
    targets = w.nodes + rng.normal(0, 1.5, w.nodes.shape)
    goal = w.params.goal[:3]
    with expander_for(w) as ex:
        for _ in range(2):  # sizes counted anew, then within the arrays of the first
            got = ex.expand_select(w.nodes, w.g_parent, targets, 0.3, goal, choose_first=choose_first)
            pairs = ex.counts()["pairs"]
        ex.expand(w.nodes, w.g_parent, w.params)
        after = ex.fetch()
    ora, n = O.select(w, w.nodes, w.g_parent, targets, 0.3, goal, choose_first=choose_first)
    print(f"{pairs} pairs of {nodes} nodes")
    assert pairs == n
    assert_select(got, ora, f"{nodes} nodes")
    ref, _ = O.expand(w)
    assert_parity(after, ref, "expansion after a selection")
