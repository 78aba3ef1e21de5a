"""Duplicate test against more visited states in one 27-cell block than the
planar check numbers together for a wave, with pairs of few candidates beside
those, against the oracle."""
import copy

import numpy as np
import pytest

from dynoplan_amd import _native as N
from dynoplan_amd import synth
from dynoplan_amd.expander import expander_for

import oracle_lib as O
from parity_util import assert_parity

pytestmark = pytest.mark.gpu

LIMIT = 1 << 20  # candidates of one pair past which a wave takes its pairs singly


@pytest.mark.parametrize("states", [LIMIT, LIMIT + 1, 1500000])
def test_crowded_block(need_gpu, states):
    w = synth._planar_workload("", N.SYS_UNICYCLE1, 61, 200, 5, 20, 10.0, 0, 6, 0, prim_fn=synth.unicycle1_primitives)
    p = copy.copy(w.params)
    p.delta, p.alpha = 2.0, 0.5  # radius 1: cells of 1 m
    rng = np.random.default_rng(states)
    # one small cluster: near every node's block, within the radius of some
    # final states and not of others; one node far from it
    v = np.empty((states, 3))
    v[:, 0:2] = [5.05, 5.05] + rng.uniform(0.0, 0.1, (states, 2))
    v[:, 2] = rng.uniform(-0.05, 0.05, states)
    w["visited"] = v
    nodes = np.array([[5.8, 5.1, 0.0], [4.2, 5.2, 0.3], [5.0, 6.1, -0.4], [5.9, 5.9, 0.1], [1.0, 1.0, 0.0],
                      [4.3, 4.1, 0.2]])
    w["nodes"] = nodes
    with expander_for(w) as ex:
        c = ex.expand(nodes, w.g_parent, p)
        gpu = ex.fetch()
    ora, co = O.expand(w, nodes=nodes, g_parent=w.g_parent, params=p)
    print(c)
    assert_parity(gpu, ora, f"{states} states in one block")
    dup = (gpu["resolution"] == N.R_DUP_VISITED).sum()
    assert dup > 0 and (gpu["resolution"] == N.R_NOVEL).sum() > 0
