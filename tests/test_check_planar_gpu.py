"""The planar check kernel at the edges of its flattened lists, bit for bit
against the oracle: more than 64 obstacles near a node (several mask chunks),
more than 4096 items per wave (several windows), primitives of one state,
empty worlds and visited sets, every pairs-per-wave split."""
import numpy as np
import pytest

from dynoplan_amd import _native as N
from dynoplan_amd import synth
from dynoplan_amd.expander import expander_for

import oracle_lib as O
from parity_util import assert_parity, counts_consistent

pytestmark = pytest.mark.gpu

UNI1, UNI2, CAR = N.SYS_UNICYCLE1, N.SYS_UNICYCLE2, N.SYS_CAR_TRAILER
PRIMS = {UNI1: synth.unicycle1_primitives, UNI2: synth.unicycle2_primitives, CAR: synth.car_trailer_primitives}


def small_boxes(w, n, half, seed):
    rng = np.random.default_rng(seed)
    b = np.zeros((n, 6))
    b[:, 0] = rng.uniform(w.lo[0], w.hi[0], n)
    b[:, 1] = rng.uniform(w.lo[1], w.hi[1], n)
    b[:, 3:5] = half
    return b


@pytest.mark.parametrize("system,prims,lmin,lmax,nodes,boxes,visited,lanes", [
    (UNI1, 300, 100, 140, 20, 900, 50, 0),     # 15 mask chunks, two item windows
    (CAR, 300, 90, 130, 20, 1024, 50, 2),      # the obstacle limit, trailer boxes
    (UNI1, 500, 1, 3, 40, 70, 120000, 0),      # short primitives, over 4096 visited candidates per wave
    (UNI2, 777, 1, 20, 33, 0, 0, 64),          # nothing to test against, one pair per wave
    (UNI2, 65, 5, 20, 1, 20, 3000, 8),         # one node, a ragged last wave
    (CAR, 1000, 10, 40, 3, 40, 1, 0),
])
def test_flattened_lists(need_gpu, system, prims, lmin, lmax, nodes, boxes, visited, lanes):
    w = synth._planar_workload("", system, 5 + prims, prims, lmin, lmax, 6.0, 3, nodes, visited,
                               prim_fn=PRIMS[system])
    w["boxes"] = small_boxes(w, boxes, 0.02, prims)
    if lmin == 1:
        # primitives of a single state: the placed start alone
        keep = np.diff(w.offsets) > 0
        off, st, ac = [0], [], []
        for j in np.flatnonzero(keep):
            a, b = w.offsets[j], w.offsets[j + 1]
            n = 1 if j % 3 == 0 else b - a
            st.append(w.states[a:a + n])
            ac.append(w.actions[a - j:a - j + n - 1])
            off.append(off[-1] + n)
        w["offsets"], w["states"], w["actions"] = np.array(off, np.int32), np.concatenate(st), np.concatenate(ac)
    with expander_for(w) as ex:
        ex.set_tiles(lanes_per_pair=lanes)
        counts = ex.expand(w.nodes, w.g_parent, w.params)
        gpu = ex.fetch()
    ora, co = O.expand(w)
    assert_parity(gpu, ora, "flattened lists")
    counts_consistent(counts)
    assert counts["pairs"] == co["pairs"] > 0
    if boxes == 900:
        assert counts["collide"] > 0
    if visited == 120000:
        assert counts["dup_visited"] > 0
