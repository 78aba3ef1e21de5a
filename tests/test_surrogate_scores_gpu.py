"""Scores of the surrogate's inference at the edges of its tiles (32 pairs, one
run of tiles per workgroup), with nodes of one or two pairs, many nodes per
tile, patches under no, few and many boxes, against the numpy restatement; and
the rejection that follows from them, exactly."""
import ctypes as C

import numpy as np
import pytest

from dynoplan_amd import _native as N
from dynoplan_amd import synth
from dynoplan_amd.expander import expander_for

from test_surrogate_gpu import bf16, fptr, patches_np, unpack

pytestmark = pytest.mark.gpu


def scores_np(theta, emb, patch, prim):
    """z and, for each pair, sum |h3 w4|: what one bound covers."""
    P = unpack(theta)
    W1b = bf16(P["W1"]).astype(np.float64)
    h = patch.astype(np.float64) @ W1b[:, :1024].T + bf16(emb[prim]).astype(np.float64) @ W1b[:, 1024:].T + P["b1"]
    for W, b in (("W2", "b2"), ("W3", "b3")):
        h = bf16(np.maximum(h, 0)).astype(np.float64) @ bf16(P[W]).astype(np.float64).T + P[b]
    h = bf16(np.maximum(h, 0)).astype(np.float64)
    w4 = P["w4"].astype(np.float64)
    return h @ w4 + float(P["b4"][0]), np.abs(h) @ np.abs(w4)


@pytest.mark.parametrize("nodes,prims,boxes", [(1, 300, 0), (1, 4000, 5), (33, 40, 500), (700, 12, 60), (65, 900, 300),
                                               (3000, 400, 150)])
def test_scores(need_gpu, nodes, prims, boxes):
    w = synth._planar_workload("", N.SYS_CAR_TRAILER, nodes + prims, prims, 5, 20, 30.0 if boxes > 200 else 14.0, boxes, nodes, 100,
                               prim_fn=synth.car_trailer_primitives)
    p = w.params
    n = int(N.load().dp_surrogate_param_count())
    theta, emb = np.zeros(n, np.float32), np.zeros((prims, 64), np.float32)
    with expander_for(w) as ex:
        ex.surrogate_init(seed=nodes)
        N.check(ex.lib.dp_surrogate_get(ex.ctx, fptr(theta), fptr(emb)))
        p.use_surrogate = 2
        c = ex.expand(w.nodes, w.g_parent, p)
        plain = ex.fetch()
        z = ex.surrogate_scores(c["pairs"])
        assert c["surrogate_reject"] == 0
        tau = float(np.float32(np.median(z))) if z.size else 0.0
        N.check(ex.lib.dp_surrogate_set_threshold(ex.ctx, C.c_float(tau)))
        p.use_surrogate = 1
        c1 = ex.expand(w.nodes, w.g_parent, p)
        sur = ex.fetch()
        z1 = ex.surrogate_scores(c["pairs"])
    print(f"{c['pairs']} pairs of {nodes} nodes")
    assert c["pairs"] > 0
    assert np.array_equal(z, z1)
    rej = z < np.float32(tau)
    assert np.array_equal(sur["verdict"] == N.V_SURROGATE_REJECT, rej) and c1["surrogate_reject"] == rej.sum()
    assert np.array_equal(sur["verdict"][~rej], plain["verdict"][~rej])
    patch = patches_np(w.nodes, w.boxes)
    for q in np.array_split(np.arange(z.size), max(1, z.size // 20000)):
        ref, size = scores_np(theta, emb, patch[plain["node"][q]], plain["prim"][q])
        # an FP32 sum next to a rounding boundary may round each of the three
        # BF16 layers one step (2^-8 of a term) the other way
        assert (np.abs(z[q] - ref) <= 2.0 ** -8 * size).all()
        if q.size > 64:  # a tile out of place would be seen
            assert (np.abs(np.roll(z[q], 32) - ref) > 2.0 ** -8 * size).any()
