"""Closest points among equal points, whose subtrees are all as near as the
closest one and fill the queue of the wave: ids and distances against brute
force, and the time of ten times the queries (8 times as long, waves of 64
queries against waves of 8; 37 where the queries that lose a task are left to a
few lanes of the deep kernel)."""
import numpy as np
import pytest
import torch

from test_gpu_knn_full_queue import _places
from test_gpu_knn_small_leaves import _seconds

pytestmark = pytest.mark.gpu


def test_lost_queries_run_in_their_wave():
    import cubql_amd as cq
    print("[gpu] closest of equal points, time", flush=True)
    P = torch.from_numpy(_places(1, 3000)).cuda()
    Q = torch.rand((200000, 3), device="cuda", generator=torch.Generator("cuda").manual_seed(2))
    bvh = cq.gpuBuilder(cq.points_to_boxes(P), cq.BuildConfig(makeLeafThreshold=16))
    few = Q[:20000].contiguous()
    assert (_seconds(lambda: cq.points.findClosest(bvh, P, Q))
            < 18 * _seconds(lambda: cq.points.findClosest(bvh, P, few)))


@pytest.mark.parametrize("leaf", [1, 16])
@pytest.mark.parametrize("nq", [1, 70, 5000, 262144])
def test_equal_points_equal_brute_force(oracle_mod, leaf, nq):
    import cubql_amd as cq
    print(f"[gpu] closest of equal points, {nq} queries, leaves of {leaf}", flush=True)
    P = _places(3, 1500)
    Q = np.random.default_rng(nq).random((nq, 3)).astype(np.float32)
    dP, dQ = torch.from_numpy(P).cuda(), torch.from_numpy(Q).cuda()
    bvh = cq.gpuBuilder(cq.points_to_boxes(dP), cq.BuildConfig(makeLeafThreshold=leaf))
    bi, bd = oracle_mod.fcp_brute(P[::1500], Q)
    for r2 in (np.inf, float(np.median(bd))):
        ids, d2 = (t.cpu().numpy() for t in cq.points.findClosest(bvh, dP, dQ, r2))
        near = bd < np.float32(r2)
        assert np.array_equal(ids, np.where(near, bi * 1500, -1))
        assert np.array_equal(d2, np.where(near, bd, np.float32(np.inf)))
