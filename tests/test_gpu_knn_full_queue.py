"""kNN queries that fill their wave's queue: many equal points, whose subtrees
are all as near as the k-th neighbour.  A query that loses a task is dropped and
runs again in a smaller group; lists against brute force, and the time of 8
neighbours against that of 16 (a longer queue), which is longer unless waves
go on with lost queries."""
import numpy as np
import pytest
import torch

from test_gpu_knn_small_leaves import _seconds

pytestmark = pytest.mark.gpu


def _places(places, copies):
    return np.random.default_rng(1).random((places, 3)).astype(np.float32).repeat(copies, 0)


@pytest.mark.parametrize("leaf", [2, 3])
def test_lost_queries_do_not_hold_up_their_wave(leaf):
    import cubql_amd as cq
    print(f"[gpu] kNN of equal points, time, leaves of {leaf}", flush=True)
    P = torch.from_numpy(_places(200, 1000)).cuda()
    Q = torch.rand((200000, 3), device="cuda", generator=torch.Generator("cuda").manual_seed(2))
    bvh = cq.gpuBuilder(cq.points_to_boxes(P), cq.BuildConfig(makeLeafThreshold=leaf))
    assert (_seconds(lambda: cq.points.findKNN(bvh, P, Q, 8))
            < 1.6 * _seconds(lambda: cq.points.findKNN(bvh, P, Q, 16)))


@pytest.mark.parametrize("k", [1, 8, 16])
@pytest.mark.parametrize("nq", [70, 5000, 262144])
def test_equal_points_equal_brute_force(oracle_mod, k, nq):
    import cubql_amd as cq
    print(f"[gpu] kNN of equal points, {nq} queries, {k} neighbours", flush=True)
    P = _places(3, 1500)
    Q = np.random.default_rng(nq).random((nq, 3)).astype(np.float32)
    dP, dQ = torch.from_numpy(P).cuda(), torch.from_numpy(Q).cuda()
    bvh = cq.gpuBuilder(cq.points_to_boxes(dP), cq.BuildConfig(makeLeafThreshold=1))
    ids, d2, found = (t.cpu().numpy() for t in cq.points.findKNN(bvh, dP, dQ, k))
    # the k lowest ids of the nearest place
    bi, bd = oracle_mod.fcp_brute(P[::1500], Q)
    assert np.array_equal(ids, bi[:, None] * 1500 + np.arange(k)[None])
    assert np.array_equal(d2, np.repeat(bd[:, None], k, 1))
    assert np.all(found == k)
