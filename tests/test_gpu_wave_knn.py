"""k nearest neighbours by wave-shared traversal against brute force: every
list length of the kernels (4, 8, 16) and the ones between, fewer prims than
k, fewer queries than lanes, batches on both sides of a wave and of the
ordering threshold, one-prim leaves (a query is seeded from many of them),
large leaves (a leaf fills a query's buffer several times), ties (the lower
id first), finite radii and clusters with outliers.  Distances are rounded
the same way on both sides, so ids and distances must be equal."""
import numpy as np
import pytest
import torch

from test_gpu_wave_queries import _cloud, _queries

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["uniform", "ties", "shell", "outliers"])
@pytest.mark.parametrize("n,leaf,nq", [(1, 8, 3), (7, 2, 65), (300, 1, 257), (4097, 8, 4099), (1000, 100, 1000),
                                       (2000, 8, 32769)])
@pytest.mark.parametrize("k", [1, 4, 5, 8, 10, 16])
def test_knn_equals_brute_force(oracle_mod, kind, n, leaf, nq, k):
    import cubql_amd as cq
    print(f"[gpu] knn {kind}: {n} points, leaf {leaf}, {nq} queries, k {k}", flush=True)
    rng = np.random.default_rng(n * 1000 + nq)
    P, Q = _cloud(kind, n, rng), _queries(kind, nq, rng)
    dP, dQ = torch.from_numpy(P).cuda(), torch.from_numpy(Q).cuda()
    bvh = cq.gpuBuilder(cq.points_to_boxes(dP), cq.BuildConfig(makeLeafThreshold=leaf))
    kk = min(k, n)
    bi, bd = oracle_mod.knn_brute(P, Q, kk)[:2]
    for r2 in (np.inf, float(np.median(bd))):
        ids, d2, found = (t.cpu().numpy() for t in cq.points.findKNN(bvh, dP, dQ, k, r2))
        near = bd < np.float32(r2)
        assert np.array_equal(found, near.sum(1))
        assert np.array_equal(ids[:, :kk], np.where(near, bi, -1))
        assert np.array_equal(d2[:, :kk], np.where(near, bd, np.float32(np.inf)))
        assert np.all(ids[:, kk:] == -1) and np.all(np.isinf(d2[:, kk:]))
