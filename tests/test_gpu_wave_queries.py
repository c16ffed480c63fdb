"""Closest points by wave-shared traversal against brute force, at the sizes
where the sharing can go wrong: fewer queries than lanes, batches on both
sides of a wave, of the query-ordering threshold (32768) and of the steps in
queries per wave, trees of one leaf and of one-prim leaves, ties (the lowest
id wins), radii that nothing or only equal distances reach, and queries far
outside, which keep many subtrees queued, and tight clusters with far-off
outliers, whose large batches are ordered by leaf.  Distances are rounded the same
way on both sides, so ids and distances must be equal."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def cq():
    import cubql_amd
    cubql_amd.lib()
    return cubql_amd


def _cloud(kind, n, rng):
    if kind == "uniform":
        return rng.random((n, 3), dtype=np.float32)
    if kind == "ties":  # every point several times, on a coarse lattice
        return rng.integers(0, 4, (n, 3)).astype(np.float32)
    if kind == "outliers":
        p = rng.integers(0, 3, (n, 1)) + 0.001 * rng.standard_normal((n, 3))
        p[::50] *= 1e6
        return p.astype(np.float32)
    shell = rng.standard_normal((n, 3))  # a shell, its queries near the centre
    return (shell / np.linalg.norm(shell, axis=1, keepdims=True)).astype(np.float32)


def _queries(kind, nq, rng):
    if kind == "uniform":
        return (rng.random((nq, 3)) * 1.2 - 0.1).astype(np.float32)
    if kind == "ties":
        return (rng.integers(0, 8, (nq, 3)) * 0.5).astype(np.float32)
    if kind == "outliers":
        return (rng.integers(0, 3, (nq, 1)) + 0.002 * rng.standard_normal((nq, 3))).astype(np.float32)
    return (rng.standard_normal((nq, 3)) * 0.02).astype(np.float32)


@pytest.mark.parametrize("kind", ["uniform", "ties", "shell", "outliers"])
@pytest.mark.parametrize("n,leaf", [(1, 8), (9, 8), (300, 1), (4097, 8)])
@pytest.mark.parametrize("nq", [1, 63, 65, 4097, 8193, 32767, 40001])
def test_closest_point_equals_brute_force(cq, oracle_mod, kind, n, leaf, nq):
    print(f"[gpu] fcp {kind}: {n} points, leaf {leaf}, {nq} queries", flush=True)
    rng = np.random.default_rng(n * 100000 + nq)
    P, Q = _cloud(kind, n, rng), _queries(kind, nq, rng)
    bvh = cq.gpuBuilder(cq.points_to_boxes(torch.from_numpy(P).cuda()), cq.BuildConfig(makeLeafThreshold=leaf))
    dP, dQ = torch.from_numpy(P).cuda(), torch.from_numpy(Q).cuda()
    bi, bd = oracle_mod.fcp_brute(P, Q)
    for r2 in (np.inf, float(np.median(bd)), 0.0):
        ids, d2 = cq.points.findClosest(bvh, dP, dQ, r2)
        near = bd < np.float32(r2)
        assert np.array_equal(ids.cpu().numpy(), np.where(near, bi, -1))
        assert np.array_equal(d2.cpu().numpy(), np.where(near, bd, np.float32(np.inf)))
