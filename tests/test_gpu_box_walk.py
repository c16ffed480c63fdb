"""Which box-query batches are put in order, and the walk they take.

A batch below 3 * 2^17 queries gains less from the wave's shared walk than its
order costs, so it is not ordered (no sort is launched).  From there on the
shared walk is checked against the oracle's walk of the same tree: ids in the
traversal's order and counts.  The flat and the peaked scene are sorted by all
three key bytes, the uniform one by two, the clustered one by leaf slots; more
than 64 open siblings send a wave's queries to the deep stack."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

WALK = 3 << 17


def _boxes(c, half):
    c = c.astype(np.float32)
    return np.hstack([c - np.float32(half), c + np.float32(half)])


@pytest.mark.parametrize("n,nq,sorts", [(50000, 50000, 0), (WALK, WALK - 1, 0), (WALK, WALK, 3), (2 * WALK + 2, WALK, 0)])
def test_only_large_batches_are_ordered(n, nq, sorts):
    import cubql_amd as cq
    print(f"[gpu] box query order {n} prims, {nq} queries", flush=True)
    rng = np.random.default_rng(n)
    B = torch.from_numpy(_boxes(rng.random((n, 3)), 0.002)).cuda()
    bvh = cq.gpuBuilder(B, cq.BuildConfig(makeLeafThreshold=4))
    cq.profile.reset()
    cq.profile.enable(True)
    try:
        cq.fixedBoxQuery.forEachPrim(bvh, B, B[:nq].contiguous(), 4)
        torch.cuda.synchronize()
    finally:
        cq.profile.enable(False)
    got = cq.profile.query("radix_onesweep")
    assert (got["launches"] if got else 0) == sorts


def _scene(name, n, rng):
    if name == "nested":
        # halving intervals: a level per prim, more than 64 of them open at once
        p = np.zeros((n, 3))
        p[:, 0] = 0.5 ** np.arange(n)
        return p
    p = rng.random((n, 3))
    if name == "flat":
        p[:, 2] = 0.5
    if name == "peaked":
        p = p ** 4
    if name == "clustered":
        p = p * 1e-4 + rng.integers(0, 2, (n, 1))
        p[0] = 1e3
    return p


@pytest.mark.parametrize("name,n,half,far", [("uniform", 3000, 0.02, 1.0), ("flat", 3000, 0.01, 1.0),
                                             ("peaked", 3000, 0.004, 1.0), ("clustered", 3000, 4e-6, 1e-4),
                                             ("nested", 140, 0.0, 0.1)])
def test_walk_equals_oracle(oracle_mod, name, n, half, far):
    import cubql_amd as cq
    print(f"[gpu] box walk {name}", flush=True)
    rng = np.random.default_rng(n)
    nq = WALK + 37
    prims = _boxes(_scene(name, n, rng), half)
    qc = _scene(name, n, rng)[rng.integers(0, n, nq)] + far * 0.01 * rng.standard_normal((nq, 3))
    Q = _boxes(qc, half)
    if name == "nested":
        # one query of a few waves overlaps everything
        Q[:: nq // 50] = [-1, -1, -1, 2, 2, 2]
    dP, dQ = torch.from_numpy(prims).cuda(), torch.from_numpy(Q).cuda()
    bvh = cq.gpuBuilder(dP, cq.BuildConfig(makeLeafThreshold=1 if name == "nested" else 4))
    keep = 6
    ids, counts = cq.fixedBoxQuery.forEachPrim(bvh, dP, dQ, keep)
    tree = oracle_mod.Tree(cq.nodes_to_numpy(bvh).view(oracle_mod.NODE_DTYPE),
                           bvh.prim_ids_tensor().cpu().numpy().view(np.uint32))
    want_ids, want_counts = oracle_mod.box_query(tree, prims, Q, keep)
    counts = counts.cpu().numpy().view(np.uint32)
    assert np.array_equal(counts, want_counts)
    assert counts.max() > (64 if name == "nested" else 1)
    got = ids.cpu().numpy().view(np.uint32)
    for j in range(keep):
        has = counts > j
        assert np.array_equal(got[has, j], np.asarray(want_ids)[has, j])
