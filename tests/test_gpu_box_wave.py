"""Box queries of large batches (wave-shared walk) against the oracle's walk
of the same tree: ids in the traversal's order and counts.  Batches end in
the middle of a wave; results per query below, at and above the kept number;
boxes that overlap nothing and everything; touching boxes (closed intervals);
trees of one leaf and of one-prim leaves."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,leaf,nq", [(3, 8, 32768), (1500, 1, 32769), (40000, 4, 40001)])
@pytest.mark.parametrize("keep", [0, 5, 64])
def test_box_query_large_batch(oracle_mod, n, leaf, nq, keep):
    import cubql_amd as cq
    print(f"[gpu] box query {n} prims, leaf {leaf}, {nq} queries, keep {keep}", flush=True)
    rng = np.random.default_rng(n + keep)
    c = rng.random((n, 3)).astype(np.float32)
    c[: n // 3] = np.round(c[: n // 3] * 8) / 8  # boxes that touch exactly
    h = np.float32(0.0625) * rng.integers(0, 2, (n, 3)).astype(np.float32)
    boxes = np.hstack([c - h, c + h])
    qc = (rng.random((nq, 3)) * 1.5 - 0.25).astype(np.float32)
    qc[::3] = np.round(qc[::3] * 8) / 8
    qh = (0.03 * rng.random((nq, 1)) ** 3).astype(np.float32) * np.ones((1, 3), np.float32)
    qh[0] = 4.0
    Q = np.hstack([qc - qh, qc + qh])
    bvh = cq.gpuBuilder(torch.from_numpy(boxes).cuda(), cq.BuildConfig(makeLeafThreshold=leaf))
    ids, counts = cq.fixedBoxQuery.forEachPrim(bvh, torch.from_numpy(boxes).cuda(), torch.from_numpy(Q).cuda(), keep)
    tree = oracle_mod.Tree(cq.nodes_to_numpy(bvh).view(oracle_mod.NODE_DTYPE),
                           bvh.prim_ids_tensor().cpu().numpy().view(np.uint32))
    want_ids, want_counts = oracle_mod.box_query(tree, boxes, Q, max(keep, 1))
    counts = counts.cpu().numpy().view(np.uint32)
    assert np.array_equal(counts, want_counts)
    assert counts.max() == n and counts.min() == 0
    if keep:
        got = ids.cpu().numpy().view(np.uint32)
        for j in range(keep):
            has = counts > j
            assert np.array_equal(got[has, j], np.asarray(want_ids)[has, j])
            assert np.all(got[~has, j] == 0xffffffff)
