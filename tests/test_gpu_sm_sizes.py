"""Spatial-median builds at the sizes where the number of passes or who
reduces a node's bounds changes: up to 1024 prims (no pass), the steps up to
64K, sizes whose nodes of two levels end just above and below the small
phase, clustered points (uneven splits) and points on a line with copies
(one-sided splits).  The tree equals the oracle's."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["uniform", "clustered", "line"])
@pytest.mark.parametrize("n", [1, 8, 9, 1023, 1024, 1025, 2048, 2049, 4096, 4097, 5000, 16385, 24000, 65537, 90000, 130000])
def test_median_build_equals_oracle(oracle_mod, kind, n):
    import cubql_amd as cq
    print(f"[gpu] median build {kind}, {n} points", flush=True)
    rng = np.random.default_rng(n)
    P = rng.random((n, 3), dtype=np.float32)
    if kind == "clustered":
        P = P ** 6
        P[::97] *= 1000
    elif kind == "line":
        P[:, 1:] = 0.5
        P[:, 0] = np.where(rng.random(n) < 0.3, np.float32(0.25), P[:, 0])
    B = oracle_mod.points_to_boxes(P)
    bvh = cq.gpuBuilder(torch.from_numpy(B).cuda(), cq.BuildConfig(makeLeafThreshold=8))
    tree = oracle_mod.Tree(cq.nodes_to_numpy(bvh).view(oracle_mod.NODE_DTYPE),
                           bvh.prim_ids_tensor().cpu().numpy().view(np.uint32))
    want = oracle_mod.sm_build(B, 8)
    assert np.array_equal(tree.prim_ids, want.prim_ids)
    assert np.array_equal(oracle_mod.canonical(tree), oracle_mod.canonical(want))
    assert oracle_mod.check_tree(tree, B, 8)[0] == 0
