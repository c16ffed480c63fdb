"""Spatial-median builds whose small nodes are finished by a workgroup each,
on both sides of the sizes where the workgroup changes (2^17 prims) and where
waves take over (2^20): leaves from one
prim to larger than a segment, pieces of 64 and 65 prims, points, boxes,
clusters, and copies (one-sided splits all the way down).  The tree equals the
oracle's, and its nodes are numbered without a gap, children after parents."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["points", "boxes", "clustered", "clustered boxes", "copies"])
@pytest.mark.parametrize("n,T", [(1, 1), (64, 8), (65, 1), (65, 64), (257, 70), (1000, 1), (1024, 300), (1025, 4),
                                 (3001, 8), (3001, 2000), (70000, 3), (1 << 17, 8),
                                 ((1 << 17) + 1, 8), (1 << 20, 8), ((1 << 20) + 1, 8)])
def test_wide_small_nodes(oracle_mod, kind, n, T):
    import cubql_amd as cq
    print(f"[gpu] median build {kind}, {n} prims, T {T}", flush=True)
    rng = np.random.default_rng(n + T)
    P = rng.random((n, 3), dtype=np.float32)
    half = np.zeros_like(P)
    if kind == "boxes":
        half = rng.random((n, 3), dtype=np.float32) * np.float32(0.01)
    elif kind.startswith("clustered"):
        # (more lists of inner nodes than one workgroup takes)
        P = P ** 8
        P[::97] *= 1000
        if kind == "clustered boxes":
            half = P * np.float32(0.01)
    elif kind == "copies":
        P = P[rng.integers(0, max(1, n // 200), n)]
    B = np.concatenate([P - half, P + half], axis=1).astype(np.float32)
    bvh = cq.gpuBuilder(torch.from_numpy(B).cuda(), cq.BuildConfig(makeLeafThreshold=T))
    nodes = cq.nodes_to_numpy(bvh).view(oracle_mod.NODE_DTYPE)
    tree = oracle_mod.Tree(nodes, bvh.prim_ids_tensor().cpu().numpy().view(np.uint32))
    want = oracle_mod.sm_build(B, T)
    assert np.array_equal(tree.prim_ids, want.prim_ids)
    assert np.array_equal(oracle_mod.canonical(tree), oracle_mod.canonical(want))
    assert oracle_mod.check_tree(tree, B, T)[0] == 0
    word = nodes.view(np.uint64).reshape(len(nodes), 4)[:, 3]
    used = np.concatenate([[0], np.arange(2, len(nodes))]) if len(nodes) > 2 else np.arange(1)
    inner = used[(word[used] >> np.uint64(48)) == 0]
    child = (word[inner] & np.uint64((1 << 48) - 1)).astype(np.int64)
    assert np.array_equal(np.sort(np.concatenate([child, child + 1])), np.arange(2, len(nodes)) if len(nodes) > 2 else [])
    assert np.all(child > inner)
