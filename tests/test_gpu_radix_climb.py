"""Boxes of radix-built trees where the climb to the root changes hands: fewer
pairs than a workgroup takes (1024), as many and a few more, trees that are one
long chain (each split parts one prim from the rest, so every node has a leaf
for a sibling), subtrees that straddle workgroups, groups of equal keys, and
leaves larger than the tree.  The tree equals the oracle's, boxes included."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["uniform", "chain", "groups", "boxes"])
@pytest.mark.parametrize("n,T", [(1, 1), (2, 1), (3, 1), (20, 30), (1024, 1), (1025, 1), (1026, 1), (2050, 1),
                                 (9000, 8), (40000, 1), (200000, 5)])
@pytest.mark.parametrize("bits", [10, 21])
def test_radix_boxes(oracle_mod, kind, n, T, bits):
    import cubql_amd as cq
    print(f"[gpu] radix {kind}, {n} prims, T {T}, {bits} bits", flush=True)
    rng = np.random.default_rng(n + T)
    P = rng.random((n, 3), dtype=np.float32)
    half = np.zeros_like(P)
    if kind == "chain":
        # powers of two along x, copies of the last ones
        P[:] = 0
        P[:, 0] = np.float32(2.0) ** -(np.arange(n) % 24)
    elif kind == "groups":
        P = P[rng.integers(0, max(1, n // 11), n)]
    elif kind == "boxes":
        half = rng.random((n, 3), dtype=np.float32) * np.float32(0.01)
    B = np.concatenate([P - half, P + half], axis=1).astype(np.float32)
    build = cq.cuda.radixBuilder if bits == 21 else cq.cuda.radix30Builder
    bvh = build(torch.from_numpy(B).cuda(), cq.BuildConfig(makeLeafThreshold=T))
    tree = oracle_mod.Tree(cq.nodes_to_numpy(bvh).view(oracle_mod.NODE_DTYPE),
                           bvh.prim_ids_tensor().cpu().numpy().view(np.uint32))
    want = oracle_mod.radix_build(B, bits, T)
    assert np.array_equal(tree.prim_ids, want.prim_ids)
    assert np.array_equal(oracle_mod.canonical(tree), oracle_mod.canonical(want))
    assert oracle_mod.check_tree(tree, B, T)[0] == 0
    assert bvh.numNodes == len(want.nodes)
