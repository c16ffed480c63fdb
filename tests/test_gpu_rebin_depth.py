"""Boxes of rebin-built trees whose broad phase has few levels (fitted a level
at a time) and many (fitted by the generic climb): uniform points, clusters
with outliers, a geometric row of points, and boxes.  Every leaf box is the
union of its prims' and every inner box that of its children, exactly."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["uniform", "clusters", "row", "boxes"])
@pytest.mark.parametrize("n,T", [(40, 1), (3000, 8), (50000, 4)])
def test_rebin_boxes(oracle_mod, kind, n, T):
    import cubql_amd as cq
    print(f"[gpu] rebin {kind}, {n} prims, T {T}", flush=True)
    rng = np.random.default_rng(n)
    P = rng.random((n, 3), dtype=np.float32)
    half = np.zeros_like(P)
    if kind == "clusters":
        P = P ** 9
        P[::101] *= 1000
    elif kind == "row":
        P[:, 0] = np.float32(2.0) ** -(np.arange(n) % 100)
    elif kind == "boxes":
        half = rng.random((n, 3), dtype=np.float32) * np.float32(0.01)
    B = np.concatenate([P - half, P + half], axis=1).astype(np.float32)
    bvh = cq.cuda.rebinRadixBuilder(torch.from_numpy(B).cuda(), cq.BuildConfig(makeLeafThreshold=T))
    tree = oracle_mod.Tree(cq.nodes_to_numpy(bvh).view(oracle_mod.NODE_DTYPE),
                           bvh.prim_ids_tensor().cpu().numpy().view(np.uint32))
    assert oracle_mod.check_tree(tree, B, T)[0] == 0
