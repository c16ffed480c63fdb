"""Closest triangles with tests dealt out over a wave, against the oracle's
traversal of the same tree: batches on both sides of a wave and of the
ordering threshold, one-triangle leaves, leaves of more triangles than are
dealt out at once, equal triangles (the lowest id wins), finite radii, and
meshes with and without an index array.  Distances and closest points are
rounded the same way on both sides and must be equal."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("indexed", [True, False])
@pytest.mark.parametrize("leaf", [1, 4, 8, 9, 50])
@pytest.mark.parametrize("nq", [1, 63, 65, 4097, 32769])
def test_closest_triangle_equals_oracle(oracle_mod, nq, leaf, indexed):
    import cubql_amd as cq
    from cubql_amd import synth
    print(f"[gpu] closest triangle: {nq} queries, leaf {leaf}, indexed {indexed}", flush=True)
    V, F = synth.noisy_icosphere(3, seed=leaf)
    F = np.concatenate([F, F[::7]])  # equal triangles with other ids
    if not indexed:
        V = np.ascontiguousarray(V[F.reshape(-1)])
        F = np.arange(len(V), dtype=np.int32).reshape(-1, 3)
    Q = (np.random.default_rng(nq).standard_normal((nq, 3)) * 0.8).astype(np.float32)
    dV, dF = torch.from_numpy(V).cuda(), torch.from_numpy(F).cuda() if indexed else None
    bvh = cq.gpuBuilder(cq.triangles.boxes(dF, dV), cq.BuildConfig(makeLeafThreshold=leaf))
    tree = oracle_mod.Tree(cq.nodes_to_numpy(bvh).view(oracle_mod.NODE_DTYPE),
                           bvh.prim_ids_tensor().cpu().numpy().view(np.uint32))
    for r2 in (np.inf, 0.05, 0.0):
        ids, d2, P = (t.cpu().numpy() for t in
                      cq.triangles.findClosest(bvh, dF, dV, torch.from_numpy(Q).cuda(), float(r2)))
        oi, od, oP = oracle_mod.fcp_tris(tree, F if indexed else None, V, Q, np.float32(r2))
        assert np.array_equal(ids, oi)
        has = oi >= 0
        assert np.array_equal(d2[has], od[has]) and np.array_equal(P[has], oP[has])
        assert np.all(np.isinf(d2[~has]))
