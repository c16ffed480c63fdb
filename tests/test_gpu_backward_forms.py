"""Distance adjoints at the edges of their work split, against 64-bit ones.

Points: k below, at and above a workgroup's 1024 terms, batches that end in
the middle of a workgroup, arbitrary ids with -1 ("none"), -2 ("incomplete"),
repeats and coincident points.  A term g (q - p) / |q - p| has at most six
roundings (difference, three of the norm, quotient, product), each of 2^-24
of its size at most |g|, and a sum of m terms at most m more: every sum is
within (m + 6) 2^-23 of the sum of its |g|, twice the bound.

Triangles: batches on both sides of a wave and a workgroup, meshes with and
without an index array, any triangle as the closest one, ids -1 among them.
The weights of a closest point sum to 1, so the three vertex gradients that
the queries of a triangle add sum to minus the sum of its query gradients.
Per query that takes the roundings of two subtractions for the third weight
and of three products (five of 2^-24 of the query gradient), and the 3 m
additions of m queries one each of the sum of their sizes: within (3 m + 8)
2^-23 of the sum of |query gradient|, over twice the bound.  (The gradients
of closest triangles are checked against 64 bits elsewhere.)"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -24


@pytest.mark.parametrize("k,nq", [(1, 1), (1, 1023), (1, 1025), (3, 341), (3, 342), (16, 65), (64, 33), (1023, 3),
                                  (1024, 2), (1025, 2), (2500, 2)])
def test_points_backward_forms(oracle_mod, k, nq):
    import cubql_amd as cq
    print(f"[gpu] points backward k={k}, {nq} queries", flush=True)
    rng = np.random.default_rng(k * 1000 + nq)
    n = 777
    P = rng.random((n, 3), dtype=np.float32)
    Q = rng.random((nq, 3), dtype=np.float32)
    Q[0] = P[5]
    ids = rng.integers(-2, n, (nq, k)).astype(np.int32)
    ids[0, 0] = 5
    g = (rng.random((nq, k)) + 0.5).astype(np.float32)
    gq = torch.full((nq, 3), 7.0, device="cuda")
    gp = torch.ones((n, 3), device="cuda")
    shape = (nq,) if k == 1 else (nq, k)
    cq.points_backward(torch.from_numpy(P).cuda(), torch.from_numpy(Q).cuda(),
                       torch.from_numpy(ids.reshape(shape)).cuda(), torch.from_numpy(g.reshape(shape)).cuda(), gq, gp)
    q64, p64 = oracle_mod.point_grad_f64(P, Q, ids, g.astype(np.float64))
    live = ids >= 0
    tol_q = (k + 6) * 2 * EPS * (g * live).sum(1)[:, None]
    sums, cnt = np.zeros(n), np.zeros(n)
    np.add.at(sums, ids[live], g[live])
    np.add.at(cnt, ids[live], 1)
    tol_p = ((cnt + 7) * 2 * EPS * (sums + 1))[:, None]  # (accumulated onto the 1 it held)
    assert np.all(np.abs(gq.cpu().numpy() - q64) <= tol_q)
    assert np.all(np.abs(gp.cpu().numpy() - 1 - p64) <= tol_p)


@pytest.mark.parametrize("nq", [1, 63, 65, 255, 257, 3001])
@pytest.mark.parametrize("indexed", [True, False])
def test_triangles_backward_forms(nq, indexed):
    import cubql_amd as cq
    from cubql_amd import synth
    print(f"[gpu] triangle backward {nq} queries, indexed {indexed}", flush=True)
    V, F = synth.noisy_icosphere(2, seed=9)
    if not indexed:
        V = np.ascontiguousarray(V[F.reshape(-1)])
        F = np.arange(len(V), dtype=np.int32).reshape(-1, 3)
    rng = np.random.default_rng(nq)
    Q = (rng.standard_normal((nq, 3))).astype(np.float32)
    ids = rng.integers(-1, len(F), nq).astype(np.int32)  # any triangle: all regions, far and near
    g = (rng.random(nq) + 0.5).astype(np.float32)
    dV, dQ = torch.from_numpy(V).cuda(), torch.from_numpy(Q).cuda()
    gq, gv = torch.full((nq, 3), 7.0, device="cuda"), torch.zeros_like(dV)
    cq.triangles.backward(torch.from_numpy(F).cuda() if indexed else None, dV, dQ, torch.from_numpy(ids).cuda(),
                          torch.from_numpy(g).cuda(), gq, gv)
    gq, gv = gq.cpu().numpy().astype(np.float64), gv.cpu().numpy().astype(np.float64)
    live = ids >= 0
    assert np.all(gq[~live] == 0)
    want, size, m = np.zeros((len(F), 3)), np.zeros((len(F), 3)), np.zeros(len(F))
    np.add.at(want, ids[live], -gq[live])
    np.add.at(size, ids[live], np.abs(gq[live]))
    np.add.at(m, ids[live], 1)
    if not indexed:
        assert np.all(np.abs(gv[F].sum(1) - want) <= ((3 * m + 8) * 2 * EPS)[:, None] * size)
        assert np.all(gv[F[m == 0]] == 0)
    # vertices shared by triangles: the whole mesh's sums
    n = live.sum()
    assert np.all(np.abs(gv.sum(0) - want.sum(0)) <= (3 * n + 8) * 2 * EPS * size.sum(0))
