"""Parts of the batched path that ordinary clouds do not reach: queries that
lose a task even alone and go to the deep kernel (counted in the workspace), ranges
of more than 16384 points with one key, which are halved before the units are made,
and leaves of more than 16384 points, units of a single leaf."""
import numpy as np
import pytest
import torch

from test_gpu_batch import _check_loss_and_grads

pytestmark = pytest.mark.gpu


def _off(sizes):
    return torch.tensor(np.concatenate([[0], np.cumsum(sizes)]), dtype=torch.int32, device="cuda")


def _deep_queries(b):
    """Queries of the last direction (targets) that the deep kernel took: the
    first word of the overflow list, the last part of the workspace."""
    words = max(b.src.shape[0], b.tgt.shape[0]) + 2
    at = b.ws.numel() - (4 * words + 255) // 256 * 256
    return int(b.ws[at:at + 4].view(torch.int32).item())


def _brute(data, queries):
    """(lowest index, squared distance) in float32, as the kernels round it."""
    ids, ds = [], []
    for q in queries.split(512):
        d = q[:, None, :] - data[None]
        d = d[..., 0] * d[..., 0] + d[..., 1] * d[..., 1] + d[..., 2] * d[..., 2]
        m = d.min(1).values
        ids.append((d == m[:, None]).int().argmax(1))
        ds.append(m)
    return torch.cat(ids).int(), torch.cat(ds)


def _check_nearest(b, so, to):
    for c in range(len(so) - 1):
        S, T = b.src[so[c]:so[c + 1]], b.tgt[to[c]:to[c + 1]]
        for nn, d2, data, q, at, base in ((b.src_nn, b.src_d2, T, S, slice(so[c], so[c + 1]), to[c]),
                                          (b.tgt_nn, b.tgt_d2, S, T, slice(to[c], to[c + 1]), so[c])):
            i, d = _brute(data, q)
            assert torch.equal(nn[at], i + int(base)), c
            assert torch.equal(d2[at], d), c


@pytest.mark.parametrize("copies,some", [(60000, True), (200, False)])
def test_deep_kernel(oracle_mod, copies, some):
    import cubql_amd as cq
    print(f"[gpu] batch deep kernel, {copies} equal points", flush=True)
    rng = np.random.default_rng(copies)
    S, T, so, to = [], [], [0], [0]
    for c in range(3):
        S.append(np.concatenate([np.tile(rng.random((1, 3)), (copies, 1)), 5 + rng.random((7, 3))]))
        T.append(rng.random((100 + c, 3)))
        so.append(so[-1] + len(S[-1]))
        to.append(to[-1] + len(T[-1]))
    S, T = (torch.from_numpy(np.concatenate(x).astype(np.float32)).cuda() for x in (S, T))
    dso, dto = (torch.tensor(x, dtype=torch.int32, device="cuda") for x in (so, to))
    b = cq.ChamferBatch(S, dso, T, dto, cq.BatchParams(leafSize=1)).run()
    torch.cuda.synchronize()
    assert (_deep_queries(b) > 0) == some
    _check_nearest(b, so, to)
    _check_loss_and_grads(oracle_mod, b, S, dso, T, dto, range(3))


@pytest.mark.parametrize("leaf", [3, 64])
def test_many_points_with_one_key(oracle_mod, leaf):
    import cubql_amd as cq
    print(f"[gpu] batch of 40000 points with one key, leaves of {leaf}", flush=True)
    rng = np.random.default_rng(leaf)
    # 40000 points in one cell of the cloud's 1024 a side, some of them equal
    close = 0.5 + 1e-5 * rng.integers(0, 60, (40000, 3))
    S = np.concatenate([close, [[0, 0, 0], [1, 1, 1]], rng.random((50, 3))]).astype(np.float32)
    T = np.concatenate([0.5 + 6e-4 * rng.random((300, 3)), rng.random((30, 3)), rng.random((40, 3))]).astype(np.float32)
    so, to = [0, 40002, 40052], [0, 330, 370]
    dS, dT = torch.from_numpy(S).cuda(), torch.from_numpy(T).cuda()
    dso, dto = (torch.tensor(x, dtype=torch.int32, device="cuda") for x in (so, to))
    b = cq.ChamferBatch(dS, dso, dT, dto, cq.BatchParams(leafSize=leaf)).run()
    torch.cuda.synchronize()
    _check_nearest(b, so, to)
    _check_loss_and_grads(oracle_mod, b, dS, dso, dT, dto, range(2))


@pytest.mark.parametrize("leaf", [16384, 16385, 40000, 70000])
def test_large_leaves(leaf):
    import cubql_amd as cq
    print(f"[gpu] batch with leaves of {leaf}", flush=True)
    sizes = [100, 16384, 16385, 20000, 0, 33000, 70000, 3]
    g = torch.Generator("cuda").manual_seed(leaf)
    S = torch.randn((sum(sizes), 3), device="cuda", generator=g)
    T = torch.randn((40 * len(sizes), 3), device="cuda", generator=g)
    so, to = _off(sizes), _off([40] * len(sizes))
    got = cq.ChamferBatch(S, so, T, to, cq.BatchParams(leafSize=leaf)).run()
    want = cq.ChamferBatch(S, so, T, to, cq.BatchParams(leafSize=8)).run()
    torch.cuda.synchronize()
    for name in ("src_nn", "src_d2", "tgt_nn", "tgt_d2"):
        assert torch.equal(getattr(got, name), getattr(want, name)), name
