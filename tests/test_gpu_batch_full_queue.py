"""Batched Chamfer against clouds of equal points, whose subtrees are all as
near as the closest point and fill the queue of the wave: nearest points and
distances against brute force, and the time with leaves of one point against
leaves of 16, a sixteenth of the subtrees (6 times as long; 12 where waves go on
with queries that have lost a task)."""
import numpy as np
import pytest
import torch

from test_gpu_knn_small_leaves import _seconds

pytestmark = pytest.mark.gpu


def _batch(clouds, n, leaf):
    import cubql_amd as cq
    g = torch.Generator("cuda").manual_seed(1)
    src = torch.randn((clouds * n, 3), device="cuda", generator=g)
    tgt = torch.full_like(src, 0.3)
    off = torch.arange(clouds + 1, device="cuda", dtype=torch.int32) * n
    return cq.ChamferBatch(src, off, tgt, off, cq.BatchParams(leafSize=leaf))


def test_lost_queries_do_not_hold_up_their_wave():
    print("[gpu] batch of equal points, time", flush=True)
    small, large = _batch(30, 3000, 1), _batch(30, 3000, 16)
    assert _seconds(small.run) < 8.5 * _seconds(large.run)


@pytest.mark.parametrize("clouds,n,leaf", [(3, 20, 1), (7, 900, 1), (40, 3000, 1), (40, 3000, 5)])
def test_equal_points_equal_brute_force(clouds, n, leaf):
    print(f"[gpu] batch of equal points: {clouds} clouds of {n}, leaves of {leaf}", flush=True)
    b = _batch(clouds, n, leaf).run()
    torch.cuda.synchronize()
    first = (torch.arange(clouds * n, device="cuda") // n * n).int()
    # every source point: the lowest of its cloud's equal points
    assert torch.equal(b.src_nn, first)
    d = b.src - b.tgt
    d = d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1] + d[:, 2] * d[:, 2]
    assert torch.allclose(b.src_d2, d, rtol=1e-6, atol=0)
    # every target point: the nearest source point of its cloud
    near = b.src_d2.view(clouds, n).argmin(1).repeat_interleave(n).int() + first
    assert torch.equal(b.tgt_nn, near)
    assert torch.equal(b.tgt_d2, b.src_d2[near.long()])
