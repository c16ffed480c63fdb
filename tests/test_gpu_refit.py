"""Refit at the sizes where its climb can go wrong: one leaf, two leaves
under the root (one thread computes both), odd numbers of leaves, leaves of
one to nine prims (four boxes are read at a time) and a chain, where every
parent has a leaf and an inner child.  Boxes are minima and maxima of the
input's, so the expected ones are exact."""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def cq():
    import cubql_amd
    cubql_amd.lib()
    return cubql_amd


def _expected(nodes, prims, boxes):
    """Node boxes from the prims up (node ids visited in post order)."""
    oc = nodes["oc"].astype(np.uint64)
    off = (oc & np.uint64((1 << 48) - 1)).astype(np.int64)
    cnt = (oc >> np.uint64(48)).astype(np.int64)
    lo, hi = {}, {}
    stack = [(0, False)]
    while stack:
        i, done = stack.pop()
        if cnt[i]:
            b = boxes[prims[off[i]:off[i] + cnt[i]]]
            lo[i], hi[i] = b[:, :3].min(0), b[:, 3:].max(0)
        elif done:
            lo[i] = np.minimum(lo[off[i]], lo[off[i] + 1])
            hi[i] = np.maximum(hi[off[i]], hi[off[i] + 1])
        else:
            stack += [(i, True), (off[i], False), (off[i] + 1, False)]
    return lo, hi


@pytest.mark.parametrize("n,leaf", [(1, 4), (2, 1), (3, 1), (9, 9), (10, 9), (257, 1), (5000, 3), (100003, 4)])
def test_refit_moved_boxes(cq, n, leaf):
    print(f"[gpu] refit {n} boxes, leaves of {leaf}", flush=True)
    rng = np.random.default_rng(n)
    c = rng.random((n, 3), dtype=np.float32)
    h = rng.random((n, 3), dtype=np.float32) * np.float32(0.05)
    bvh = cq.gpuBuilder(torch.from_numpy(np.hstack([c - h, c + h])).cuda(), cq.BuildConfig(makeLeafThreshold=leaf))
    c = c + rng.standard_normal((n, 3)).astype(np.float32) * np.float32(0.1)
    boxes = np.hstack([c - h, c + h])
    cq.refit(bvh, torch.from_numpy(boxes).cuda())
    torch.cuda.synchronize()
    nodes, prims = cq.nodes_to_numpy(bvh), bvh.prim_ids_tensor().cpu().numpy().view(np.uint32)
    lo, hi = _expected(nodes, prims, boxes)
    for i in lo:
        assert np.array_equal(nodes["lo"][i], lo[i]) and np.array_equal(nodes["hi"][i], hi[i]), i


@pytest.mark.parametrize("builder", ["radixBuilder", "rebinRadixBuilder", "sahBuilder"])
@pytest.mark.parametrize("n", [255, 513, 20001])
def test_refit_numberings(cq, builder, n):
    """Spans of nodes that hold whole subtrees, parts of them, or neither."""
    print(f"[gpu] refit {builder}, {n} boxes", flush=True)
    rng = np.random.default_rng(n)
    c = rng.random((n, 3), dtype=np.float32)
    build = getattr(cq.cuda, builder)
    bvh = build(torch.from_numpy(np.hstack([c, c])).cuda(), cq.BuildConfig(makeLeafThreshold=1))
    boxes = np.hstack([c - np.float32(0.3), c + rng.random((n, 3), dtype=np.float32)])
    cq.refit(bvh, torch.from_numpy(boxes).cuda())
    torch.cuda.synchronize()
    nodes, prims = cq.nodes_to_numpy(bvh), bvh.prim_ids_tensor().cpu().numpy().view(np.uint32)
    lo, hi = _expected(nodes, prims, boxes)
    for i in lo:
        assert np.array_equal(nodes["lo"][i], lo[i]) and np.array_equal(nodes["hi"][i], hi[i]), i


@pytest.mark.parametrize("depth", [1, 2, 300, 1000])
def test_refit_chain(cq, depth):
    from test_gpu_deep import _chain
    print(f"[gpu] refit chain of depth {depth}", flush=True)
    nodes, prims = _chain(depth)
    rng = np.random.default_rng(depth)
    lo = rng.standard_normal((depth + 1, 3)).astype(np.float32)
    boxes = np.hstack([lo, lo + rng.random((depth + 1, 3), dtype=np.float32)])
    dN = torch.from_numpy(nodes.view(np.uint8)).cuda()
    dI = torch.from_numpy(prims.view(np.int32)).cuda()
    dB = torch.from_numpy(boxes).cuda()
    bvh = cq.BVH3f(dN.data_ptr(), len(nodes), dI.data_ptr(), len(prims))
    assert cq.lib().cubql_refit_f3(C.byref(bvh), C.c_void_p(dB.data_ptr()),
                                   C.c_void_p(torch.cuda.current_stream().cuda_stream), None) == 0
    torch.cuda.synchronize()
    got = dN.cpu().numpy().view(nodes.dtype)
    want_lo, want_hi = _expected(nodes, prims, boxes)
    for i in want_lo:
        assert np.array_equal(got["lo"][i], want_lo[i]) and np.array_equal(got["hi"][i], want_hi[i]), i
