"""Device memory of a rebin build: scratch is taken before the nodes and nothing
after them, for shallow trees and for deep ones, so that a build needs no more
than its scratch and the tree whatever the input."""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("deep", [False, True])
@pytest.mark.parametrize("n,T", [(3000, 1), (200000, 8)])
def test_nodes_are_the_last_allocation(oracle_mod, deep, n, T):
    import cubql_amd as cq
    print(f"[gpu] rebin memory, {n} prims, deep {deep}", flush=True)
    P = np.random.default_rng(n).random((n, 3))
    if deep:
        P = P ** 20
        P[::101] *= 1000
    B = np.hstack([P, P]).astype(np.float32)
    mem = cq.TorchMemory(torch.device("cuda", torch.cuda.current_device()))
    sizes = []

    def malloc(pp, size, stream, user):
        sizes.append(size)
        return mem._m(pp, size, stream, user)

    cb = cq._MALLOC_CB(malloc)
    mem.resource = cq.MemResource(cb, mem._f, None)
    bvh = cq.cuda.rebinRadixBuilder(torch.from_numpy(B).cuda(), cq.BuildConfig(makeLeafThreshold=T), mem=mem)
    assert sizes[-1] == 32 * bvh.numNodes
    tree = oracle_mod.Tree(cq.nodes_to_numpy(bvh).view(oracle_mod.NODE_DTYPE),
                           bvh.prim_ids_tensor().cpu().numpy().view(np.uint32))
    assert oracle_mod.check_tree(tree, B, T)[0] == 0
