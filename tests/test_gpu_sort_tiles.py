"""Radix sort at the edges of its tiles and of the step from small to large
tiles (2^21 pairs), for few and many key bits, against a stable argsort."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

SMALL, LARGE32, LARGE64, STEP = 512 * 8, 512 * 20, 512 * 16, 1 << 21


@pytest.mark.parametrize("bits,n", [(b, n) for b in (24, 47) for n in (2, 63, SMALL - 1, SMALL, SMALL + 1, 3 * SMALL + 7,
                                                                      STEP - 1, STEP, STEP + 1)]
                         + [(24, 206 * LARGE32 - 1), (24, 206 * LARGE32 + 1), (47, 257 * LARGE64 - 1),
                            (47, 257 * LARGE64 + 1)])
def test_sort_tile_edges(bits, n):
    import cubql_amd as cq
    print(f"[gpu] sort {bits} bits, {n} pairs", flush=True)
    rng = np.random.default_rng(n)
    k = rng.integers(0, 1 << bits, size=n, dtype=np.uint64)
    k[rng.random(n) < 0.2] = k[0]  # equal keys across tiles keep their order
    k = k.astype(np.uint32) if bits <= 32 else k
    v = rng.integers(0, 1 << 31, size=n, dtype=np.int64).astype(np.int32)
    kt = torch.from_numpy(k.view(np.int32 if bits <= 32 else np.int64)).cuda()
    vt = torch.from_numpy(v).cuda()
    cq.radix_sort_pairs(kt, vt, bits)
    order = np.argsort(k, kind="stable")
    assert np.array_equal(kt.cpu().numpy().view(k.dtype), k[order])
    assert np.array_equal(vt.cpu().numpy(), v[order])
