"""SAH builds where the binning and its sums change form: sizes on both sides
of a binning tile (1024 prims here, more from 262144 on) and of several, of a small node (256) and
of a row of lanes (16 prims), bin counts on both sides of 16, sorted prims
(neighbours share bins), coordinates of both zeros, infinite extents, and
copies (no plane separates them).  The tree equals the oracle's."""
import numpy as np
import pytest

from test_gpu_sah import _check_equal, _random_boxes, cq  # noqa: F401

pytestmark = pytest.mark.gpu
F32 = np.float32


@pytest.mark.parametrize("kind", ["random", "sorted", "zeros", "infinite", "copies"])
@pytest.mark.parametrize("n,nb,T,cap", [(5, 16, 1, 100), (16, 2, 1, 100), (17, 16, 2, 100), (33, 16, 4, 4),
                                        (64, 3, 1, 2), (255, 16, 1, 100), (256, 15, 1, 3), (257, 17, 1, 100),
                                        (700, 16, 16, 100), (1024, 16, 2, 100), (1025, 16, 2, 100),
                                        (3000, 16, 4, 5), (8192, 16, 4, 100), (8193, 7, 3, 8),
                                        (65536, 16, 4, 100), (65537, 32, 4, 100), (90000, 16, 1, 1 << 15)])
def test_sah_equals_oracle(cq, oracle_mod, kind, n, nb, T, cap):  # noqa: F811
    print(f"[gpu] sah {kind}: {n} prims, {nb} bins, T {T}, cap {cap}", flush=True)
    B = _random_boxes(n, seed=n + nb)
    rng = np.random.default_rng(n)
    if kind == "sorted":
        B = B[np.argsort(B[:, 0])]
    elif kind == "zeros":
        # a plane of boxes at either zero, half of them flat
        B[:, 2] = np.where(rng.random(n) < 0.5, F32(0.0), F32(-0.0))
        B[:, 5] = np.where(rng.random(n) < 0.5, B[:, 2], F32(0.0))
    elif kind == "infinite":
        B[::5, 4] = np.inf
    elif kind == "copies":
        B = B[rng.integers(0, max(1, n // 9), n)]
    _check_equal(cq, oracle_mod, B, T, nb, cap)
