"""Loss and adjoint of the batched Chamfer path where a workgroup's chunk of
queries (2048) and its window of neighbour slots (2560) have their edges:
clouds that end within, at and just past a chunk, many clouds in one chunk,
targets far more numerous than the window, targets that collect a whole
cloud, empty clouds, and each output left out.  FP64 evaluation of the
returned neighbours; the gradients by the rule of gradtol.py, the loss within
(terms + 8) roundings of itself (a distance carries less than eight, the sum
over n terms in any order n - 1)."""
import numpy as np
import pytest
import torch

from gradtol import EPS, check_chamfer_grads

pytestmark = pytest.mark.gpu

SIZES = {
    "one_chunk": ([2048], [2048]),
    "chunk_edges": ([2047, 2049, 1, 4096, 63], [2561, 2560, 2559, 1, 5000]),
    "small_clouds": ([3, 64, 1, 65, 0, 17] * 60, [64, 5, 2, 1, 9, 0] * 60),
    "window": ([3000, 40000, 500], [60000, 30, 20000]),
    "point_targets": ([9000, 1], [1, 9000]),
}


@pytest.mark.parametrize("kind", sorted(SIZES))
def test_batch_backward(oracle_mod, kind):
    import cubql_amd as cq
    print(f"[gpu] batch backward {kind}", flush=True)
    rng = np.random.default_rng(len(kind))
    so, to = (np.concatenate([[0], np.cumsum(n)]) for n in SIZES[kind])
    S, T = (rng.random((o[-1], 3)).astype(np.float32) for o in (so, to))
    d = [torch.from_numpy(x).cuda() for x in (S, so.astype(np.int32), T, to.astype(np.int32))]
    B = cq.ChamferBatch(*d).run()
    nn_s, nn_t, gs, gt, loss = (x.cpu().numpy() for x in (B.src_nn, B.tgt_nn, B.grad_src, B.grad_tgt, B.loss))
    for c in range(len(so) - 1):
        (sb, se), (tb, te) = so[c:c + 2], to[c:c + 2]
        if sb == se or tb == te:
            assert loss[c] == 0 and not gs[sb:se].any() and not gt[tb:te].any()
            continue
        a, b, ls, lt = S[sb:se], T[tb:te], nn_s[sb:se] - tb, nn_t[tb:te] - sb
        check_chamfer_grads(oracle_mod, a, b, ls, lt, gs[sb:se], gt[tb:te], label=f"{kind} {c}")
        l64 = (np.linalg.norm(a.astype(np.float64) - b[ls].astype(np.float64), axis=1).mean()
               + np.linalg.norm(b.astype(np.float64) - a[lt].astype(np.float64), axis=1).mean())
        assert abs(loss[c] - l64) <= (len(a) + len(b) + 8) * EPS * l64
    # outputs left out one at a time: the rest as before, up to the order of
    # the sums (terms of at most 1 / cloud size each)
    for out in ("grad_src", "grad_tgt", "loss"):
        P = cq.ChamferBatch(*d)
        for t in (P.grad_src, P.grad_tgt, P.loss):
            t.fill_(7.0)
        setattr(P, out, None)
        P.run()
        for name, ref in (("grad_src", gs), ("grad_tgt", gt), ("loss", loss)):
            if name != out:
                got = getattr(P, name).cpu().numpy()
                assert np.allclose(got, ref, rtol=1e-4, atol=1e-5), (out, name)
