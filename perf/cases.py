"""The workloads this library's speed is judged by.

Twelve listed cases cover the work a program has the library do through its
Python entry points -- builds, point, kNN and triangle queries with their
adjoints, refits, box queries and the batched Chamfer path -- from calls of
a few thousand points, where launches and host time count, to ten million.
draw() gives further cases of the same kinds and ranges.

kind     one pass
build    a BVH over n prim boxes by one of the builders
match    a BVH over a cloud, then the closest point for every query (the
         correspondence step of a registration loop, clouds new each step)
fcp      closest points on a tree at hand
knn      k nearest neighbours on a tree at hand or rebuilt in the pass, with
         or without the adjoint
tri      closest triangles of a mesh, and the adjoint of the distances
collide  refit of a tree to moved boxes, then every box's overlaps
chamfer  bidirectional closest points and Chamfer adjoint of many cloud pairs
"""
from __future__ import annotations

import math

import torch

import cubql_amd as cq

DEV = "cuda"


# ------------------------------------------------------------------- cases

def listed():
    return [
        # the smallest calls: scan matching of one sparse lidar sweep, closest
        # points beyond the correspondence radius rejected
        {"name": "match_3k", "kind": "match", "n": 3001, "nq": 2777, "leaf": 8, "radius": 0.2},
        # an ordinary registration step: 100,000 points against 100,000
        {"name": "match_100k", "kind": "match", "n": 100000, "nq": 100000, "leaf": 8, "radius": math.inf},
        # the default builder over a large scan
        {"name": "build_median_10m", "kind": "build", "method": "median", "data": "uniform", "n": 10000000,
         "leaf": 8},
        # a fast rebuild each frame of a particle simulation
        {"name": "build_radix_3m", "kind": "build", "method": "radix", "data": "uniform", "n": 3000017,
         "leaf": 8},
        # a high-quality build over a mesh that is queried many times
        {"name": "build_sah_1.3m", "kind": "build", "method": "sah", "data": "mesh", "n": 1313006, "leaf": 4},
        # picking on a scene at hand: the smallest query batch
        {"name": "fcp_1k_of_1m", "kind": "fcp", "data": "uniform", "n": 1000000, "nq": 1000, "leaf": 8,
         "radius": math.inf},
        # resampling a scan onto another of the same size
        {"name": "fcp_10m", "kind": "fcp", "data": "uniform", "n": 10000000, "nq": 10000000, "leaf": 8,
         "radius": math.inf},
        # neighbourhoods of a sample of a large scan
        {"name": "knn8_1m_of_10m", "kind": "knn", "data": "uniform", "n": 10000000, "nq": 1000000, "k": 8,
         "leaf": 8, "rebuild": False, "backward": False},
        # a training step on clustered points with outliers, which move each
        # step: robust rebuild, neighbour distances and their gradients
        {"name": "knn16_mixture_grad_2m", "kind": "knn", "data": "mixture", "n": 2000000, "nq": 2000000,
         "k": 16, "leaf": 8, "rebuild": True, "backward": True},
        # a training step of a mesh fit: distances of samples to the mesh and their gradients
        {"name": "tri_grad_4m", "kind": "tri", "n": 1313006, "nq": 4000000, "leaf": 4},
        # one step of a simulation's broad phase: moved boxes, refit, overlapping pairs
        {"name": "collide_1m", "kind": "collide", "n": 1000003, "leaf": 4, "keep": 16},
        # a training step over a batch of point clouds of very different sizes
        {"name": "chamfer_4096", "kind": "chamfer", "clouds": 4096, "lo": 64, "hi": 65536, "leaf": 16,
         "graph": True},
    ]


def _log(rng, lo, hi):
    """A whole number spread over [lo, hi] by its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["match", "build", "build", "fcp", "knn", "tri", "collide", "chamfer"])
    if kind == "match":
        return {"kind": kind, "n": _log(rng, 1000, 300000), "nq": _log(rng, 1000, 300000),
                "leaf": rng.choice([4, 8, 16]), "radius": rng.choice([math.inf, 0.2])}
    if kind == "build":
        method, data, most = rng.choice([("median", "uniform", 10000000), ("median", "mesh", 2000000),
                                         ("radix", "uniform", 10000000), ("radix30", "uniform", 10000000),
                                         ("sah", "mesh", 1313006)])
        return {"kind": kind, "method": method, "data": data, "n": _log(rng, 2000, most),
                "leaf": rng.choice([2, 4, 8])}
    if kind == "fcp":
        data = rng.choice(["uniform", "uniform", "mixture"])
        most = 10000000 if data == "uniform" else 2000000
        return {"kind": kind, "data": data, "n": _log(rng, 100000, most), "nq": _log(rng, 1000, most),
                "leaf": rng.choice([4, 8]), "radius": rng.choice([math.inf, 0.05])}
    if kind == "knn":
        data = rng.choice(["uniform", "mixture"])
        most = 10000000 if data == "uniform" else 2000000
        return {"kind": kind, "data": data, "n": _log(rng, 100000, most), "nq": _log(rng, 10000, 1000000),
                "k": rng.choice([3, 5, 8, 10, 16]), "leaf": 8, "rebuild": rng.random() < 0.5, "backward": rng.random() < 0.5}
    if kind == "tri":
        return {"kind": kind, "n": _log(rng, 20000, 1313006), "nq": _log(rng, 20000, 4000000),
                "leaf": rng.choice([4, 8])}
    if kind == "collide":
        return {"kind": kind, "n": _log(rng, 10000, 1000003), "leaf": rng.choice([4, 8]),
                "keep": rng.choice([8, 16, 32])}
    return {"kind": kind, "clouds": _log(rng, 64, 2048), "lo": 64, "hi": rng.choice([2048, 16384, 65536]),
            "leaf": rng.choice([8, 16]), "graph": rng.random() < 0.5}


# ------------------------------------------------------------------ inputs

def _gen(seed, salt=0):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 64 + salt)
    return g


def _uniform(n, g, lo=0.0, hi=1.0):
    return torch.rand((n, 3), generator=g, device=DEV) * (hi - lo) + lo


def _mixture(n, g, mix_seed):
    """64 Gaussian clusters of very different widths in a box of side 2000
    (the mixture from mix_seed), 1% of the points on a sphere of radius 1e6."""
    m = _gen(mix_seed, 63)
    centre = torch.rand((64, 3), generator=m, device=DEV) * 2e3 - 1e3
    sigma = 10.0 ** (-4.0 + 3.0 * torch.rand((64, 1), generator=m, device=DEV))
    which = torch.randint(64, (n,), generator=g, device=DEV)
    normal = torch.randn((n, 3), generator=g, device=DEV)
    far = torch.rand(n, generator=g, device=DEV) < 0.01
    p = centre[which] + sigma[which] * normal
    out = normal * (1e6 / normal.norm(dim=1, keepdim=True).clamp_min(1e-20))
    return torch.where(far[:, None], out, p).contiguous()


def _points(data, n, g, seed):
    return _uniform(n, g) if data == "uniform" else _mixture(n, g, seed)


def _mesh(n, g):
    """A bumpy torus of about n triangles: (triangles [n,3] int32, vertices)."""
    nv = max(8, int(round(math.sqrt(n / 3.2))))
    nu = -(-n // (2 * nv))
    iu = torch.arange(nu, device=DEV)
    iv = torch.arange(nv, device=DEV)
    u, v = torch.meshgrid(iu * (2 * math.pi / nu), iv * (2 * math.pi / nv), indexing="ij")
    r = 0.4 + 0.01 * torch.randn((nu, nv), generator=g, device=DEV)
    ring = 1.0 + r * torch.cos(v)
    verts = torch.stack([ring * torch.cos(u), ring * torch.sin(u), r * torch.sin(v)], -1).reshape(-1, 3)
    a = (iu[:, None] * nv + iv[None, :]).reshape(-1)
    b = (((iu + 1) % nu)[:, None] * nv + iv[None, :]).reshape(-1)
    c = (((iu + 1) % nu)[:, None] * nv + ((iv + 1) % nv)[None, :]).reshape(-1)
    d = (iu[:, None] * nv + ((iv + 1) % nv)[None, :]).reshape(-1)
    tris = torch.stack([torch.stack([a, b, c], 1), torch.stack([a, c, d], 1)], 1).reshape(-1, 3)
    return tris[:n].to(torch.int32).contiguous(), verts.float().contiguous()


def _clouds(clouds, lo, hi, g, side):
    """(points, offsets): cloud sizes log-uniform in [lo, hi] (the case's,
    whatever the seed), each cloud a Gaussian blob of its own scale in
    [0.1, 10]."""
    u = torch.rand(clouds, generator=_gen(clouds, side), device=DEV, dtype=torch.float64)
    size = torch.exp(math.log(lo) + u * (math.log(hi + 1) - math.log(lo))).floor().long().clamp(lo, hi)
    off = torch.zeros(clouds + 1, dtype=torch.int32, device=DEV)
    off[1:] = size.cumsum(0)
    scale = 0.1 + 9.9 * torch.rand(clouds, generator=g, device=DEV)
    n = int(off[-1])
    return torch.randn((n, 3), generator=g, device=DEV) * scale.repeat_interleave(size)[:, None], off


def _config(case):
    if case.get("method") == "sah":
        return cq.BuildConfig(makeLeafThreshold=case["leaf"], maxAllowedLeafSize=case["leaf"])
    return cq.BuildConfig(makeLeafThreshold=case["leaf"])


def _sqr(radius):
    return radius * radius if math.isfinite(radius) else math.inf


_BUILDERS = {"median": cq.gpuBuilder, "radix": cq.cuda.radixBuilder, "radix30": cq.cuda.radix30Builder,
             "sah": cq.cuda.sahBuilder}


def prepare(case, seed):
    kind, g = case["kind"], _gen(seed)
    s = {"kind": kind, "cfg": _config(case), "mem": cq.TorchMemory(torch.device(DEV, torch.cuda.current_device()))}
    if kind == "build":
        s["build"] = _BUILDERS[case["method"]]
        # One scene for all seeds, which give the prims' order and the unit
        # of length (a power of two), so that every seed's tree has the same
        # number of nodes.
        base, unit = _gen(case["n"], 3), 2.0 ** (int(seed) % 7 - 3)
        if case["data"] == "mesh":
            tris, verts = _mesh(case["n"], base)
            first = int(torch.randint(case["n"], (1,), generator=g, device=DEV))
            s["boxes"] = cq.triangles.boxes(tris.roll(first, 0).contiguous(), verts * unit)
        else:
            p = _points(case["data"], case["n"], base, case["n"])
            order = torch.randperm(case["n"], generator=g, device=DEV)
            s["boxes"] = cq.points_to_boxes(p[order] * unit)
    elif kind == "match":
        s["points"], s["queries"] = _match_inputs(case, g)
        s["r2"] = _sqr(case["radius"])
    elif kind in ("fcp", "knn"):
        s["points"] = _points(case["data"], case["n"], g, seed)
        s["queries"] = _points(case["data"], case["nq"], g, seed)
        s["build"] = cq.gpuBuilder if case["data"] == "uniform" else cq.cuda.rebinRadixBuilder
        if not case.get("rebuild"):
            s["bvh"] = s["build"](cq.points_to_boxes(s["points"]), s["cfg"])
        if kind == "fcp":
            s["r2"] = _sqr(case["radius"])
        else:
            s["k"] = case["k"]
            if case["backward"]:
                s["grad"] = torch.rand((case["nq"], case["k"]), generator=g, device=DEV)
    elif kind == "tri":
        s["tris"], s["verts"] = _mesh(case["n"], g)
        t = torch.randint(case["n"], (case["nq"],), generator=g, device=DEV)
        w = torch.rand((case["nq"], 3), generator=g, device=DEV)
        w = w / w.sum(1, keepdim=True)
        q = (s["verts"][s["tris"][t].long()] * w[:, :, None]).sum(1)
        s["queries"] = (q + 0.05 * torch.randn((case["nq"], 3), generator=g, device=DEV)).contiguous()
        s["grad"] = torch.rand(case["nq"], generator=g, device=DEV)
        cfg = cq.BuildConfig(makeLeafThreshold=case["leaf"], maxAllowedLeafSize=case["leaf"])
        s["bvh"] = cq.cuda.sahBuilder(cq.triangles.boxes(s["tris"], s["verts"]), cfg)
    elif kind == "collide":
        # boxes of the mean spacing, some longer; the tree is that of the
        # step before (one for all seeds, which give the move)
        step, base = case["n"] ** (-1.0 / 3.0), _gen(case["n"], 3)
        centre = _uniform(case["n"], base)
        half = step * (0.15 + 0.7 * torch.rand((case["n"], 3), generator=base, device=DEV) ** 2)
        s["bvh"] = cq.gpuBuilder(torch.cat([centre - half, centre + half], 1).contiguous(), s["cfg"])
        centre = centre + 0.3 * step * torch.randn((case["n"], 3), generator=g, device=DEV)
        s["boxes"] = torch.cat([centre - half, centre + half], 1).contiguous()
        s["keep"] = case["keep"]
    else:
        src, so = _clouds(case["clouds"], case["lo"], case["hi"], g, 1)
        tgt, to = _clouds(case["clouds"], case["lo"], case["hi"], g, 2)
        s["batch"] = cq.ChamferBatch(src, so, tgt, to, cq.BatchParams(leafSize=case["leaf"]))
        s["graph"] = case["graph"]
        if case["graph"]:
            s["batch"].capture()
    return s


def _match_inputs(case, g):
    """A cloud on a bumpy shell and queries from another, slightly moved, view of it."""
    def shell(n):
        d = torch.randn((n, 3), generator=g, device=DEV)
        d = d / d.norm(dim=1, keepdim=True).clamp_min(1e-20)
        return d * (1.0 + 0.1 * torch.sin(7 * d[:, :1]) + 0.002 * torch.randn((n, 1), generator=g, device=DEV))
    return shell(case["n"]).contiguous(), (shell(case["nq"]) + 0.02).contiguous()


# -------------------------------------------------------------------- pass

def _tree(bvh):
    """A tree's arrays: boxes, offset and count words, prim order."""
    nodes = bvh.nodes_tensor()
    return {"boxes": nodes[:, :6], "words": nodes[:, 6:].view(torch.int64), "prims": bvh.prim_ids_tensor()}


def run(s):
    kind = s["kind"]
    if kind == "build":
        return _tree(s["build"](s["boxes"], s["cfg"], mem=s["mem"]))
    if kind == "match":
        bvh = cq.gpuBuilder(cq.points_to_boxes(s["points"]), s["cfg"], mem=s["mem"])
        ids, d2 = cq.points.findClosest(bvh, s["points"], s["queries"], s["r2"])
        return {"ids": ids, "d2": d2}
    if kind == "fcp":
        ids, d2 = cq.points.findClosest(s["bvh"], s["points"], s["queries"], s["r2"])
        return {"ids": ids, "d2": d2}
    if kind == "knn":
        bvh = s.get("bvh")
        if bvh is None:
            bvh = s["build"](cq.points_to_boxes(s["points"]), s["cfg"], mem=s["mem"])
        ids, d2, found = cq.points.findKNN(bvh, s["points"], s["queries"], s["k"])
        out = {"ids": ids, "d2": d2, "found": found}
        if "bvh" not in s:
            # (the rebin builder does not fix the numbering of its nodes)
            out["prims"] = bvh.prim_ids_tensor()
        if "grad" in s:
            gq = torch.empty_like(s["queries"])
            gp = torch.zeros_like(s["points"])
            cq.points_backward(s["points"], s["queries"], ids, s["grad"], gq, gp, mem=s["mem"])
            out.update(grad_queries=gq, grad_points=gp)
        return out
    if kind == "tri":
        ids, d2, cp = cq.triangles.findClosest(s["bvh"], s["tris"], s["verts"], s["queries"])
        gq = torch.empty_like(s["queries"])
        gv = torch.zeros_like(s["verts"])
        cq.triangles.backward(s["tris"], s["verts"], s["queries"], ids, s["grad"], gq, gv)
        return {"ids": ids, "d2": d2, "closest": cp, "grad_queries": gq, "grad_verts": gv}
    if kind == "collide":
        cq.refit(s["bvh"], s["boxes"])
        ids, counts = cq.fixedBoxQuery.forEachPrim(s["bvh"], s["boxes"], s["boxes"], s["keep"])
        return {"tree": _tree(s["bvh"]), "ids": ids, "counts": counts}
    b = s["batch"]
    b.replay() if s["graph"] else b.run()
    return {"src_nn": b.src_nn, "src_d2": b.src_d2, "tgt_nn": b.tgt_nn, "tgt_d2": b.tgt_d2, "loss": b.loss,
            "grad_src": b.grad_src, "grad_tgt": b.grad_tgt}


# ------------------------------------------------------- least work, 64 bits

def _tree_bytes(n, leaf):
    """Nodes (about 2.9 n / leaf of 32 bytes) and prim order."""
    return 32.0 * 2.9 * n / leaf + 4.0 * n


def _touched(n, leaf, nq, prim):
    """What nq queries cannot do without of a tree and its prims: all of it,
    or one path and one leaf each where that is less."""
    path = 64.0 * max(1.0, math.log2(max(2.0, n / leaf))) + leaf * (prim + 4.0)
    return min(_tree_bytes(n, leaf) + prim * n, nq * path)


def work(case):
    """Bytes of one pass with each input read once and each output written
    once; the arithmetic of one descent per query."""
    kind = case["kind"]
    if kind == "chamfer":
        mean = (case["hi"] - case["lo"]) / math.log(case["hi"] / case["lo"])
        n = case["clouds"] * mean
        return {"bytes": 2 * n * (12 + 4 + 4 + 12), "flops": 2 * n * 40.0 * math.log2(max(2.0, mean / case["leaf"]))}
    n, leaf = case["n"], case["leaf"]
    depth = max(1.0, math.log2(max(2.0, n / leaf)))
    if kind == "build":
        return {"bytes": 24.0 * n + _tree_bytes(n, leaf), "flops": 6.0 * n * depth}
    if kind == "match":
        nq = case["nq"]
        return {"bytes": 12.0 * n + 12.0 * n + 20.0 * nq, "flops": 6.0 * n * depth + 40.0 * nq * depth}
    if kind == "collide":
        return {"bytes": 24.0 * n + 2 * _tree_bytes(n, leaf) + (4.0 * case["keep"] + 4.0) * n,
                "flops": 40.0 * n * depth}
    nq = case["nq"]
    if kind == "fcp":
        return {"bytes": 20.0 * nq + _touched(n, leaf, nq, 12.0), "flops": 40.0 * nq * depth}
    if kind == "knn":
        k = case["k"]
        b = (16.0 + 8.0 * k) * nq + _touched(n, leaf, nq, 12.0)
        if case["rebuild"]:
            b += 12.0 * n + 4.0 * n
        if case["backward"]:
            b += (24.0 + 8.0 * k) * nq + 24.0 * n
        return {"bytes": b, "flops": 40.0 * nq * depth + 8.0 * nq * k}
    return {"bytes": 32.0 * nq + _touched(n, leaf, nq, 18.0) + (12.0 + 4.0 + 4.0 + 12.0) * nq + 6.0 * n * 2,
            "flops": 40.0 * nq * depth + 100.0 * nq}


_PAIRS = 3e10  # query-point pairs that 64-bit brute force goes through in seconds


def exact(case, seed):
    """Squared distances (and the query gradient) by brute force in 64 bits
    where there are few enough pairs; ids and trees have no such value."""
    kind = case["kind"]
    if kind == "match" and case["n"] * case["nq"] <= _PAIRS:
        p, q = _match_inputs(case, _gen(seed))
        d2 = _nearest(p, q, 1)[0][:, 0]
        r2 = _sqr(case["radius"])
        return {"ids": None, "d2": torch.where(d2 < r2, d2, math.inf) if math.isfinite(r2) else d2}
    if kind in ("fcp", "knn") and case["data"] == "uniform" and case["n"] * case["nq"] <= _PAIRS:
        g = _gen(seed)
        p, q = _uniform(case["n"], g), _uniform(case["nq"], g)
        if kind == "fcp":
            d2 = _nearest(p, q, 1)[0][:, 0]
            r2 = _sqr(case["radius"])
            return {"ids": None, "d2": torch.where(d2 < r2, d2, math.inf) if math.isfinite(r2) else d2}
        d2, ids = _nearest(p, q, case["k"])
        out = {"ids": None, "d2": d2, "found": None}
        if case["rebuild"]:
            out["prims"] = None
        if case["backward"]:
            grad = torch.rand((case["nq"], case["k"]), generator=g, device=DEV).double()
            diff = q.double()[:, None, :] - p.double()[ids]
            term = grad[:, :, None] * diff / d2.sqrt()[:, :, None]
            gp = torch.zeros((case["n"], 3), dtype=torch.float64, device=DEV)
            gp.index_add_(0, ids.reshape(-1), -term.reshape(-1, 3))
            out.update(grad_queries=term.sum(1), grad_points=gp)
        return out
    return None


def _nearest(p, q, k):
    p, q = p.double(), q.double()
    rows = max(1, int(2e8 // p.shape[0]))
    d, i = [], []
    for b in range(0, q.shape[0], rows):
        x = q[b:b + rows]
        m = sum((x[:, j, None] - p[None, :, j]) ** 2 for j in range(3))
        v, w = (m.min(1, keepdim=True) if k == 1 else m.topk(k, dim=1, largest=False, sorted=True))
        d.append(v)
        i.append(w)
    return torch.cat(d), torch.cat(i)
