"""The work that a user of the smoothing library has it do, as cases that can be timed and compared.

Every case goes through the public Python classes (multigpuegtsmoothing_amd.egt): a whole smoothing call on a point
cloud, on a mesh or on a batch of clouds, a neighbour search whose rows stay on the GPU, a query search against a
reference cloud that the program keeps, and the training of the search-radius model. Inputs come from the seed
alone and are drawn on the GPU, from the same families as the seeded clouds of multigpuegtsmoothing_amd.datasets.

kind      what one run() is
cloud     GridStructure, [proposal], kNN, [EGG + Taubin], [normals], output points, close
mesh      GridMeshCuda from host arrays, one-ring rows, EGG + Taubin, [normals], output points, close
batch     BatchGrid, [proposal], kNN with a k per cloud, EGG + Taubin, output points, close
knn       GridStructure, kNN; the rows and the sorted-to-original map stay on the GPU
query     GRIDCUDAKNNCompact of new queries against a kept reference handle
train     a new RadiusModel trained on a kept cloud
"""
import math

import numpy as np
import torch

from multigpuegtsmoothing_amd import egt as E

LAMBDA, MU = 0.5, -0.53


def listed():
    return [
        # nearest reference point of a handful of tracked points: the smallest call, all latency
        {"name": "query_300", "kind": "query", "shape": "sphere", "n": 100_000, "nq": 300, "k": 1, "host": True},
        # a second scan of the same surface looked up in the first (registration), rows stay on the GPU
        {"name": "query_4m", "kind": "query", "shape": "torus", "n": 4_000_000, "nq": 4_000_000, "k": 16,
         "host": False},
        # a small object, a few smoothing steps, normals: interactive use
        {"name": "cloud_1500", "kind": "cloud", "shape": "sphere", "n": 1_500, "k": 8, "iters": 20, "normals": True,
         "host": True, "start_level": 0, "lanes": 1, "learned": False, "regularized": False},
        # the command line's ordinary job: 100,000 noisy points of a sphere from host arrays, 150 iterations
        {"name": "cloud_100k", "kind": "cloud", "shape": "sphere", "n": 100_000, "k": 40, "iters": 150,
         "normals": False, "host": True, "start_level": 0, "lanes": 1, "learned": False, "regularized": False},
        # a scan of a million points (an odd number), short lists, light smoothing, normals
        {"name": "cloud_1m", "kind": "cloud", "shape": "torus", "n": 1_000_003, "k": 16, "iters": 50,
         "normals": True, "host": False, "start_level": 0, "lanes": 1, "learned": False, "regularized": False},
        # a large scan of uneven density, resident on the GPU, start level tuned once for such scans, normals
        {"name": "cloud_4m", "kind": "cloud", "shape": "torus", "n": 4_000_000, "k": 40, "iters": 300,
         "normals": True, "host": False, "start_level": 2, "lanes": 1, "learned": False, "regularized": False},
        # the largest single cloud: volumetric clusters and planes, the learned proposal as its tuner sets it
        {"name": "cloud_16m", "kind": "cloud", "shape": "mixture", "n": 16_000_000, "k": 40, "iters": 150,
         "normals": False, "host": False, "start_level": 0, "lanes": 1, "learned": True, "regularized": False},
        # neighbour lists alone at the longest k, a wave per query, for a consumer on the GPU
        {"name": "knn_4m", "kind": "knn", "shape": "mixture", "n": 4_000_000, "k": 64, "start_level": 0, "lanes": 64},
        # a closed triangle mesh of 655,200 vertices, 150 iterations, normals
        {"name": "mesh_655k", "kind": "mesh", "nu": 1_170, "nv": 560, "k": 40, "iters": 150, "normals": True,
         "alpha": 1e-8},
        # an uneven batch of scanned objects in one handle, mixed list lengths, learned proposal
        {"name": "batch_192", "kind": "batch", "count": 192, "lo": 5_000, "hi": 500_000, "iters": 100,
         "learned": True},
        # a batch of small objects
        {"name": "batch_24", "kind": "batch", "count": 24, "lo": 500, "hi": 5_000, "iters": 50, "learned": False},
        # training the radius model for a kind of cloud (plain search, features, forward, backward, Adam)
        {"name": "train_300k", "kind": "train", "shape": "torus", "n": 300_000, "k": 40, "epochs": 4},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["cloud"] * 6 + ["mesh", "batch", "batch", "knn", "knn", "query", "query", "train"])
    if kind == "cloud":
        n = _log(rng, 500, 6_000_000)
        return {"kind": kind, "shape": rng.choice(["sphere", "torus", "mixture"]), "n": n,
                "k": rng.choice([8, 12, 16, 24, 33, 40, 40, 64]), "iters": min(_log(rng, 5, 300), 600_000_000 // n),
                "normals": rng.random() < 0.5, "host": rng.random() < 0.5,
                "start_level": rng.choice([0, 0, E.START_LEVEL_OCCUPANCY]), "lanes": rng.choice([1, 1, 64]),
                "learned": n >= 50_000 and rng.random() < 0.3, "regularized": rng.random() < 0.1}
    if kind == "mesh":
        return {"kind": kind, "nu": _log(rng, 24, 1_200), "nv": _log(rng, 16, 560), "k": rng.choice([8, 16, 40]),
                "iters": _log(rng, 5, 150), "normals": rng.random() < 0.5, "alpha": rng.choice([1e-8, 0.65])}
    if kind == "batch":
        lo = _log(rng, 200, 5_000)
        return {"kind": kind, "count": _log(rng, 2, 64), "lo": lo, "hi": lo * rng.choice([4, 20, 60]),
                "iters": _log(rng, 5, 100), "learned": lo >= 2_000 and rng.random() < 0.5}
    if kind == "knn":
        return {"kind": kind, "shape": rng.choice(["sphere", "torus", "mixture"]), "n": _log(rng, 1_000, 4_000_000),
                "k": rng.choice([4, 8, 16, 24, 40, 56, 64]), "start_level": rng.choice([0, E.START_LEVEL_OCCUPANCY]),
                "lanes": rng.choice([1, 64])}
    if kind == "query":
        return {"kind": kind, "shape": rng.choice(["sphere", "torus", "mixture"]), "n": _log(rng, 5_000, 4_000_000),
                "nq": _log(rng, 100, 4_000_000), "k": rng.choice([1, 1, 8, 16, 40]), "host": rng.random() < 0.3}
    return {"kind": kind, "shape": rng.choice(["sphere", "torus"]), "n": _log(rng, 50_000, 400_000),
            "k": rng.choice([16, 40]), "epochs": rng.choice([1, 2, 4])}


# ---- inputs ---------------------------------------------------------------------------------------------------------


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _uniform(g, n, lo, hi):
    return torch.rand(n, generator=g, device="cuda", dtype=torch.float64) * (hi - lo) + lo


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float64)


def _sphere(n, g):
    """Unit sphere with isotropic noise of 0.005."""
    v = _normal(g, n, 3)
    return v / v.norm(dim=1, keepdim=True) + 0.005 * _normal(g, n, 3)


def _torus(n, g):
    """Torus R=1, r=0.3, density 1 to 10 along the major angle, noise 0.003."""
    m = int(2.3 * n) + 1_000
    t = _uniform(g, m, 0.0, 2.0 * math.pi)
    t = t[_uniform(g, m, 0.0, 10.0) < 1.0 + 4.5 * (1.0 - torch.cos(t))][:n]
    p = _uniform(g, m, 0.0, 2.0 * math.pi)
    p = p[_uniform(g, m, 0.0, 1.3) < 1.0 + 0.3 * torch.cos(p)][:n]
    w = 1.0 + 0.3 * torch.cos(p)
    return torch.stack([w * torch.cos(t), w * torch.sin(t), 0.3 * torch.sin(p)], 1) + 0.003 * _normal(g, n, 3)


def _rotation(r):
    q, rr = np.linalg.qr(r.standard_normal((3, 3)))
    return q * np.sign(np.diag(rr))


def _mixture(n, g):
    """12 anisotropic Gaussian clusters (axis ratios up to 20:1) and 4 noisy planar patches, in random order. The
    clusters' layout is one fixed scene (every seed draws other points of it), so passes on different seeds cost alike."""
    r = np.random.default_rng(4)
    w = np.exp(r.uniform(np.log(1.0), np.log(20.0), 16))
    counts = np.floor(w / w.sum() * n).astype(np.int64)
    counts[0] += n - counts.sum()
    parts = []
    for c in range(16):
        m = int(counts[c])
        centre, rot = r.uniform(-1, 1, 3), _rotation(r)
        if c < 12:
            scale = np.exp(r.uniform(np.log(0.02), np.log(0.3)))
            axes = scale * np.array([1.0, np.exp(r.uniform(np.log(1 / 20), 0)), np.exp(r.uniform(np.log(1 / 20), 0))])
            p = _normal(g, m, 3) * torch.from_numpy(axes).cuda()
        else:
            half = r.uniform(0.2, 0.8, 2)
            p = torch.stack([_uniform(g, m, -half[0], half[0]), _uniform(g, m, -half[1], half[1]),
                             0.002 * _normal(g, m)], 1)
        parts.append(p @ torch.from_numpy(rot.T.copy()).cuda() + torch.from_numpy(centre).cuda())
    return torch.cat(parts)[torch.randperm(n, generator=g, device="cuda")]


def _points(shape, n, seed):
    """(n, 3) float32 on the GPU."""
    g = _gen(seed)
    p = _sphere(n, g) if shape == "sphere" else _torus(n, g) if shape == "torus" else _mixture(n, g)
    return p.to(torch.float32)


def _split(p):
    out = tuple(p[:, i].contiguous() for i in range(3))
    torch.cuda.synchronize()  # the library runs on its own streams
    return out


def _host(xyz):
    return tuple(t.cpu().numpy() for t in xyz)


def _batch_sizes(count, lo, hi):
    """Sizes log-uniform in [lo, hi] and k from {16, 40, 64}, fixed by the case."""
    r = np.random.default_rng(5000 + count)
    sizes = np.floor(np.exp(r.uniform(np.log(lo), np.log(hi), count))).astype(np.int64)
    return sizes, r.choice(np.array([16, 40, 64], np.int32), count).astype(np.int32)


def _superquadrics(sizes, seed):
    """Superquadric surfaces (exponents in [0.3, 3]), one after another, each with noise of 1e-3 of its size."""
    r, g = np.random.default_rng(seed), _gen(seed)
    count, n = len(sizes), int(sizes.sum())
    cloud = torch.repeat_interleave(torch.arange(count, device="cuda"), torch.from_numpy(sizes).cuda())
    e = torch.from_numpy(r.uniform(0.3, 3.0, (count, 2))).cuda()[cloud]
    a_host = r.uniform(0.5, 2.0, (count, 3))
    a = torch.from_numpy(a_host).cuda()[cloud]
    eta, om = _uniform(g, n, -math.pi / 2, math.pi / 2), _uniform(g, n, -math.pi, math.pi)

    def sp(v, x):
        return torch.sign(v) * torch.abs(v) ** x

    ce, se = torch.cos(eta), torch.sin(eta)
    p = torch.stack([a[:, 0] * sp(ce, e[:, 0]) * sp(torch.cos(om), e[:, 1]),
                     a[:, 1] * sp(ce, e[:, 0]) * sp(torch.sin(om), e[:, 1]), a[:, 2] * sp(se, e[:, 0])], 1)
    p = p + 2e-3 * torch.from_numpy(a_host.max(1)).cuda()[cloud][:, None] * _normal(g, n, 3)
    return _split(p.to(torch.float32))


def _mesh(nu, nv, seed):
    """Closed triangle mesh of a torus (nu x nv vertices), vertices moved along the normal by U(-0.01, 0.01)."""
    r = np.random.default_rng(seed)
    iu, iv = np.meshgrid(np.arange(nu), np.arange(nv), indexing="ij")
    u, v = 2 * np.pi * iu.ravel() / nu, 2 * np.pi * iv.ravel() / nv
    rad = 0.4 + r.uniform(-0.01, 0.01, nu * nv)
    w = 1.0 + rad * np.cos(v)
    xyz = tuple(np.ascontiguousarray(t, np.float32) for t in (w * np.cos(u), w * np.sin(u), rad * np.sin(v)))
    at = lambda i, j: ((i % nu) * nv + j % nv).ravel()  # noqa: E731
    a, b, c, d = at(iu, iv), at(iu + 1, iv), at(iu, iv + 1), at(iu + 1, iv + 1)
    tri = np.concatenate([np.stack([a, b, d], 1), np.stack([a, d, c], 1)]).astype(np.uint32)
    return xyz, tri


def _model(shape, k, seed):
    """A radius model trained on a cloud of the same family."""
    with E.GridStructure(_split(_points(shape, 100_000, seed + 7)), 1, 1e-6, 1024, 4) as g:
        m = E.RadiusModel(seed=17)
        m.train(g, k, epochs=2)
    return m


def prepare(case, seed):
    kind = case["kind"]
    if kind == "cloud":
        xyz = _split(_points(case["shape"], case["n"], seed))
        s = dict(case, xyz=_host(xyz) if case["host"] else xyz)
        if case["learned"]:
            s["model"] = _model(case["shape"], case["k"], seed)
    elif kind == "mesh":
        xyz, tri = _mesh(case["nu"], case["nv"], seed)
        s = dict(case, xyz=xyz, tri=tri)
    elif kind == "batch":
        sizes, ks = _batch_sizes(case["count"], case["lo"], case["hi"])
        s = dict(case, sizes=sizes, ks=ks, xyz=_superquadrics(sizes, seed))
        if case["learned"]:
            ts, tk = _batch_sizes(12, 5_000, 20_000)
            m = E.RadiusModel(seed=13)
            with E.BatchGrid(ts, device=_superquadrics(ts, seed + 7)) as b:
                m.train(b, tk, epochs=2)
            s["model"] = m
    elif kind == "knn":
        s = dict(case, xyz=_split(_points(case["shape"], case["n"], seed)), grid=None)
    elif kind == "query":
        ref = _split(_points(case["shape"], case["n"], seed))
        q = _split(_points(case["shape"], case["nq"], seed + 1_000_003))
        s = dict(case, grid=E.GridStructure(ref, 1, 1e-6, 1024, 4), queries=_host(q) if case["host"] else q)
    else:
        ref = _split(_points(case["shape"], case["n"], seed))
        s = dict(case, seed=int(seed), grid=E.GridStructure(ref, 1, 1e-6, 1024, 4))
    return s


# ---- one pass -------------------------------------------------------------------------------------------------------


class _View:
    """Device memory of a handle as torch takes it, without a copy."""

    def __init__(self, ptr, shape):
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "typestr": "<i4", "version": 2}


def _device_ints(ptr, *shape):
    return torch.as_tensor(_View(ptr, shape), device="cuda")


def _finish(provider, normals):
    out = dict(zip("xyz", E.getOutputPoints(provider)))
    if normals:
        out["normals"] = list(E.Normal_CUDA(provider).GetNormals())
    provider.close()
    return out


def run(s):
    kind = s["kind"]
    if kind == "cloud":
        g = E.GridStructure(s["xyz"], 1, 1e-6, 1024, 4)
        if s["learned"]:
            s["model"].propose(g, s["k"])
            g.set_option(E.OPT_LEARNED_MODE, 3)
            g.set_option(E.OPT_LEARNED_LEVEL_OFFSET, 1)
        g.set_option(E.OPT_START_LEVEL, s["start_level"])
        g.set_option(E.OPT_KNN_LANES, s["lanes"])
        g.set_option(E.OPT_TAUBIN_REGULARIZED, int(s["regularized"]))
        g.GRIDCUDAKNNSELF_COMPACT(s["k"], 1e8)
        E.EGT_CUDA(g).PerformSmoothing(s["iters"], LAMBDA, MU, 0.65)
        return _finish(g, s["normals"])
    if kind == "mesh":
        m = E.GridMeshCuda(s["xyz"], s["tri"])
        m.GetNeighborsFromTriangles(s["k"])
        E.EGT_CUDA(m).PerformSmoothing(s["iters"], LAMBDA, MU, s["alpha"])
        return _finish(m, s["normals"])
    if kind == "batch":
        b = E.BatchGrid(s["sizes"], device=s["xyz"])
        if s["learned"]:
            s["model"].propose(b, s["ks"])
            b.set_option(E.OPT_LEARNED_MODE, 3)
        b.knn(s["ks"])
        E.EGT_CUDA(b).PerformSmoothing(s["iters"], LAMBDA, MU, 0.65)
        return _finish(b, False)
    if kind == "knn":
        if s["grid"] is not None:  # the last pass's rows were views of its handle
            s["grid"].close()
        g = s["grid"] = E.GridStructure(s["xyz"], 1, 1e-6, 1024, 4)
        g.set_option(E.OPT_START_LEVEL, s["start_level"])
        g.set_option(E.OPT_KNN_LANES, s["lanes"])
        g.GRIDCUDAKNNSELF_COMPACT(s["k"], 1e8)
        return {"rows": _device_ints(g.GetKNNIndexesDevice(), s["n"], s["k"]),
                "original": _device_ints(g.GetOriginalRefIndexesDevice(), s["n"])}
    if kind == "query":
        g = s["grid"]
        g.GRIDCUDAKNNCompact(s["queries"], s["k"], 1e8)
        if s["host"]:
            return {"rows": g.GetKNNIndexesQuery()}
        ptr, nq, k = g.GetKNNIndexesQueryDevice()
        return {"rows": _device_ints(ptr, nq, k)}
    m = E.RadiusModel(seed=s["seed"])
    mse = m.train(s["grid"], s["k"], epochs=s["epochs"])
    out = {"params": m.get_params(), "mse": mse, "safety": m.safety, "bound_safety": m.bound_safety}
    m.close()
    return out


# ---- what a pass cannot do without ----------------------------------------------------------------------------------


def _smoothing_flops(n, k, iters):
    """The k distances, the filter's tests of each listed neighbour against half of the nearer ones (about 20
    operations each) and, per pass and kept neighbour (about 0.36 k of them on surfaces, at most 16), a distance, an
    exponential and three weighted sums."""
    kept = min(0.9 * k, max(6.0, 0.36 * k))
    return n * k * 8.0 + n * k * k * 0.5 * 20.0 + 2.0 * iters * n * kept * 20.0


def work(case):
    """Inputs read once, outputs written once, and the operations of the method itself."""
    kind = case["kind"]
    if kind == "cloud":
        n, k = case["n"], case["k"]
        return {"bytes": n * (24 + 12 * case["normals"]), "flops": _smoothing_flops(n, k, case["iters"])}
    if kind == "mesh":
        n = case["nu"] * case["nv"]
        return {"bytes": n * (24 + 24 + 12 * case["normals"]), "flops": _smoothing_flops(n, 6, case["iters"])}
    if kind == "batch":
        sizes, ks = _batch_sizes(case["count"], case["lo"], case["hi"])
        return {"bytes": float(sizes.sum()) * 24,
                "flops": sum(_smoothing_flops(float(n), int(k), case["iters"]) for n, k in zip(sizes, ks))}
    if kind == "knn":
        return {"bytes": case["n"] * (16 + 4 * case["k"]), "flops": case["n"] * case["k"] * 8.0}
    if kind == "query":
        return {"bytes": case["nq"] * (12 + 4 * case["k"]) + (0 if case["nq"] < case["n"] else 12 * case["n"]),
                "flops": case["nq"] * case["k"] * 8.0}
    # forward and backward of 28 -> 64 -> 64 -> 1, 3 x 2 operations a weight and sample
    return {"bytes": case["n"] * 12.0, "flops": case["epochs"] * case["n"] * 6.0 * (28 * 64 + 64 * 64 + 64)
            + case["n"] * case["k"] * 8.0}


# ---- the same in 64 bits ---------------------------------------------------------------------------------------------

EXACT_MOST = 130_000  # points of a cloud searched by brute force


def _knn64(p, k):
    """The k nearest other points by exact distance, nearest first; None where a distance comes near the reach at which
    the library's search rule may leave a row empty."""
    n = p.shape[0]
    out = torch.empty(n, k, dtype=torch.int64, device=p.device)
    step = max(1, min(n, 100_000_000 // n))
    for a in range(0, n, step):
        q = p[a:a + step]
        d = sum((q[:, i, None] - p[None, :, i]) ** 2 for i in range(3))
        d[torch.arange(len(q)), torch.arange(a, a + len(q))] = math.inf
        v, j = d.topk(k, dim=1, largest=False, sorted=True)
        if float(v[:, -1].max()) > 0.12 ** 2:
            return None
        out[a:a + step] = j
    return out


def _egg64(p, nb, alpha):
    """The elliptic Gabriel filter: slot j is dropped when a nearer listed neighbour lies inside the ellipsoid around the
    middle of the edge, semi-axis |edge| / 2 along it and alpha |edge| / 2 across it."""
    keep = nb >= 0
    k = nb.shape[1]
    step = max(1, 12_000_000 // (k * k))
    for a in range(0, p.shape[0], step):
        o, q = p[a:a + step, None, :], p[nb[a:a + step].clamp(min=0)]
        axis = q - o
        half = axis.norm(dim=2) / 2
        axis = axis / axis.norm(dim=2, keepdim=True).clamp(min=1e-300)
        mid = (q + o) / 2
        for j in range(1, k):
            rel = q[:, :j] - mid[:, j:j + 1]
            along = (rel * axis[:, j:j + 1]).sum(2)
            across = (rel * rel).sum(2) - along * along
            inside = along * along + across.clamp(min=0) / (alpha * alpha) < (half[:, j:j + 1] ** 2)
            inside &= nb[a:a + step, :j] >= 0
            keep[a:a + step, j] &= ~(inside.any(1) & (half[:, j] >= 1e-6))
    return keep


def _smooth64(xyz, nb, alpha, iters, regularized):
    """Normalization to the bounding cube, filter, Taubin passes, back to input units. nb: rows of neighbours, nearest
    first, -1 for none, or a function of the normalized points that gives them."""
    p = torch.stack([torch.as_tensor(t, device="cuda").double() for t in xyz], 1)
    lo, hi = float(p.min()) - 1e-6, float(p.max()) + 1e-6
    p = (p - lo) / (hi - lo)
    nb = nb(p) if callable(nb) else nb
    if nb is None:
        return None
    keep = _egg64(p, nb, alpha)
    at, keep = nb.clamp(min=0), keep.double()
    for scale in [LAMBDA, MU] * iters:
        d = p[at] - p[:, None, :]
        d2 = (d * d).sum(2)
        w = keep * ((1.0 / (d2 + 1e-8) if scale < 0 else torch.ones_like(d2)) if regularized else torch.exp(-d2))
        s = w.sum(1)
        s = torch.where(s == 0, torch.full_like(s, 1e-8), s)
        p = p + scale * (w[:, :, None] * d).sum(1) / s[:, None]
    p = p * (hi - lo) + lo
    return {c: p[:, i].cpu().numpy() for i, c in enumerate("xyz")}


def _ring64(xyz, tri, k):
    """One-ring rows of a closed mesh, nearest first."""
    t = torch.from_numpy(tri.astype(np.int64)).cuda()
    p = torch.stack([torch.from_numpy(c).cuda().double() for c in xyz], 1)
    n = p.shape[0]
    e = torch.cat([t[:, [0, 1]], t[:, [1, 2]], t[:, [2, 0]]])
    e = torch.unique(torch.cat([e, e.flip(1)]), dim=0)
    d = (p[e[:, 0]] - p[e[:, 1]]).norm(dim=1)
    order = torch.argsort(d, stable=True)
    order = order[torch.argsort(e[order, 0], stable=True)]
    e = e[order]
    first = torch.searchsorted(e[:, 0].contiguous(), torch.arange(n, device="cuda"))
    slot = torch.arange(len(e), device="cuda") - first[e[:, 0]]
    nb = torch.full((n, k), -1, dtype=torch.int64, device="cuda")
    in_row = slot < k
    nb[e[in_row, 0], slot[in_row]] = e[in_row, 1]
    return nb[:, :max(1, min(k, int(slot.max()) + 1))].contiguous()


def exact(case, seed):
    """Smoothed coordinates in 64 bits. Normals have no such value: their sign follows a spanning forest whose choices
    hang on the last bits; nor has a model after hundreds of steps. Rows are whole numbers and are compared as they are."""
    kind = case["kind"]
    if kind == "cloud" and case["n"] <= EXACT_MOST and case["shape"] != "mixture":
        s = prepare(dict(case, learned=False), seed)
        return _smooth64(s["xyz"], lambda p: _knn64(p, case["k"]), 0.65, case["iters"], case["regularized"])
    if kind == "mesh":
        s = prepare(case, seed)
        return _smooth64(s["xyz"], _ring64(s["xyz"], s["tri"], case["k"]), case["alpha"], case["iters"], False)
    return None
