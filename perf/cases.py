"""Performance cases of the KNN framework, timed through its public entry points.

Each case is one unit of work that a program using this package repeats: a query of a tree it
keeps, a query with its backward, a replay of a captured many-cloud step, or a rebuild of the tree
of a cloud that changed followed by a query.  Sizes come from the workloads of ``workloads.py`` and
``bench.py`` (plain_cpu, plain_gpu, the reference's default depth, diff_sphere, d8_mixture,
fp64_normal, batch_clouds) and, where those leave a gap (single lookups, d = 2, k > 32, rebuilds),
are round generic ones.

Fields of a case: ``op`` ("query", "grad", "batch", "rebuild"), ``dims``, ``dtype``, ``n`` reference
points, ``q`` queries, ``k``, ``cloud`` (the distribution), ``levels`` ("auto" or "default", the
reference's rule) and ``tie`` (tie policy); "batch" has ``clouds``, ``n_min`` and ``n_max`` instead of
``n``, ``q`` and ``k``.
"""
import math

import numpy as np
import torch

import torch_kdtree_amd as tk

_DTYPES = {"float32": torch.float32, "float64": torch.float64}


def _case(name, op, dims, dtype, n, q, k, cloud, levels="auto", tie="reference"):
    c = dict(op=op, dims=dims, dtype=dtype, n=n, q=q, k=k, cloud=cloud, levels=levels, tie=tie)
    if name:
        c["name"] = name
    return c


def _batch(name, clouds, n_min, n_max):
    c = dict(op="batch", dims=3, dtype="float32", clouds=clouds, n_min=n_min, n_max=n_max)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # a handful of lookups in a map, as a controller or a picking tool makes them: latency
        _case("lookup", "query", 3, "float32", 100_000, 16, 8, "uniform"),
        # the reference's own benchmark size (plain_cpu) at its default depth: one small frame
        _case("frame", "query", 3, "float32", 100_000, 10_000, 5, "normal", levels="default"),
        # one sensor sweep matched against a local map, odd sizes; coordinates in whole millimetres tie,
        # so the tie order that does not depend on the tree
        _case("sweep", "query", 3, "float32", 250_007, 65_537, 10, "rounded", tie="lower_index"),
        # image or height-field coordinates
        _case("planar", "query", 2, "float32", 262_144, 300_000, 4, "uniform"),
        # the headline workload (plain_gpu): the largest call
        _case("plain", "query", 3, "float32", 4_000_000, 16_000_000, 16, "plain"),
        # the same kind of cloud in a tree of the reference's default depth (13)
        _case("default_depth", "query", 3, "float32", 1_000_000, 1_000_000, 8, "plain", levels="default"),
        # double precision (fp64_normal)
        _case("fp64", "query", 3, "float64", 500_000, 500_000, 16, "normal"),
        # wide neighbourhoods (density, normals, outlier tests): lists beyond 32 entries
        _case("wide_k", "query", 3, "float32", 200_000, 100_000, 100, "gmm"),
        # a training step on a surface (diff_sphere): forward and backward
        _case("surface_grad", "grad", 3, "float32", 1_000_000, 1_000_000, 8, "sphere"),
        # feature space (d8_mixture): forward and backward
        _case("features_grad", "grad", 8, "float32", 500_000, 500_000, 32, "mixture"),
        # many clouds of uneven size in one captured training step (batch_clouds, a quarter of it)
        _batch("clouds", 64, 1_000, 500_000),
        # a cloud that changed: its tree built anew on the GPU, then queried
        _case("rebuild", "rebuild", 3, "float32", 500_000, 200_000, 8, "gmm"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["small", "query", "query", "large", "wide", "double", "grad", "features", "batch", "rebuild"])
    levels = rng.choice(["auto", "auto", "default"])
    tie = rng.choice(["reference", "reference", "reference", "lower_index"])
    d = rng.choice([2, 3, 3, 3])
    cloud = rng.choice(["uniform", "normal", "gmm", "rounded"])
    if op == "small":
        return _case(None, "query", d, "float32", _log_int(rng, 1_000, 1_000_000), _log_int(rng, 1, 4_095),
                     rng.randint(1, 32), cloud, levels, tie)
    if op == "query":
        d = rng.choice([1, 2, 3, 3, 3, 8])
        if d == 8:  # many more leaves a query: fewer queries
            return _case(None, "query", d, "float32", _log_int(rng, 5_000, 500_000), _log_int(rng, 1_000, 50_000),
                         rng.randint(1, 32), "mixture", levels, tie)
        return _case(None, "query", d, "float32", _log_int(rng, 5_000, 1_000_000), _log_int(rng, 4_096, 300_000),
                     rng.randint(1, 32), cloud, levels, tie)
    if op == "large":
        return _case(None, "query", d, "float32", _log_int(rng, 100_000, 4_000_000),
                     _log_int(rng, 500_000, 8_000_000), rng.randint(1, 16), rng.choice(["plain", "gmm", "uniform"]),
                     "auto", tie)
    if op == "wide":
        return _case(None, "query", d, "float32", _log_int(rng, 5_000, 500_000), _log_int(rng, 100, 100_000),
                     rng.randint(33, 128), cloud, levels, tie)
    if op == "double":
        return _case(None, "query", d, "float64", _log_int(rng, 5_000, 1_000_000), _log_int(rng, 1_000, 1_000_000),
                     rng.randint(1, 32), cloud, levels, tie)
    if op == "grad":
        return _case(None, "grad", 3, "float32", _log_int(rng, 5_000, 1_000_000), _log_int(rng, 1_000, 1_000_000),
                     rng.randint(1, 16), rng.choice(["sphere", "gmm"]), levels, "reference")
    if op == "features":
        return _case(None, "grad", 8, "float32", _log_int(rng, 20_000, 500_000), _log_int(rng, 1_000, 300_000),
                     rng.randint(4, 32), "mixture", "auto", "reference")
    if op == "batch":
        return _batch(None, rng.randint(4, 64), 1_000, _log_int(rng, 5_000, 300_000))
    return _case(None, "rebuild", d, "float32", _log_int(rng, 20_000, 1_000_000), _log_int(rng, 1_000, 500_000),
                 rng.randint(1, 16), rng.choice(["uniform", "gmm"]), "auto", "reference")


# ---------------------------------------------------------------------------------------------
# Inputs: drawn in float64 on the GPU from the seed alone, then cast
# ---------------------------------------------------------------------------------------------
def _device():
    return torch.device("cuda", torch.cuda.current_device())


def _mixture(g, count, d, comps, sigma, dev, centers, shape=None):
    lab = torch.randint(0, comps, (count,), generator=g, device=dev)
    z = torch.randn((count, d), generator=g, device=dev, dtype=torch.float64)
    if shape is None:
        return centers[lab] + sigma * z
    out = torch.empty_like(z)
    for c in range(comps):  # anisotropic components
        m = lab == c
        out[m] = centers[c] + z[m] @ shape[c].T
    return out


def _cloud(case, g, dev, n, q):
    """Reference points and queries of a case, float64."""
    d, kind = case["dims"], case["cloud"]
    rand = lambda *s: torch.rand(s, generator=g, device=dev, dtype=torch.float64)  # noqa: E731
    randn = lambda *s: torch.randn(s, generator=g, device=dev, dtype=torch.float64)  # noqa: E731
    if kind == "uniform":
        return rand(n, d), rand(q, d)
    if kind == "normal":
        return randn(n, d) * 1e3, randn(q, d) * 1e3
    if kind == "rounded":  # whole millimetres in a box of 50 m
        return torch.round(rand(n, d) * 5e4) / 1e3, torch.round(rand(q, d) * 5e4) / 1e3
    if kind == "gmm":
        cen = rand(32, d)
        return _mixture(g, n, d, 32, 0.02, dev, cen), _mixture(g, q, d, 32, 0.02, dev, cen)
    if kind == "plain":  # half of the queries over a slightly larger box, half clustered
        ref, cen = rand(n, d), rand(32, d)
        h = q // 2
        return ref, torch.cat([rand(h, d) * 1.2 - 0.1, _mixture(g, q - h, d, 32, 0.02, dev, cen)])
    if kind == "sphere":  # a bumpy sphere, queries near the surface
        def surface(count):
            v = randn(count, 3)
            v = v / v.norm(dim=1, keepdim=True)
            rad = 1 + 0.05 * torch.sin(4 * v[:, 0]) * torch.cos(3 * v[:, 1]) + 0.03 * torch.sin(5 * v[:, 2])
            return v * rad[:, None]
        ref = surface(n)
        qry = ref[:q] if q <= n else torch.cat([ref, surface(q - n)])
        return ref, qry + 0.01 * randn(q, 3)
    if kind == "mixture":  # 64 anisotropic components, variances log-uniform in [0.01, 1]
        cen, comps = rand(64, d), []
        for _ in range(64):
            a = np.random.default_rng(int(torch.randint(0, 2**31, (1,), generator=g, device=dev))).standard_normal((d, d))
            rot, r = np.linalg.qr(a)
            comps.append(torch.from_numpy(rot * np.sign(np.diag(r))[None, :]).to(dev))
        var = torch.exp(rand(64, d) * math.log(100.0) + math.log(0.01))
        shape = [c * v.sqrt()[None, :] for c, v in zip(comps, var)]
        return (_mixture(g, n, d, 64, None, dev, cen, shape), _mixture(g, q, d, 64, None, dev, cen, shape))
    raise ValueError(kind)


def _inputs(case, seed):
    dev = _device()
    g = torch.Generator(device=dev)
    g.manual_seed(int(seed) * 7919 + 17)
    dt = _DTYPES[case["dtype"]]
    ref, qry = _cloud(case, g, dev, case["n"], case["q"])
    w = torch.rand((case["q"], case["k"]), generator=g, device=dev, dtype=dt) if case["op"] == "grad" else None
    return ref.to(dt).contiguous(), qry.to(dt).contiguous(), w


def _batch_inputs(case, seed):
    """Clouds (ref, queries, k, weights): N log-uniform, Q = U(0.5, 2) N, k in {1, 4, 16}, uniform or
    an 8-component mixture."""
    dev = _device()
    meta = np.random.default_rng(int(seed) * 7919 + 17)
    g = torch.Generator(device=dev)
    g.manual_seed(int(seed) * 7919 + 17)
    # sizes at fixed quantiles of the log-uniform law, so that the total is the same for every seed
    m = case["clouds"]
    u = (np.arange(m) + 0.5) / m
    ns = np.round(case["n_min"] * (case["n_max"] / case["n_min"]) ** u).astype(int)
    fac = 0.5 + 1.5 * ((np.arange(m) * 7 % m) + 0.5) / m
    out = []
    for i in range(m):
        n, q, k = int(ns[i]), max(1, int(round(fac[i] * ns[i]))), (1, 4, 16)[i % 3]
        if meta.random() < 0.5:
            ref = torch.rand((n, 3), generator=g, device=dev)
            qry = torch.rand((q, 3), generator=g, device=dev)
        else:
            cen = torch.rand((8, 3), generator=g, device=dev, dtype=torch.float64)
            ref = _mixture(g, n, 3, 8, 0.02, dev, cen).float()
            qry = _mixture(g, q, 3, 8, 0.02, dev, cen).float()
        out.append((ref, qry, k, torch.rand((q, k), generator=g, device=dev)))
    return out


# ---------------------------------------------------------------------------------------------
# State, pass, work
# ---------------------------------------------------------------------------------------------
def prepare(case, seed):
    if case["op"] == "batch":
        clouds = _batch_inputs(case, seed)
        batch = tk.build_kd_tree_batch([c[0] for c in clouds], device=_device())
        return dict(op="batch", step=tk.BatchStep(batch, [c[1] for c in clouds], [c[2] for c in clouds],
                                                  weights=[c[3] for c in clouds]))
    ref, qry, w = _inputs(case, seed)
    st = dict(op=case["op"], q=qry, k=case["k"])
    levels = "auto" if case["levels"] == "auto" else None
    if case["op"] == "rebuild":
        st.update(ref=ref, levels=levels)
        return st
    if case["op"] == "grad":
        ref.requires_grad_(True)
        qry.requires_grad_(True)
        st.update(ref=ref, w=w)
    st["tree"] = tk.build_kd_tree(ref, levels=levels, tie_break=case["tie"])
    return st


def run(state):
    op = state["op"]
    if op == "query":
        return state["tree"].query(state["q"], nr_nns_searches=state["k"])
    if op == "grad":
        # the upstream gradient w of sum(w * dists) handed to the backward, as an outer model does
        dists, inds = state["tree"].query(state["q"], nr_nns_searches=state["k"])
        gq, gr = torch.autograd.grad(dists, (state["q"], state["ref"]), grad_outputs=state["w"])
        return dists.detach(), inds, gq, gr
    if op == "batch":
        s = state["step"]
        s.replay()
        return s.dist, s.idx, s.orig, s.grad_queries, s.grad_refs
    # a cloud that changed: its tree built anew on the GPU, then queried
    tree = tk.build_kd_tree(state["ref"], levels=state["levels"], builder="gpu")
    return (*tree.query(state["q"], nr_nns_searches=state["k"]), tree.structured_points, tree.shuffled_ind)


def _batch_totals(case):
    m = case["clouds"]
    u = (np.arange(m) + 0.5) / m
    ns = np.round(case["n_min"] * (case["n_max"] / case["n_min"]) ** u)
    fac = 0.5 + 1.5 * ((np.arange(m) * 7 % m) + 0.5) / m
    q = np.maximum(1, np.round(fac * ns))
    k = np.array([(1, 4, 16)[i % 3] for i in range(m)])
    return float(ns.sum()), float(q.sum()), float((q * k).sum())


def work(case):
    """Points and queries read once, distances and indices written once (and, with gradients, the
    upstream gradient read and both gradients written); 3d - 1 operations for each neighbour's
    distance, 5d more for its gradient terms."""
    s = 8 if case["dtype"] == "float64" else 4
    d = case["dims"]
    if case["op"] == "batch":
        n, q, qk = _batch_totals(case)
    else:
        n, q, qk = float(case["n"]), float(case["q"]), float(case["q"]) * case["k"]
    nbytes = (n + q) * d * s + qk * (s + 8)
    flops = qk * (3 * d - 1)
    if case["op"] == "batch":
        nbytes += qk * 4
    if case["op"] in ("grad", "batch"):
        nbytes += qk * s + (n + q) * d * s
        flops += qk * 5 * d
    if case["op"] == "rebuild":
        nbytes += n * (d * s + 8)
    return {"bytes": nbytes, "flops": flops}


# ---------------------------------------------------------------------------------------------
# 64-bit values
# ---------------------------------------------------------------------------------------------
_EXACT_PAIRS = 21_000_000_000


def _exact_knn(ref, qry, k):
    """k nearest of every query by exhaustive float64 distances: (distances, indices)."""
    r, q = ref.detach().double(), qry.detach().double()
    rt = [r[:, a].contiguous() for a in range(r.shape[1])]
    ds, ix = [], []
    step = max(1, min(q.shape[0], 200_000_000 // r.shape[0]))
    for b in range(0, q.shape[0], step):
        qb = q[b:b + step]
        acc = torch.zeros((qb.shape[0], r.shape[0]), dtype=torch.float64, device=r.device)
        for a, col in enumerate(rt):
            diff = qb[:, a:a + 1] - col[None, :]
            acc += diff * diff
        v, i = torch.topk(acc, k, dim=1, largest=False, sorted=True)
        ds.append(v)
        ix.append(i)
    return torch.cat(ds), torch.cat(ix)


def exact(case, seed):
    if case["op"] == "batch" or case["n"] * case["q"] > _EXACT_PAIRS:
        return None
    ref, qry, w = _inputs(case, seed)
    dist, idx = _exact_knn(ref, qry, case["k"])
    if case["op"] == "grad":
        diff = qry.double()[:, None, :] - ref.double()[idx]
        term = 2.0 * w.double()[:, :, None] * diff
        gr = torch.zeros_like(ref, dtype=torch.float64)
        gr.index_add_(0, idx.reshape(-1), -term.reshape(-1, ref.shape[1]))
        return dist, None, term.sum(1), gr
    if case["op"] == "rebuild":
        return dist, None, None, None
    return dist, None
