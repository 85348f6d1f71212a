"""The work that is timed: what a user of this package has it do, through its public entry points.

Four kinds of calls:

  energy   ClusterEnergy on device tensors: the fixed-assignment energy of frozen labels, forward alone
           (an evaluation, as in a serving loop or a line search) or forward and backward (a training step);
  cluster  Context.process() of one mesh that the context holds (built, with its initial labels), and the
           labels read back: the clustering a program runs again for other seeds or options;
  batch    the same for many small meshes packed in one context, isotropic and QEM mixed;
  remesh   the whole call of the remeshing classes on host arrays: SetInput, Remesh, GetOutput (upload,
           device build, initial sampling, clustering, output mesh).

Meshes are the synthetic surfaces of the package's tests and benchmark (icosphere, star-shaped icosphere,
cube, displaced torus), of sizes from 1,500 to 16.8 million vertices.
"""
import math

import numpy as np
import torch

import acvd_amd
from acvd_amd import meshgen
from acvd_amd.energy import ClusterEnergy

ISO, QEM = acvd_amd.METRIC_ISOTROPIC, acvd_amd.METRIC_QEM
QEM_LEVEL = 3


def listed():
    return [
        # A coarse mesh's energy, evaluated in a loop: a call of a few microseconds of device work.
        {"name": "energy_iso_forward_2k", "kind": "energy", "metric": "iso", "nu": 61, "nv": 42, "meshes": 1,
         "per_cluster": 15, "step": False},
        # A training step on one small QEM mesh: launches and the autograd function count.
        {"name": "energy_qem_step_10k", "kind": "energy", "metric": "qem", "nu": 127, "nv": 81, "meshes": 1,
         "per_cluster": 20, "step": True},
        # A ragged batch, isotropic and QEM meshes of odd sizes mixed.
        {"name": "energy_mixed_step_12_ragged", "kind": "energy", "metric": "mixed", "nu": 301, "nv": 203,
         "meshes": 12, "per_cluster": 30, "step": True},
        # One isotropic mesh of a million vertices (CVT energy and gradient).
        {"name": "energy_iso_step_1m", "kind": "energy", "metric": "iso", "nu": 1024, "nv": 1024, "meshes": 1,
         "per_cluster": 42, "step": True},
        # The benchmark's energy workload: 16 QEM tori of 1024 x 1024 vertices, 25,000 clusters each.
        {"name": "energy_qem_step_16x1m", "kind": "energy", "metric": "qem", "nu": 1024, "nv": 1024, "meshes": 16,
         "per_cluster": 42, "step": True},
        # The smallest clustering of the tests: latency of the passes.
        {"name": "cluster_iso_ico_2k", "kind": "cluster", "mesh": "icosphere", "a": 4, "b": 0, "metric": "iso",
         "per_cluster": 15, "gradation": 0.0},
        # The benchmark's first small configuration: an icosphere of 40,962 vertices into 2,000 clusters.
        {"name": "cluster_iso_ico_41k", "kind": "cluster", "mesh": "icosphere", "a": 6, "b": 0, "metric": "iso",
         "per_cluster": 20.48, "gradation": 0.0},
        # Its second: a cube of 960,002 vertices into 20,000 clusters, QEM.
        {"name": "cluster_qem_cube_960k", "kind": "cluster", "mesh": "cube", "a": 400, "b": 0, "metric": "qem",
         "per_cluster": 48, "gradation": 0.0},
        # Its headline: a torus of 8,388,608 vertices into 100,000 clusters, QEM, weights by curvature^1.5.
        {"name": "cluster_qem_torus_8m", "kind": "cluster", "mesh": "torus", "a": 4096, "b": 2048, "metric": "qem",
         "per_cluster": 83.88608, "gradation": 1.5},
        # Many meshes at once (the benchmark's batched leg, fewer of them).
        {"name": "batch_32_star_icospheres", "kind": "batch", "meshes": 32, "lmin": 4, "lmax": 7,
         "per_cluster": 15},
        # A whole call at an ordinary, odd size, curvature-weighted QEM (ACVDQ with a gradation).
        {"name": "remesh_qem_torus_350k", "kind": "remesh", "mesh": "torus", "a": 701, "b": 503, "metric": "qem",
         "per_cluster": 50, "gradation": 1.5},
        # A coarse input: subdivided on the device before it is clustered, quadric placement after (ACVD).
        {"name": "remesh_iso_coarse_10k", "kind": "remesh", "mesh": "star", "a": 5, "b": 0, "metric": "iso",
         "per_cluster": 4, "gradation": 0.0},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _grid(rng, lo, hi):
    """Sides of a torus grid of lo..hi vertices, odd and even, up to 3:1."""
    n = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    nu = max(16, int(round(math.sqrt(n * math.exp(rng.uniform(-0.5, 1.0))))))
    return nu, max(16, int(round(n / nu)))


def draw(rng):
    kind = rng.choice(["energy", "energy", "cluster", "cluster", "batch", "remesh"])
    if kind == "energy":
        nu, nv = _grid(rng, 1500, 4.0e6)
        meshes = rng.randint(1, 12) if nu * nv <= 150000 else rng.randint(1, 2)
        return {"kind": kind, "metric": rng.choice(["iso", "qem", "mixed"]), "nu": nu, "nv": nv, "meshes": meshes,
                "per_cluster": round(math.exp(rng.uniform(math.log(10), math.log(150))), 2),
                "step": rng.random() < 0.7}
    if kind == "batch":
        lmin = rng.randint(3, 5)
        return {"kind": kind, "meshes": _log_int(rng, 4, 40), "lmin": lmin, "lmax": rng.randint(lmin + 1, 7),
                "per_cluster": round(rng.uniform(10, 40), 2)}
    mesh = rng.choice(["torus", "torus", "icosphere", "star", "cube"])
    big = kind == "cluster"
    a, b = 0, 0
    if mesh == "torus":
        a, b = _grid(rng, 1500, 2.0e6 if big else 3.0e5)
    elif mesh == "cube":
        a = _log_int(rng, 16, 400 if big else 200)
    else:
        a = rng.randint(4, 7)
    return {"kind": kind, "mesh": mesh, "a": a, "b": b, "metric": rng.choice(["iso", "qem"]),
            "per_cluster": round(math.exp(rng.uniform(math.log(12), math.log(100))), 2),
            "gradation": rng.choice([0.0, 1.5])}


# ------------------------------------------------------------------ surfaces
def _torus(nu, nv, seed):
    """Torus R = 1, r = 0.35, the tube radius displaced by 32 seeded sinusoids, FP32 positions: the
    benchmark's surface.  Each sinusoid is a sum of two products of one factor per direction."""
    rng = np.random.default_rng(seed)
    fu, fv = rng.integers(0, 33, 32), rng.integers(0, 33, 32)
    amp, ph = 0.01 * rng.uniform(0.2, 1.0, 32) / 4, rng.uniform(0, 2 * np.pi, 32)
    u, v = 2 * np.pi * np.arange(nu) / nu, 2 * np.pi * np.arange(nv) / nv
    pu = np.outer(u, fu) + ph
    pv = np.outer(v, fv)
    r = 0.35 + np.sin(pu) @ (amp * np.cos(pv)).T + np.cos(pu) @ (amp * np.sin(pv)).T
    ring = 1.0 + r * np.cos(v)
    xyz = np.empty((nu, nv, 3), np.float32)
    xyz[:, :, 0] = ring * np.cos(u)[:, None]
    xyz[:, :, 1] = ring * np.sin(u)[:, None]
    xyz[:, :, 2] = r * np.sin(v)
    i = np.arange(nu * nv, dtype=np.int32).reshape(nu, nv)
    j, k = np.roll(i, -1, 0), np.roll(i, -1, 1)
    d = np.roll(j, -1, 1)
    tri = np.empty((nu, nv, 2, 3), np.int32)
    tri[:, :, 0, 0], tri[:, :, 0, 1], tri[:, :, 0, 2] = i, j, d
    tri[:, :, 1, 0], tri[:, :, 1, 1], tri[:, :, 1, 2] = i, d, k
    return xyz.reshape(-1, 3), tri.reshape(-1, 3)


def _surface(case, seed):
    if case["mesh"] == "torus":
        return _torus(case["a"], case["b"], seed)
    if case["mesh"] == "cube":
        return meshgen.cube(case["a"], seed)
    if case["mesh"] == "star":
        return meshgen.star_icosphere(case["a"], seed)
    return meshgen.icosphere(case["a"], seed, 0.02)


def _vertices(case):
    if case["mesh"] == "torus":
        return case["a"] * case["b"]
    if case["mesh"] == "cube":
        return 6 * case["a"] ** 2 + 2
    return 10 * 4 ** case["a"] + 2


def _clusters(n, case):
    return max(4, int(n / case["per_cluster"]))


# -------------------------------------------------------------------- energy
def _energy_meshes(case):
    """(nu, nv, metric) of each mesh; the meshes of a mixed batch differ in size and metric."""
    out = []
    for m in range(case["meshes"]):
        nu, nv = case["nu"], case["nv"]
        if case["metric"] == "mixed":
            nu, nv = max(16, nu * (m + 2) // (m + 3) - 3 * m), max(16, nv - 7 * m)
        qem = case["metric"] == "qem" or (case["metric"] == "mixed" and m % 2 == 1)
        out.append((nu, nv, QEM if qem else ISO))
    return out


def _patches(nu, nv, per_cluster, rng):
    """Labels of a settled clustering of a torus grid: about round patches in staggered columns with an
    uneven border, some vertices of each border with the neighbour, and now and then a vertex without a
    cluster.  Returns (labels, number of clusters)."""
    cols = max(1, int(round(nu / math.sqrt(per_cluster))))
    rows = max(1, int(round(nu * nv / per_cluster / cols)))
    u = np.arange(nu)[:, None] + rng.uniform(-0.7, 0.7, (nu, nv))
    v = np.arange(nv)[None, :] + rng.uniform(-0.7, 0.7, (nu, nv))
    cu = np.floor(u * cols / nu).astype(np.int64) % cols
    cv = np.floor(v * rows / nv + 0.5 * (cu & 1)).astype(np.int64) % rows
    lab = (cu * rows + cv).astype(np.int32).reshape(-1)
    K = cols * rows
    lab[rng.random(nu * nv) < 1e-4] = K
    return lab, K


def _energy_inputs(case, seed):
    """Per mesh (xyz, tri, weights, labels, K, metric), and the upstream gradient per mesh."""
    rng = np.random.default_rng(seed)
    meshes = []
    for nu, nv, metric in _energy_meshes(case):
        xyz, tri = _torus(nu, nv, int(rng.integers(1 << 30)))
        lab, K = _patches(nu, nv, case["per_cluster"], rng)
        # weights: the cell's area times a smooth density, uneven by two orders of magnitude
        r = np.hypot(np.hypot(xyz[:, 0], xyz[:, 1]) - 1.0, xyz[:, 2])
        area = (2 * np.pi / nu) * np.hypot(xyz[:, 0], xyz[:, 1]) * (2 * np.pi / nv) * r
        dens = np.exp(2.0 * np.sin(7 * xyz[:, 0] + 1.0) + 0.4 * rng.standard_normal(nu * nv))
        meshes.append((xyz, tri, (area * dens).astype(np.float32), lab, K, metric))
    return meshes, rng.uniform(0.5, 1.5, len(meshes))


def _prepare_energy(case, seed):
    meshes, g = _energy_inputs(case, seed)
    energy = ClusterEnergy(0)
    for xyz, tri, _, _, K, metric in meshes:
        energy.add_mesh(len(xyz), tri, K, metric, QEM_LEVEL)
    dev = torch.device("cuda", 0)
    cat = [torch.from_numpy(np.concatenate([m[k] for m in meshes])).to(dev) for k in (0, 2, 3)]
    step = case["step"]
    return {"kind": "energy", "energy": energy, "step": step, "xyz": cat[0].requires_grad_(step),
            "w": cat[1].requires_grad_(step), "labels": cat[2], "g": torch.from_numpy(g).to(dev)}


def _run_energy(s):
    if not s["step"]:
        with torch.no_grad():
            return {"energy": s["energy"](s["xyz"], s["w"], s["labels"])}
    e = s["energy"](s["xyz"], s["w"], s["labels"])
    dx, dw = torch.autograd.grad(e, (s["xyz"], s["w"]), grad_outputs=s["g"])
    return {"energy": e.detach(), "dxyz": dx, "dw": dw}


class _TruncatedStep(torch.autograd.Function):
    """y = A+ r with A's pseudo-inverse over the eigenvalues above 1e-3 of the largest, at most `level` of
    them; the derivative of the truncated pseudo-inverse couples kept and dropped directions."""

    @staticmethod
    def forward(ctx, A, r, level):
        lam, V = torch.linalg.eigh(A)
        mag = lam.abs()
        top = mag.max(-1, keepdim=True).values
        rank = mag.argsort(dim=-1, descending=True, stable=True).argsort(dim=-1)
        keep = (top > 0) & (mag * (1.0 / torch.where(top > 0, top, torch.ones_like(top))) > 1e-3) & (rank < level)
        inv = torch.where(keep, 1.0 / torch.where(keep, lam, torch.ones_like(lam)), torch.zeros_like(lam))
        vr = torch.einsum("kij,ki->kj", V, r)
        y = torch.einsum("kij,kj->ki", V, inv * vr)
        ctx.save_for_backward(lam, V, keep, inv, vr, y)
        return y

    @staticmethod
    def backward(ctx, gy):
        lam, V, keep, inv, vr, y = ctx.saved_tensors
        vg = torch.einsum("kij,ki->kj", V, gy)
        h = torch.einsum("kij,kj->ki", V, inv * vg)
        gap = lam[:, :, None] - lam[:, None, :]
        pair = keep[:, :, None] & ~keep[:, None, :] & (gap != 0)
        den = torch.where(pair, lam[:, :, None] * gap, torch.ones_like(gap))
        num = vg[:, None, :] * vr[:, :, None] + vg[:, :, None] * vr[:, None, :]
        coef = torch.where(pair, num / den, torch.zeros_like(gap))  # [kept, dropped]
        G = -h[:, :, None] * y[:, None, :] + torch.einsum("kia,kba,kjb->kij", V, coef, V)
        return 0.5 * (G + G.transpose(1, 2)), h, None


def _exact_energy(case, seed):
    meshes, g = _energy_inputs(case, seed)
    es, dxs, dws = [], [], []
    for (xyz, tri, w, lab, K, metric), gm in zip(meshes, g):
        x = torch.from_numpy(xyz).double().requires_grad_()
        wt = torch.from_numpy(w).double().requires_grad_()
        t, l = torch.from_numpy(tri).long(), torch.from_numpy(lab).long()
        has = (l >= 0) & (l < K)
        lc = torch.where(has, l, torch.full_like(l, K))
        W = torch.zeros(K + 1, dtype=torch.float64).index_add(0, lc, wt)
        S = torch.zeros(K + 1, 3, dtype=torch.float64).index_add(0, lc, wt[:, None] * x)
        c = S / torch.where(W > 0, W, torch.ones_like(W))[:, None]
        q = c
        if metric == QEM:
            x0, x1, x2 = x[t[:, 0]], x[t[:, 1]], x[t[:, 2]]
            n = torch.linalg.cross(x1 - x0, x2 - x0)
            d = -(n * x0).sum(-1, keepdim=True)
            nn, nd = n[:, :, None] * n[:, None, :], n * d
            A = torch.zeros(K + 1, 3, 3, dtype=torch.float64)
            b = torch.zeros(K + 1, 3, dtype=torch.float64)
            for j in range(3):
                A = A.index_add(0, lc[t[:, j]], nn)
                b = b.index_add(0, lc[t[:, j]], nd)
            r = -b - (A @ c[:, :, None])[:, :, 0]
            q = c + _TruncatedStep.apply(A, r, QEM_LEVEL)
        e = (wt * ((x - q[lc]) ** 2).sum(-1))[has].sum()
        if case["step"]:
            gx, gw = torch.autograd.grad(e * float(gm), (x, wt))
            dxs.append(gx)
            dws.append(gw)
        es.append(e.detach())
    out = {"energy": torch.stack(es)}
    if case["step"]:
        out["dxyz"], out["dw"] = torch.cat(dxs), torch.cat(dws)
    return out


# ---------------------------------------------------------------- clustering
def _settled(ctx):
    """The context built, with the reference's initial sampling as its initial labels (the benchmark's start)."""
    ctx.build()
    ctx.initial_sampling()
    for m in range(ctx.num_meshes):
        ctx.set_initial_labels(m, ctx.labels(m))
    return ctx


def _prepare_cluster(case, seed):
    xyz, tri = _surface(case, seed)
    ctx = acvd_amd.Context(0)
    ctx.set_input(xyz, tri)
    qem = case["metric"] == "qem"
    ctx.set_params(0, number_of_clusters=_clusters(len(xyz), case), metric=QEM if qem else ISO,
                   unconstrained_initialization=int(qem), gradation=case["gradation"], seed=seed & 0xFFFF)
    if case["gradation"] > 0:
        ctx.set_indicator(0, meshgen.mean_curvature(xyz, tri))
    return {"kind": "cluster", "ctx": _settled(ctx)}


def _prepare_batch(case, seed):
    ctx = acvd_amd.Context(0)
    levels = meshgen.batch_levels(case["meshes"], case["lmin"], case["lmax"], 4)
    for m, level in enumerate(levels):
        xyz, tri = meshgen.star_icosphere(int(level), 1000 * (seed % 100003) + m)
        ctx.add_input(xyz, tri)
        ctx.set_params(m, number_of_clusters=_clusters(len(xyz), case), metric=QEM if m % 2 else ISO,
                       unconstrained_initialization=m % 2, seed=m)
    return {"kind": "batch", "ctx": _settled(ctx)}


def _run_cluster(s):
    ctx = s["ctx"]
    ctx.process()
    # over 64 outputs would be many arrays: the labels of a batch in one
    return {"labels": np.concatenate([ctx.labels(m) for m in range(ctx.num_meshes)])}


# -------------------------------------------------------------------- remesh
def _prepare_remesh(case, seed):
    xyz, tri = _surface(case, seed)
    cls = acvd_amd.QIsotropicDiscreteRemeshing if case["metric"] == "qem" else acvd_amd.IsotropicDiscreteRemeshing
    return {"kind": "remesh", "mesh": acvd_amd.Mesh(xyz, tri), "cls": cls, "K": _clusters(len(xyz), case),
            "gradation": case["gradation"], "seed": seed & 0xFFFF}


def _run_remesh(s):
    r = s["cls"].New()
    r.SetInput(s["mesh"])
    r.SetNumberOfClusters(s["K"])
    r.SetSeed(s["seed"])
    r.GetMetric().SetGradation(s["gradation"])
    if r.METRIC == QEM:
        r.GetMetric().SetQuadricsOptimizationLevel(QEM_LEVEL)
        r.SetUnconstrainedInitialization(1)
    r.Remesh()
    out = r.GetOutput()
    if r.METRIC == ISO:
        out = r.QuadricPostProcessing(1)
    # the number of triangles depends on the clustering: rows after the last are -1
    tri = np.full((4 * s["K"], 3), -1, np.int32)
    tri[:len(out.triangles)] = out.triangles
    res = {"labels": r.GetClustering(), "points": out.points, "triangles": tri}
    r.Delete()
    return res


# ---------------------------------------------------------------- interface
def prepare(case, seed):
    if case["kind"] == "energy":
        return _prepare_energy(case, seed)
    if case["kind"] == "cluster":
        return _prepare_cluster(case, seed)
    if case["kind"] == "batch":
        return _prepare_batch(case, seed)
    return _prepare_remesh(case, seed)


def run(state):
    if state["kind"] == "energy":
        return _run_energy(state)
    if state["kind"] in ("cluster", "batch"):
        return _run_cluster(state)
    return _run_remesh(state)


def exact(case, seed):
    """Energies and gradients in 64 bits; labels are whole numbers, and an output mesh follows from its labels."""
    return _exact_energy(case, seed) if case["kind"] == "energy" else None


def work(case):
    """Each input read once, each output written once."""
    if case["kind"] == "energy":
        b = f = 0.0
        for nu, nv, metric in _energy_meshes(case):
            n = nu * nv
            b += 20.0 * n + 8 + (24.0 * n if metric == QEM else 0.0)  # position, weight, label; triangles
            f += (18.0 + (160.0 if metric == QEM else 0.0)) * n
            if case["step"]:
                b += 16.0 * n + 8  # the gradients
                f += (24.0 + (500.0 if metric == QEM else 0.0)) * n
        return {"bytes": b, "flops": f}
    if case["kind"] == "batch":
        levels = meshgen.batch_levels(case["meshes"], case["lmin"], case["lmax"], 4)
        n = float(sum(10 * 4 ** int(v) + 2 for v in levels))
        # position and weight, quadric of every second mesh, adjacency, labels in and out
        return {"bytes": n * (16 + 20 + 28 + 8), "flops": 50.0 * n}
    n = float(_vertices(case))
    if case["kind"] == "cluster":
        return {"bytes": n * (16 + (40 if case["metric"] == "qem" else 0) + 28 + 8), "flops": 50.0 * n}
    k = float(_clusters(n, case))
    levels = 0
    while n * 4 ** levels < 10 * k:  # inputs of fewer than 10 vertices per cluster are subdivided
        levels += 1
    return {"bytes": n * (24 + 24) + 4 * n * 4 ** levels + 48 * k, "flops": 200.0 * n * 4 ** levels}
