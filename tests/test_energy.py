"""Fixed-assignment energy and its adjoint (no reference counterpart: the
reference never differentiates its energy).

Pins (CPU): the dual-number derivatives of the oracle (oracle/energy_ref.h)
equal the closed form of the isotropic gradient (dE/dx_i = 2 w_i (x_i - c),
dE/dw_i = |x_i - c|^2) and FP64 central differences of the QEM energy.
GPU: the forward equals the oracle's FP64 energy (rtol 1e-9; FP32 inputs read
as FP64 on both sides); the adjoint equals the oracle's derivatives at every
coordinate (tolerance 1e-5 of the largest component: FP32 outputs) and FP64
central differences (step 1e-6) at 1,000 seeded coordinates with relative
error <= 1e-4 (relative to max(|fd|, 1e-3 max|fd|)); autograd plumbing and
batches of mixed metrics."""
import numpy as np
import pytest

import acvd_amd
from acvd_amd import meshgen
from oracle import pyoracle as po

ISO, QEM = acvd_amd.METRIC_ISOTROPIC, acvd_amd.METRIC_QEM


def small_problem(metric, level=3, seed=4):
    xyz, tri = meshgen.icosphere(3, seed, 0.05)
    rng = np.random.default_rng(seed)
    x = np.asarray(xyz, np.float32).astype(np.float64)
    w = rng.uniform(0.5, 2.0, len(x)).astype(np.float32).astype(np.float64)
    K = 40
    lab = po.RefMesh(xyz, tri).fill_holes(K, meshgen.seed_labels(len(x), K, seed))
    return x, w, tri, lab, K


def test_iso_dual_derivatives_match_closed_form():
    x, w, tri, lab, K = small_problem(ISO)
    ref = po.EnergyRef(len(x), tri, lab, K, ISO)
    n = len(x)
    coords = np.arange(4 * n)
    d = ref.derivatives(x, w, coords)
    W = np.bincount(lab, weights=w, minlength=K + 1)[:K]
    S = np.stack([np.bincount(lab, weights=w * x[:, k], minlength=K + 1)[:K] for k in range(3)], 1)
    c = S / W[:, None]
    diff = x - c[lab]
    gx = 2.0 * w[:, None] * diff
    gw = (diff ** 2).sum(1)
    np.testing.assert_allclose(d[:3 * n], gx.reshape(-1), rtol=1e-9, atol=1e-12)
    np.testing.assert_allclose(d[3 * n:], gw, rtol=1e-9, atol=1e-12)
    # and the energy itself
    assert np.isclose(ref.total(x, w), float((w * gw).sum()), rtol=1e-12)


@pytest.mark.parametrize("level", [1, 2, 3])
def test_qem_dual_derivatives_match_central_differences(level):
    x, w, tri, lab, K = small_problem(QEM, level)
    ref = po.EnergyRef(len(x), tri, lab, K, QEM, level)
    rng = np.random.default_rng(level)
    coords = rng.choice(4 * len(x), 300, replace=False)
    d = ref.derivatives(x, w, coords)
    fd = ref.central_differences(x, w, coords, 1e-6)
    scale = np.abs(fd).max()
    err = np.abs(d - fd) / np.maximum(np.abs(fd), 1e-3 * scale)
    assert np.quantile(err, 0.99) < 1e-5 and err.max() < 1e-3, (np.quantile(err, 0.99), err.max())


def test_qem_point_is_quadric_minimiser_for_full_rank_clusters():
    # with level 3 and full-rank cluster quadrics the QEM energy does not
    # depend on the centroid: perturbing a weight only moves the direct term
    x, w, tri, lab, K = small_problem(QEM)
    ref = po.EnergyRef(len(x), tri, lab, K, QEM, 3)
    n = len(x)
    coords = 3 * n + np.arange(0, n, 7)
    d = ref.derivatives(x, w, coords)
    fd = ref.central_differences(x, w, coords, 1e-6)
    np.testing.assert_allclose(d, fd, rtol=1e-5, atol=1e-9)


# ------------------------------------------------------------------- GPU
def gpu_inputs(x, w, lab, K):
    import torch
    dev = torch.device("cuda", 0)
    lab_gpu = np.where((lab >= 0) & (lab < K), lab, K).astype(np.int32)
    return (torch.tensor(x, dtype=torch.float32, device=dev).contiguous(),
            torch.tensor(w, dtype=torch.float32, device=dev).contiguous(),
            torch.tensor(lab_gpu, dtype=torch.int32, device=dev).contiguous())


@pytest.mark.gpu
@pytest.mark.parametrize("metric,level", [(ISO, 3), (QEM, 1), (QEM, 2), (QEM, 3)])
def test_gpu_energy_forward_and_adjoint_match_oracle(gpu_ready, metric, level):
    from acvd_amd.energy import ClusterEnergy
    x, w, tri, lab, K = small_problem(metric, level)
    ref = po.EnergyRef(len(x), tri, lab, K, metric, level)
    ce = ClusterEnergy(0)
    ce.add_mesh(len(x), tri, K, metric, level)
    tx, tw, tl = gpu_inputs(x, w, lab, K)
    e = ce.forward_raw(tx, tw, tl).cpu().numpy()
    assert np.isclose(e[0], ref.total(x, w), rtol=1e-9), (e[0], ref.total(x, w))
    import torch
    dx, dw = ce.backward_raw(tx, tw, tl, torch.ones(1, dtype=torch.float64, device=tx.device))
    g = np.concatenate([dx.cpu().numpy().reshape(-1), dw.cpu().numpy()]).astype(np.float64)
    d = ref.derivatives(x, w, np.arange(4 * len(x)))
    scale = np.abs(d).max()
    assert np.abs(g - d).max() < 1e-5 * scale, np.abs(g - d).max() / scale


@pytest.mark.gpu
def test_gpu_adjoint_against_central_differences_torus(gpu_ready):
    """1,000 seeded coordinates (positions and weights) of a QEM torus with
    frozen labels from a GPU clustering."""
    import torch
    from acvd_amd.energy import ClusterEnergy
    xyz, tri = meshgen.torus(256, 128, 5)
    H = meshgen.mean_curvature(xyz, tri)
    K = 1500
    ctx = acvd_amd.Context()
    ctx.set_input(xyz, tri)
    ctx.set_params(0, number_of_clusters=K, metric=QEM, unconstrained_initialization=1, gradation=1.5, seed=5)
    ctx.set_indicator(0, H)
    ctx.process()
    lab = ctx.labels(0)
    xw, _ = ctx.items(0)
    x = np.asarray(xyz, np.float32).astype(np.float64)
    w = xw[:, 3].astype(np.float64)
    ce = ClusterEnergy(0)
    ce.add_mesh(len(x), tri, K, QEM, 3)
    tx, tw, tl = gpu_inputs(x, w, lab, K)
    E = ce(tx.requires_grad_(), tw.requires_grad_(), tl)
    E.sum().backward()
    g = np.concatenate([tx.grad.cpu().numpy().reshape(-1), tw.grad.cpu().numpy()]).astype(np.float64)
    ref = po.EnergyRef(len(x), tri, lab, K, QEM, 3)
    assert np.isclose(E.item(), ref.total(x, w), rtol=1e-9)
    rng = np.random.default_rng(5)
    coords = rng.choice(4 * len(x), 1000, replace=False)
    fd = ref.central_differences(x, w, coords, 1e-6)
    fd7 = ref.central_differences(x, w, coords, 1e-7)
    dual = ref.derivatives(x, w, coords)
    scale = np.abs(dual).max()
    # the QEM energy is not differentiable where a cluster's kept eigen-set
    # changes; such coordinates show difference quotients that depend on the step
    smooth = np.abs(fd - fd7) <= 1e-3 * np.maximum(np.abs(fd), 1e-3 * scale)
    assert smooth.sum() >= 990
    err = np.abs(g[coords] - fd) / np.maximum(np.abs(fd), 1e-3 * scale)
    # fourth-order differences (Richardson over steps 1e-6 and 2e-6): the
    # second-order quotient's h^2 f''' term dominates its error where the
    # third derivative is large
    fd2 = ref.central_differences(x, w, coords, 2e-6)
    fd4 = (4.0 * fd - fd2) / 3.0
    err4 = np.abs(g[coords] - fd4) / np.maximum(np.abs(fd4), 1e-3 * scale)
    smooth4 = smooth & (np.abs(fd2 - fd) <= 1e-3 * np.maximum(np.abs(fd), 1e-3 * scale))
    print(f"FD check: {int(smooth.sum())} smooth coordinates, median rel err {np.median(err[smooth]):.2e}, "
          f"max {err[smooth].max():.2e}; fourth order max {err4[smooth4].max():.2e}")
    assert np.quantile(err[smooth], 0.99) <= 1e-4 and err[smooth].max() <= 1e-3
    assert smooth4.sum() >= 990 and err4[smooth4].max() <= 1e-4
    # the dual-number derivative is exact at the point, smooth or not
    err_dual = np.abs(g[coords] - dual) / np.maximum(np.abs(dual), 1e-3 * scale)
    print(f"dual check: max rel err {err_dual.max():.2e}")
    assert err_dual.max() <= 1e-6, err_dual.max()


@pytest.mark.gpu
def test_gpu_energy_batch_equals_separate(gpu_ready):
    import torch
    from acvd_amd.energy import ClusterEnergy
    probs = [small_problem(ISO, 3, 4), small_problem(QEM, 3, 6)]
    ce = ClusterEnergy(0)
    xs, ws, ls = [], [], []
    singles = []
    for (x, w, tri, lab, K), metric in zip(probs, (ISO, QEM)):
        ce.add_mesh(len(x), tri, K, metric, 3)
        tx, tw, tl = gpu_inputs(x, w, lab, K)
        xs.append(tx), ws.append(tw), ls.append(tl)
        one = ClusterEnergy(0)
        one.add_mesh(len(x), tri, K, metric, 3)
        e1 = one.forward_raw(tx, tw, tl)
        d1 = one.backward_raw(tx, tw, tl, torch.ones(1, dtype=torch.float64, device=tx.device))
        singles.append((e1.item(), d1))
    tx, tw, tl = torch.cat(xs).contiguous(), torch.cat(ws).contiguous(), torch.cat(ls).contiguous()
    e = ce.forward_raw(tx, tw, tl).cpu().numpy()
    dx, dw = ce.backward_raw(tx, tw, tl, torch.ones(2, dtype=torch.float64, device=tx.device))
    n0 = len(probs[0][0])
    for k, (e1, (dx1, dw1)) in enumerate(singles):
        assert np.isclose(e[k], e1, rtol=1e-12)
        sl = slice(0, n0) if k == 0 else slice(n0, None)
        np.testing.assert_allclose(dx[sl].cpu().numpy(), dx1.cpu().numpy(), rtol=1e-6, atol=1e-7)
        np.testing.assert_allclose(dw[sl].cpu().numpy(), dw1.cpu().numpy(), rtol=1e-6, atol=1e-7)


def ring_problem(shape):
    """Meshes whose rings of faces are not one closed fan of at most 7 neighbours:
    a hub of 9 / 16 / 17 / 70 faces, an open grid (boundary vertices), two cones
    joined at their tip (a bowtie, with a degenerate face and a vertex without
    faces), and scattered labels (every ring meets many clusters; more clusters
    than a block's table holds)."""
    rng = np.random.default_rng(7)
    if shape.startswith("hub"):
        n = int(shape[3:])
        t = 2 * np.pi * np.arange(n) / n
        x = np.concatenate([[[0, 0, 0.4]], np.stack([np.cos(t), np.sin(t), 0.1 * np.cos(3 * t)], 1), [[0, 0, -0.6]]])
        i = np.arange(n)
        tri = np.concatenate([np.stack([np.zeros(n, int), 1 + i, 1 + (i + 1) % n], 1),
                              np.stack([np.full(n, n + 1), 1 + (i + 1) % n, 1 + i], 1)])
        lab, K = rng.integers(0, 4, len(x)), 4
    elif shape == "grid":
        n = 19
        u, v = np.meshgrid(np.arange(n), np.arange(n), indexing="ij")
        x = np.stack([u / n, v / n, 0.05 * rng.standard_normal((n, n))], -1).reshape(-1, 3)
        i = (u * n + v)[:-1, :-1].reshape(-1)
        tri = np.concatenate([np.stack([i, i + n, i + n + 1], 1), np.stack([i, i + n + 1, i + 1], 1)])
        lab, K = (u // 5 * 4 + v // 5).reshape(-1), 18  # two clusters stay empty
        lab[rng.random(len(lab)) < 0.1] = 18
    elif shape == "bowtie":
        x0, _, t0, _, _ = ring_problem("hub6")
        x1 = x0[1:] * [1, 1, -1] + [0, 0, 0.8]
        x = np.concatenate([x0, x1, [[3, 3, 3]]])
        t1 = np.where(t0 == 0, 0, t0 + len(x0) - 1)[:, ::-1]
        tri = np.concatenate([t0, t1, [[1, 1, 2]]])
        lab, K = rng.integers(0, 3, len(x)), 3
    else:
        xyz, tri = meshgen.icosphere(4 if shape == "scattered4" else 5, 3, 0.05)
        x, K = np.asarray(xyz), 60 if shape == "scattered4" else 5000
        lab = rng.integers(0, K, len(x))
    x = np.asarray(x, np.float32).astype(np.float64)
    w = rng.uniform(0.5, 2.0, len(x)).astype(np.float32).astype(np.float64)
    return x, w, np.ascontiguousarray(tri, np.int32), lab.astype(np.int32), K


@pytest.mark.gpu
@pytest.mark.parametrize("shape", ["hub9", "hub16", "hub17", "hub70", "grid", "bowtie", "scattered4", "scattered5"] +
                         [f"hub{n}" for n in (7, 8, 14, 15, 21, 22, 31, 32, 33, 37)])  # a ring's chunks; rows past a ring
@pytest.mark.parametrize("metric", [ISO, QEM])
def test_gpu_energy_rings_match_oracle(gpu_ready, metric, shape):
    """Against the oracle on meshes with every form of ring, alone, behind
    another mesh of 37 vertices (rings and blocks not aligned to the mesh) and
    behind one of 17,600 too (rows built on the device).
    Tolerances: the energy sums FP64 terms in another order (1e-9), the gradients
    are rounded to FP32 (1e-5 of the largest component, as above)."""
    import torch
    from acvd_amd.energy import ClusterEnergy
    x, w, tri, lab, K = ring_problem(shape)
    ref = po.EnergyRef(len(x), tri, np.where(lab < K, lab, K), K, metric, 2)
    e_ref, d = ref.total(x, w), ref.derivatives(x, w, np.arange(4 * len(x)))
    pad = ring_problem("hub35")
    xyz_t, tri_t = meshgen.torus(160, 110, 2)  # past the contexts whose rows the host builds
    torus = (np.asarray(xyz_t, np.float64), np.ones(17600), np.asarray(tri_t, np.int32),
             (np.arange(17600) // 50).astype(np.int32), 352)
    for lead in ([], [(pad, QEM)], [(torus, QEM), (pad, QEM)]):
        meshes = lead + [((x, w, tri, lab, K), metric)]
        ce = ClusterEnergy(0)
        for (mx, _, mt, _, mk), mm in meshes:
            ce.add_mesh(len(mx), mt, mk, mm, 2)
        parts = [gpu_inputs(mx, mw, ml, mk) for (mx, mw, _, ml, mk), _ in meshes]
        tx, tw, tl = (torch.cat(t).contiguous() for t in zip(*parts))
        e = ce.forward_raw(tx, tw, tl).cpu().numpy()
        assert np.isclose(e[-1], e_ref, rtol=1e-9), (e[-1], e_ref)
        g = torch.full((len(meshes),), 1.5, dtype=torch.float64, device=tx.device)
        dx, dw = (t[-len(x):].cpu().numpy() / 1.5 for t in ce.backward_raw(tx, tw, tl, g))
        got = np.concatenate([dx.reshape(-1), dw]).astype(np.float64)
        assert np.abs(got - d).max() < 1e-5 * np.abs(d).max(), np.abs(got - d).max() / np.abs(d).max()


@pytest.mark.gpu
@pytest.mark.parametrize("large", [False, True])
def test_gpu_energy_of_many_small_meshes(gpu_ready, large):
    """Meshes of 3 to 700 vertices, isotropic and QEM in turn, several to a wave and
    some over a few blocks; with `large` one of 150,000 vertices among them (blocks of
    several steps).  The small ones against the oracle, the large one against itself
    alone.  Tolerances: FP64 sums in another order (1e-9), gradients in FP32 (1e-5 of
    the largest component, as above; 1e-6 against itself)."""
    import torch
    from acvd_amd.energy import ClusterEnergy
    rng = np.random.default_rng(11)
    shapes = [ring_problem(f"hub{n}") for n in (3, 10, 62, 63, 64, 254, 510, 698)] + [ring_problem("grid")]
    shapes.append((np.asarray([[0, 0, 0], [1, 0, 0], [0, 1, 0.5]], np.float64), np.ones(3), np.asarray([[0, 1, 2]], np.int32),
                   np.asarray([0, 0, 1], np.int32), 2))
    order = rng.integers(0, len(shapes), 120)
    meshes = [(shapes[k], QEM if rng.random() < 0.5 else ISO) for k in order]
    if large:
        xyz, tri = meshgen.torus(500, 300, 4)
        x = np.asarray(xyz, np.float32).astype(np.float64)
        meshes.insert(60, ((x, rng.uniform(0.5, 2.0, len(x)), np.asarray(tri, np.int32),
                            (np.arange(len(x)) // 40).astype(np.int32), len(x) // 40), QEM))
    ce = ClusterEnergy(0)
    for (x, _, tri, _, K), metric in meshes:
        ce.add_mesh(len(x), tri, K, metric, 2)
    parts = [gpu_inputs(x, w, lab, K) for (x, w, _, lab, K), _ in meshes]
    tx, tw, tl = (torch.cat(t).contiguous() for t in zip(*parts))
    e = ce.forward_raw(tx, tw, tl).cpu().numpy()
    g = torch.arange(1, len(meshes) + 1, dtype=torch.float64, device=tx.device)
    dx, dw = (t.cpu().numpy() for t in ce.backward_raw(tx, tw, tl, g))
    off = 0
    for j, ((x, w, tri, lab, K), metric) in enumerate(meshes):
        s = slice(off, off + len(x))
        off += len(x)
        if len(x) > 10000:
            alone = ClusterEnergy(0)
            alone.add_mesh(len(x), tri, K, metric, 2)
            e_ref = alone.forward_raw(*parts[j]).item()
            d = np.concatenate([t.cpu().numpy().reshape(-1) for t in alone.backward_raw(*parts[j], g[j:j + 1])]) / (j + 1)
            tol = 1e-6
        else:
            ref = po.EnergyRef(len(x), tri, np.where(lab < K, lab, K), K, metric, 2)
            w = w.astype(np.float32).astype(np.float64)
            e_ref, d = ref.total(x, w), ref.derivatives(x, w, np.arange(4 * len(x)))
            tol = 1e-5
        assert np.isclose(e[j], e_ref, rtol=1e-9, atol=1e-30), (j, len(x), metric, e[j], e_ref)
        got = np.concatenate([dx[s].reshape(-1), dw[s]]).astype(np.float64) / (j + 1)
        assert np.abs(got - d).max() <= tol * np.abs(d).max() + 1e-30, (j, len(x), metric)


@pytest.mark.gpu
@pytest.mark.parametrize("n,K", [(1, 1), (63, 5), (1025, 40), (4096, 1024), (4096, 1025), (4097, 1024)])
def test_gpu_iso_energy_at_the_small_path(gpu_ready, n, K):
    """Either side of the sizes that one block takes, against the closed form in
    FP64 (sums of at most 4,097 terms in another order: 1e-12; gradients in FP32)."""
    import torch
    from acvd_amd.energy import ClusterEnergy
    rng = np.random.default_rng(n)
    x = rng.standard_normal((n, 3)).astype(np.float32)
    w = rng.uniform(0.5, 2.0, n).astype(np.float32)
    lab = np.sort(rng.integers(0, K + 1, n)).astype(np.int32)  # runs, empty clusters, unlabelled items
    ce = ClusterEnergy(0)
    ce.add_mesh(n, [[0, 0, 0]], K, ISO)
    tx, tw, tl = gpu_inputs(x, w, lab, K)
    e = ce.forward_raw(tx, tw, tl)
    dx, dw = ce.backward_raw(tx, tw, tl, torch.full((1,), 2.0, dtype=torch.float64, device=tx.device))
    x64, w64 = x.astype(np.float64), w.astype(np.float64)
    W = np.bincount(lab, weights=w64, minlength=K + 1)
    c = np.stack([np.bincount(lab, weights=w64 * x64[:, k], minlength=K + 1) for k in range(3)], 1)
    c /= np.where(W > 0, W, 1)[:, None]
    d = np.where((lab < K)[:, None], x64 - c[lab], 0.0)
    np.testing.assert_allclose(e.item(), (w64 * (d ** 2).sum(1)).sum(), rtol=1e-12, atol=1e-30)
    np.testing.assert_allclose(dx.cpu().numpy(), 4.0 * w64[:, None] * d, rtol=1e-6, atol=1e-12)
    np.testing.assert_allclose(dw.cpu().numpy(), 2.0 * (d ** 2).sum(1), rtol=1e-6, atol=1e-12)


@pytest.mark.gpu
def test_gpu_energy_errors(gpu_ready):
    import torch
    from acvd_amd.energy import ClusterEnergy
    x, w, tri, lab, K = small_problem(ISO)
    ce = ClusterEnergy(0)
    with pytest.raises(acvd_amd.AcvdError):
        ce.add_mesh(len(x), tri, 0, ISO)
    ce.add_mesh(len(x), tri, K, ISO)
    tx, tw, tl = gpu_inputs(x, w, lab, K)
    with pytest.raises(acvd_amd.AcvdError):
        ce.backward_raw(tx, tw, tl, torch.ones(1, dtype=torch.float64, device=tx.device))  # no forward yet
    with pytest.raises(acvd_amd.AcvdError):
        ce.forward_raw(tx.double(), tw, tl)
