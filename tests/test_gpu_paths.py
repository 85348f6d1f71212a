"""Every kernel path of a pass on meshes small enough for the CPU replay.

A context of at most 196,608 items scans and evaluates in one kernel, a larger
one in two, one of more than 700,000 items with tile sets once few items move.
The limits are lowered here (acvd_set_path_limits), and the passes launched per
path are checked, so that fixed and frozen clusters, QEM, batches, long rows and
other launch shapes run on each of them.  Labels equal the replay bit for bit."""
import numpy as np
import pytest

import acvd_amd
from acvd_amd import meshgen
from oracle import pyoracle as po
from tests.test_gpu_parity import centroid_split

pytestmark = pytest.mark.gpu

ISO, QEM = acvd_amd.METRIC_ISOTROPIC, acvd_amd.METRIC_QEM

# (fused_items, tile_min_items), paths that must and paths that must not run
PATHS = {
    "fused": ((1 << 40, 1 << 40), {"fused"}),
    "list": ((0, 1 << 40), {"list"}),
    "tiles": ((0, 0), {"list", "tiles"}),
    "fused-tiles": ((1 << 40, 0), {"fused", "tiles"}),
}


@pytest.fixture(autouse=True)
def clear_oracle_flags():
    yield
    po.set_fixed(None)
    po.set_frozen(None)


def set_path(ctx, path):
    ctx.set_path_limits(*PATHS[path][0])
    # tile sets as soon as a pass moves at most K items, looked at every fourth pass
    ctx.set_tuning(tile_on_divisor=1, chunk_passes=4, short_chunk_passes=2)


def check_path(ctx, path):
    ran = {k for k, n in ctx.path_passes().items() if n > 0}
    assert ran == PATHS[path][1], (path, ctx.path_passes())


def replay(ctx, mid, K, metric, init, seed, unc, **kw):
    rp, col = ctx.adjacency(mid)
    xw, q = ctx.items(mid)
    return po.replay_run(rp, col, xw, q, ctx.scales(mid), K, metric, init, seed=seed, unconstrained=unc, **kw)


def fixed_items(n_items, n, seed):
    return np.sort(np.random.default_rng(seed).choice(n_items, n, replace=False)).astype(np.int32)


@pytest.mark.parametrize("path", list(PATHS))
@pytest.mark.parametrize("metric,unc,kind", [(ISO, 0, "plain"), (QEM, 1, "plain"), (QEM, 0, "plain"),
                                             (QEM, 1, "long rows"), (ISO, 0, "long rows"), (QEM, 1, "fixed"),
                                             (QEM, 0, "fixed"), (ISO, 0, "fixed"), (QEM, 0, "frozen"),
                                             (ISO, 0, "frozen"), (ISO, 0, "few clusters"),
                                             (QEM, 1, "few clusters")])
def test_one_mesh_on_every_path(gpu_ready, path, metric, unc, kind):
    print(path, metric, unc, kind, flush=True)
    xyz, tri = centroid_split(*meshgen.icosphere(4, 9, 0.02)) if kind == "long rows" else meshgen.icosphere(5, 4, 0.03)
    K = 20 if kind == "few clusters" else 400  # 20: many proposals meet at a cluster
    ctx = acvd_amd.Context()
    ctx.set_input(xyz, tri)
    ctx.set_params(0, number_of_clusters=K, metric=metric, unconstrained_initialization=unc, seed=5)
    if kind == "fixed":
        fixed = fixed_items(len(xyz), 16, 2)
        po.set_fixed(fixed)
        ctx.set_fixed_clusters(0, fixed)
    m = po.RefMesh(xyz, tri)
    init = m.initial_sampling(metric, K)
    if kind == "frozen":
        init = m.fill_holes(K, init)
        frozen = (np.random.default_rng(3).random(K) < 0.5).astype(np.int32)
        po.set_frozen(frozen)
        ctx.set_frozen_clusters(0, frozen)
    ctx.set_initial_labels(0, init)
    set_path(ctx, path)
    ctx.process()
    check_path(ctx, path)
    rlab, rst = replay(ctx, 0, K, metric, init, 5, unc)
    assert ctx.stats(0)["loops"] == rst["loops"]
    np.testing.assert_array_equal(ctx.labels(0), rlab)


@pytest.mark.parametrize("path", list(PATHS))
@pytest.mark.parametrize("anchored", [False, True])
def test_batch_on_every_path(gpu_ready, path, anchored):
    print(path, anchored, flush=True)
    specs = [(meshgen.icosphere(4, 6, 0.03), QEM, 170, 1), (meshgen.star_icosphere(4, 7), ISO, 170, 0),
             (meshgen.cube(20, 14, 1e-4), QEM, 160, 0), (meshgen.icosphere(3, 8, 0.02), ISO, 40, 0),
             (meshgen.icosphere(4, 9, 0.02), ISO, 6, 0)]  # the last with many proposals per cluster
    ctx = acvd_amd.Context()
    want = []
    for k, ((xyz, tri), metric, K, unc) in enumerate(specs):
        mid = ctx.add_input(xyz, tri)
        fixed = fixed_items(len(xyz), 6, 3) if anchored and k == 0 else None
        ctx.set_params(mid, number_of_clusters=K, metric=metric, unconstrained_initialization=unc, seed=mid)
        ctx.set_fixed_clusters(mid, fixed)
        po.set_fixed(fixed)
        init = po.RefMesh(xyz, tri).initial_sampling(metric, K)
        ctx.set_initial_labels(mid, init)
        want.append((fixed, init))
    set_path(ctx, path)
    ctx.process()
    check_path(ctx, path)
    for mid, ((xyz, tri), metric, K, unc) in enumerate(specs):
        po.set_fixed(want[mid][0])
        np.testing.assert_array_equal(ctx.labels(mid), replay(ctx, mid, K, metric, want[mid][1], mid, unc)[0],
                                      err_msg=f"mesh {mid}")


@pytest.mark.parametrize("path", ["list", "tiles"])
def test_shapes_on_every_path(gpu_ready, path):
    """Segment counts and chunk lengths where the scan has a work list and tile sets."""
    xyz, tri = meshgen.icosphere(5, 21, 0.03)
    K = 400
    ctx = acvd_amd.Context()
    ctx.set_input(xyz, tri)
    ctx.set_params(0, number_of_clusters=K, metric=QEM, unconstrained_initialization=1, seed=1)
    init = po.RefMesh(xyz, tri).initial_sampling(QEM, K)
    ctx.set_initial_labels(0, init)
    ref = None
    for t in ({"sweep_segments": 7}, {"sweep_segments": 64, "tile_on_divisor": 2},
              {"chunk_passes": 3, "short_chunk_passes": 1}, {"sweep_segments": 2048, "chunk_passes": 16}):
        print(path, t, flush=True)
        set_path(ctx, path)
        ctx.set_tuning(**t)
        ctx.process()
        check_path(ctx, path)
        if ref is None:
            ref, _ = replay(ctx, 0, K, QEM, init, 1, 1)
        np.testing.assert_array_equal(ctx.labels(0), ref)


def test_build_of_small_and_large_meshes(gpu_ready):
    """A batch whose small meshes go to the device together, around two large ones, some
    with an indicator: items, adjacency and labels of every mesh as alone."""
    specs = [(meshgen.icosphere(2, 1, 0.02), ISO, False), (meshgen.icosphere(3, 2, 0.02), QEM, True),
             (meshgen.icosphere(6, 3, 0.02), QEM, True), (meshgen.cube(60, 4, 1e-4), ISO, False),
             (meshgen.icosphere(1, 5, 0.02), QEM, False), (meshgen.torus(33, 17, 6), ISO, True),
             (meshgen.cube(12, 7, 1e-4), QEM, True)]

    def add(ctx, k):
        (xyz, tri), metric, graded = specs[k]
        mid = ctx.add_input(xyz, tri)
        ctx.set_params(mid, number_of_clusters=len(xyz) // 15, metric=metric, unconstrained_initialization=metric,
                       seed=k, gradation=1.0 if graded else 0.0)
        if graded:
            ctx.set_indicator(mid, 1.0 + np.random.default_rng(k).random(len(xyz)))
        ctx.set_initial_labels(mid, meshgen.seed_labels(len(xyz), len(xyz) // 15, 3))

    ctx = acvd_amd.Context()
    for k in range(len(specs)):
        add(ctx, k)
    ctx.process()
    for k in range(len(specs)):
        alone = acvd_amd.Context()
        add(alone, k)
        alone.process()
        for got, want in zip((*ctx.items(k), *ctx.adjacency(k), ctx.scales(k), ctx.labels(k)),
                             (*alone.items(0), *alone.adjacency(0), alone.scales(0), alone.labels(0))):
            np.testing.assert_array_equal(got, want, err_msg=f"mesh {k}")
        alone.close()


def test_build_memory_is_given_back(gpu_ready):
    """A context of 2,097,152 items holds its arrays (258 bytes an item with 50 items
    a cluster, summed from the build's plan; 5 % for rounding) and at most 64 MiB of the
    temporaries of its build, sampling and output (88 bytes an item)."""
    import torch
    xyz, tri = meshgen.torus(2048, 1024, 5)
    torch.zeros(1, device="cuda")
    free = torch.cuda.mem_get_info()[0]
    ctx = acvd_amd.Context()
    ctx.set_input(np.asarray(xyz, np.float32), tri)
    ctx.set_params(0, number_of_clusters=len(xyz) // 50, metric=QEM, unconstrained_initialization=1)
    ctx.process()
    ctx.output(0, 1)
    held = free - torch.cuda.mem_get_info()[0]
    print(f"{held / len(xyz):.1f} bytes an item", flush=True)
    assert held <= 1.05 * 258 * len(xyz) + (64 << 20)


def test_a_context_built_again(gpu_ready):
    """One context of more than 32 MB of arrays (one allocation) taken through other
    meshes, metrics, flags and shapes, larger and smaller: labels as from a new one."""
    big = meshgen.torus(500, 400, 3)
    small = meshgen.icosphere(4, 2, 0.02)
    larger = meshgen.torus(700, 430, 4)

    def setup(ctx, meshes, metric, fixed=False, frozen=False):
        for k, (xyz, tri) in enumerate(meshes):
            mid = 0
            if k == 0:
                ctx.set_input(xyz, tri)
            else:
                mid = ctx.add_input(xyz, tri)
            K = len(xyz) // 40
            ctx.set_params(mid, number_of_clusters=K, metric=metric, unconstrained_initialization=metric, seed=9,
                           max_number_of_loops=12)
            if fixed:
                ctx.set_fixed_clusters(mid, fixed_items(len(xyz), 9, 1))
            ctx.set_initial_labels(mid, meshgen.seed_labels(len(xyz), K, 3))
            if frozen:
                ctx.set_frozen_clusters(mid, (np.arange(K) % 3 == 0).astype(np.int32))
        ctx.process()
        return [ctx.labels(k) for k in range(len(meshes))]

    steps = [dict(meshes=[big], metric=QEM, fixed=True), dict(meshes=[big], metric=ISO),
             dict(meshes=[big, small], metric=QEM), dict(meshes=[larger], metric=QEM, frozen=True),
             dict(meshes=[small], metric=ISO), dict(meshes=[small, big], metric=ISO, fixed=True),
             dict(meshes=[larger], metric=QEM)]
    ctx = acvd_amd.Context()
    for k, step in enumerate(steps):
        print(k, step["metric"], [len(m[0]) for m in step["meshes"]], flush=True)
        if k % 2:
            ctx.set_tuning(sweep_segments=512 + k)
        got = setup(ctx, **step)
        fresh = acvd_amd.Context()
        for a, b in zip(got, setup(fresh, **step)):
            np.testing.assert_array_equal(a, b, err_msg=f"step {k}")
        fresh.close()


@pytest.mark.parametrize("path", list(PATHS))
def test_timed_runs_count_the_kernels_that_ran(gpu_ready, path):
    xyz, tri = meshgen.icosphere(5, 4, 0.03)
    ctx = acvd_amd.Context()
    ctx.set_input(xyz, tri)
    ctx.set_params(0, number_of_clusters=400, metric=QEM, unconstrained_initialization=1, seed=5)
    ctx.set_initial_labels(0, meshgen.seed_labels(len(xyz), 400, 3))
    set_path(ctx, path)
    ctx.process()
    lab = ctx.labels(0)
    ctx.set_timing(True)
    ctx.process()
    np.testing.assert_array_equal(ctx.labels(0), lab)
    n, ms, passes = ctx.stats(0)["kernel_launches"], ctx.stats(0)["kernel_ms"], ctx.path_passes()
    assert n[0] == passes["list"] + passes["tiles"]
    assert n[1] == n[2] == n[3] == sum(passes.values())
    assert all((a > 0) == (b > 0) for a, b in zip(n, ms)), (n, ms)
