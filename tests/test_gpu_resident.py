"""The one-launch CG (the operator held on the chip) against the CG with one launch per iteration.

Both solve to cg_tolerance TOL = 1e-12, so a step's velocities differ by at most a few TOL times the operator's
conditioning (dt^2 K / M <= 1e2 at these sizes): 1e-9 in FP64 and with the FP64 refinement around FP32 alike, whose
outer test is the same. The recurrence is the same, so the iteration counts differ by at most one (the sums are bracketed
differently) on the block meshes; FP32 inner solves, and the hundreds of iterations that the slivers of a random mesh take,
follow their own rounding, so their counts are not compared.
"""
import functools
import threading
import time

import numpy as np
import pytest

from opensurgsim_amd import femgpu
from opensurgsim_amd import meshgen as mg

pytestmark = pytest.mark.gpu
TOL, BOUND = 1e-12, 1e-9


def block(n):
    x0, tets, _ = mg.block_tet_mesh(*n)
    return x0, tets, mg.face_nodes(*n, 1, 0)


def irregular(points=900, seed=3):
    """Delaunay mesh of random points (uneven node degrees) with a node that no element uses."""
    from scipy.spatial import Delaunay
    p = np.random.RandomState(seed).rand(points, 3) * 0.1
    t = Delaunay(p).simplices
    vol = mg.tet_volumes(p, t)
    t[vol < 0] = t[vol < 0][:, [0, 1, 3, 2]]
    t = t[np.abs(vol) > 2e-9]
    used = np.unique(t)
    remap = np.full(points, -1)
    remap[used] = np.arange(used.size)
    return np.concatenate([p[used], [[0.2, 0.2, 0.2]]]), remap[t].astype(np.int32), np.arange(5)


def star(points):
    """A hub joined to every point of a sphere: one block row of points + 1 blocks, and as many halo columns."""
    from scipy.spatial import ConvexHull
    k = np.arange(points) + 0.5
    ph, th = np.arccos(1 - 2 * k / points), np.pi * (1 + 5 ** 0.5) * k
    p = 0.1 * np.stack([np.cos(th) * np.sin(ph), np.sin(th) * np.sin(ph), np.cos(ph)], 1)
    tri = ConvexHull(p).simplices
    t = np.concatenate([np.full((len(tri), 1), points), tri], 1)
    x0 = np.concatenate([p, [[0.0, 0.0, 0.0]]])
    vol = mg.tet_volumes(x0, t)
    t[vol < 0] = t[vol < 0][:, [0, 1, 3, 2]]
    return x0, t.astype(np.int32), np.arange(3)


def run(mesh, precision, steps=2, **opts):
    x0, tets, bc = mesh
    g = femgpu.FemGpu(0)
    g.upload_mesh(femgpu.TET_COROTATIONAL, x0, tets, 5e4, 0.4, 1000.0)
    g.add_bc_nodes(bc)
    g.set_options(**dict(dict(dt=1e-3, cg_tolerance=TOL, precision=precision), **opts))
    g.set_state(v=0.01 * np.random.RandomState(1).standard_normal(x0.size))
    its = []
    for _ in range(steps):
        assert g.step(1) == femgpu.FEM_OK
        its.append(g.stats()["last_cg_iterations"])
    x, v = g.state()
    conv = g.stats()["converged"]
    g.close()
    return x, v, its, conv


def both(monkeypatch, mesh, precision, **kw):
    monkeypatch.delenv("FEM_CG_KERNELS", raising=False)
    a = run(mesh, precision, **kw)
    monkeypatch.setenv("FEM_CG_KERNELS", "fused")
    return a, run(mesh, precision, **kw)


def same(a, b, precision, counts=True):
    assert np.linalg.norm(a[1] - b[1]) <= BOUND * np.linalg.norm(b[1])
    assert np.linalg.norm(a[0] - b[0]) <= BOUND * np.linalg.norm(b[0])
    if counts and precision == femgpu.FP64:
        assert all(abs(i - j) <= 1 for i, j in zip(a[2], b[2])), (a[2], b[2])
    assert a[3] == b[3] == 1


# one workgroup, two, an odd count; the fewest and the most blocks per lane; the largest meshes that fit
@pytest.mark.parametrize("n", [(1, 1, 1), (3, 3, 3), (5, 4, 6), (9, 7, 8), (21, 18, 20), (34, 33, 35), (40, 40, 40)])
@pytest.mark.parametrize("precision", [femgpu.FP64, femgpu.FP32_REFINED])
def test_block_meshes(monkeypatch, n, precision):
    a, b = both(monkeypatch, block(n), precision)
    same(a, b, precision)


@pytest.mark.parametrize("precision", [femgpu.FP64, femgpu.FP32_REFINED])
def test_beyond_the_chip_and_largest_fp32(monkeypatch, precision):
    a, b = both(monkeypatch, block((50, 48, 49)), precision, steps=1)
    same(a, b, precision)


# FP32 CG does not converge on the random mesh's slivers, with either CG: FP64 alone there
@pytest.mark.parametrize("mesh, precision", [(irregular, femgpu.FP64)] + [
    (functools.partial(star, n), p) for n in (700, 1500) for p in (femgpu.FP64, femgpu.FP32_REFINED)])
def test_uneven_rows(monkeypatch, mesh, precision):
    a, b = both(monkeypatch, mesh(), precision)
    same(a, b, precision, counts=False)


@pytest.mark.parametrize("cap", [1, 2, 5])
def test_iteration_cap(monkeypatch, cap):
    a, b = both(monkeypatch, block((6, 7, 5)), femgpu.FP64, cg_max_iterations=cap, steps=1)
    assert a[2] == b[2] == [cap] and a[3] == b[3] == 0
    assert np.linalg.norm(a[1] - b[1]) <= 1e-12 * np.linalg.norm(b[1])


def test_zero_right_hand_side():
    x0, tets, bc = block((3, 3, 3))
    g = femgpu.FemGpu(0)
    g.upload_mesh(femgpu.TET_COROTATIONAL, x0, tets, 5e4, 0.4, 1000.0)
    g.add_bc_nodes(bc)
    g.set_options(dt=1e-3, cg_tolerance=TOL, gravity_enabled=0)
    for _ in range(3):
        assert g.step(1) == femgpu.FEM_OK
    x, v = g.state()
    assert g.stats()["last_cg_iterations"] == 0 and not v.any() and np.array_equal(x, x0.reshape(-1))
    g.close()


@pytest.mark.parametrize("precision", [femgpu.FP64, femgpu.FP32_REFINED])
def test_gives_up_waiting_and_solves_anyway(monkeypatch, precision):
    """No wait is allowed: the first one gives up, and the solve goes on with one launch per iteration."""
    mesh = block((12, 11, 13))
    monkeypatch.delenv("FEM_CG_KERNELS", raising=False)
    monkeypatch.setenv("FEM_CG_WAIT_US", "0")
    a = run(mesh, precision, steps=3)
    monkeypatch.delenv("FEM_CG_WAIT_US")
    b = run(mesh, precision, steps=3)
    same(a, b, precision)


def test_repeats_bit_for_bit_and_from_threads(monkeypatch):
    monkeypatch.delenv("FEM_CG_KERNELS", raising=False)
    meshes = [block((12, 11, 13)), block((21, 18, 20))]
    want = [run(m, femgpu.FP64, steps=6) for m in meshes]
    got = [None, None]

    def work(i):
        got[i] = run(meshes[i], femgpu.FP64, steps=6)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    for w, g in zip(want, got):
        assert np.array_equal(w[0], g[0]) and np.array_equal(w[1], g[1])


def test_changes_between_precisions(monkeypatch):
    """A context that changes between FP64 and FP32 + refinement: FP64 frames are those of a context that stays in FP64 bit for
    bit, and only the first change to each waits for its partition of the mesh on the host (3 ms and more at this size, a later
    change 0.1 ms)."""
    monkeypatch.delenv("FEM_CG_KERNELS", raising=False)
    x0, tets, bc = block((40, 40, 40))
    v0 = 0.01 * np.random.RandomState(1).standard_normal(x0.size)
    g, h = femgpu.FemGpu(0), femgpu.FemGpu(0)
    for c in (g, h):
        c.upload_mesh(femgpu.TET_COROTATIONAL, x0, tets, 5e4, 0.4, 1000.0)
        c.add_bc_nodes(bc)
    h.set_options(dt=1e-3, cg_tolerance=TOL, precision=femgpu.FP64)
    h.set_state(x0, v0)
    assert h.step(1) == femgpu.FEM_OK
    want = h.state()
    took = []
    for _ in range(5):
        took.append(0.0)
        for precision in (femgpu.FP64, femgpu.FP32_REFINED):
            t0 = time.perf_counter()
            g.set_options(dt=1e-3, cg_tolerance=TOL, precision=precision)
            took[-1] += time.perf_counter() - t0
            g.set_state(x0, v0)
            assert g.step(1) == femgpu.FEM_OK
            x, v = g.state()
            if precision == femgpu.FP64:
                assert np.array_equal(x, want[0]) and np.array_equal(v, want[1])
            else:
                assert np.linalg.norm(v - want[1]) <= BOUND * np.linalg.norm(want[1])
    print("two changes: %s ms" % " ".join("%.2f" % (1e3 * t) for t in took), flush=True)
    assert min(took[1:]) < 0.5 * took[0]
    g.close()
    h.close()


def test_small_body_beside_a_long_solve():
    """A body of 4 workgroups steps beside one of 25 whose solves take hundreds of iterations, on its own stream from another
    thread: it does not wait for the other's solve to end. Its median frame is held to half of the other's; it took 0.16 of it
    alone and all of it when one solve kept out every other one."""
    def body(n, young):
        x0, tets, bc = block(n)
        g = femgpu.FemGpu(0)
        g.upload_mesh(femgpu.TET_COROTATIONAL, x0, tets, young, 0.45, 1000.0)
        g.add_bc_nodes(bc)
        g.set_options(dt=1e-3, cg_tolerance=1e-8)
        return g, x0, 0.01 * np.random.RandomState(1).standard_normal(x0.size)

    def frames(b, more):
        t, i = [], 0
        while more(i):
            if i % 10 == 0:
                b[0].set_state(b[1], b[2])
            t0 = time.perf_counter()
            assert b[0].step(1) == femgpu.FEM_OK
            t.append(time.perf_counter() - t0)
            i += 1
        return sorted(t)[len(t) // 2]

    small, large = body((7, 8, 6), 5e4), body((14, 14, 14), 5e6)
    for b in (small, large):
        frames(b, lambda i: i < 20)
    stop, got = threading.Event(), []
    thread = threading.Thread(target=lambda: got.append(frames(large, lambda i: not stop.is_set())))
    thread.start()
    try:
        beside = frames(small, lambda i: i < 300)
    finally:
        stop.set()
        thread.join(60)
    print("median frame beside: %.3f ms, the other's %.3f ms" % (1e3 * beside, 1e3 * got[0]), flush=True)
    assert beside < 0.5 * got[0]
    small[0].close()
    large[0].close()


def run_batch(sizes, precision, steps=2):
    off, parts = [0], []
    for n in sizes:
        x0, tets, bc = block(n)
        parts.append((x0, tets + off[-1], bc + off[-1]))
        off.append(off[-1] + len(x0))
    x0, tets, bc = (np.concatenate([p[i] for p in parts]) for i in range(3))
    g = femgpu.FemGpu(0)
    g.upload_mesh(femgpu.TET_COROTATIONAL, x0, tets.astype(np.int32), 5e4, 0.4, 1000.0)
    g.add_bc_nodes(bc)
    g.set_batch_tuning(128, 8)
    g.set_instances(off, np.resize([5e-4, 1e-3, 2e-3], len(sizes)))
    g.set_options(dt=1e-3, cg_tolerance=TOL, precision=precision)
    g.set_state(v=0.01 * np.random.RandomState(1).standard_normal(x0.size))
    assert g.step(steps) == femgpu.FEM_OK
    x, v = g.state()
    its, _, conv = g.instance_stats()
    g.close()
    return x, v, its, conv


# one instance, uneven ones in one launch, more than one launch holds, and one that does not fit beside others that do
@pytest.mark.parametrize("sizes", [[(4, 5, 3)], [(3, 3, 3), (9, 8, 7), (14, 3, 6), (6, 6, 6), (20, 18, 19)],
                                   [(10, 9, 11)] * 70, [(48, 50, 49), (5, 5, 5), (12, 9, 10)]],
                         ids=["one", "uneven", "launches", "oversize"])
@pytest.mark.parametrize("precision", [femgpu.FP64, femgpu.FP32_REFINED])
def test_batches(monkeypatch, sizes, precision):
    monkeypatch.delenv("FEM_CG_KERNELS", raising=False)
    a = run_batch(sizes, precision)
    monkeypatch.setenv("FEM_CG_KERNELS", "fused")
    b = run_batch(sizes, precision)
    for i in (0, 1):
        assert np.linalg.norm(a[i] - b[i]) <= BOUND * np.linalg.norm(b[i])
    assert a[3].all() and b[3].all()
    if precision == femgpu.FP64:
        assert np.abs(a[2] - b[2]).max() <= 1


def test_batch_gives_up_waiting(monkeypatch):
    sizes = [(6, 7, 5), (9, 8, 7)]
    monkeypatch.delenv("FEM_CG_KERNELS", raising=False)
    b = run_batch(sizes, femgpu.FP64)
    monkeypatch.setenv("FEM_CG_WAIT_US", "0")
    a = run_batch(sizes, femgpu.FP64)
    assert np.linalg.norm(a[1] - b[1]) <= BOUND * np.linalg.norm(b[1])


# fewer columns than fit side by side, more, and a mesh that takes the chip alone; a zero column among them. With no wait allowed
# the step gives up first where it has several workgroups, and the columns go on with the launch per iteration from the start
@pytest.mark.parametrize("n, columns", [((3, 4, 3), 1), ((3, 4, 3), 70), ((12, 11, 13), 11), ((34, 33, 35), 3)])
@pytest.mark.parametrize("wait", [None, "0"])
def test_compliance_columns(monkeypatch, n, columns, wait):
    x0, tets, bc = block(n)
    B = np.random.RandomState(2).standard_normal((x0.size, columns))
    B[:, columns // 2] = 0.0 if columns > 1 else B[:, 0]
    got = []
    for env in (None, "fused"):
        monkeypatch.setenv("FEM_CG_KERNELS", env) if env else monkeypatch.delenv("FEM_CG_KERNELS", raising=False)
        monkeypatch.setenv("FEM_CG_WAIT_US", wait) if wait else monkeypatch.delenv("FEM_CG_WAIT_US", raising=False)
        g = femgpu.FemGpu(0)
        g.upload_mesh(femgpu.TET_COROTATIONAL, x0, tets, 5e4, 0.4, 1000.0)
        g.add_bc_nodes(bc)
        g.set_options(dt=1e-3, cg_tolerance=TOL)
        assert g.step(1) == femgpu.FEM_OK
        got.append(g.apply_compliance(B))
        g.close()
    for j in range(columns):
        assert np.linalg.norm(got[0][:, j] - got[1][:, j]) <= BOUND * np.linalg.norm(got[1][:, j])
    for node in bc:
        assert not got[0][3 * node:3 * node + 3].any()


@pytest.mark.parametrize("entry", ["device", "noalloc", "host"])
def test_columns_give_up_waiting(monkeypatch, entry):
    """Columns that give up themselves: the step before them is the direct solver's, so that they are the context's first
    conjugate gradients. They are solved again by the multi-column CG, whose rounding is another one, and so equal those of a
    context without one-launch solves bit for bit; with the usual limit the same calls do not."""
    import torch
    x0, tets, bc = block((12, 11, 13))
    b = torch.from_numpy(np.random.RandomState(4).standard_normal((11, x0.size))).cuda()
    got = {}
    for kernels, wait in ((None, "0"), (None, None), ("fused", None)):
        monkeypatch.setenv("FEM_CG_KERNELS", kernels) if kernels else monkeypatch.delenv("FEM_CG_KERNELS", raising=False)
        monkeypatch.setenv("FEM_CG_WAIT_US", wait) if wait else monkeypatch.delenv("FEM_CG_WAIT_US", raising=False)
        g = femgpu.FemGpu(0)
        g.upload_mesh(femgpu.TET_COROTATIONAL, x0, tets, 5e4, 0.4, 1000.0)
        g.add_bc_nodes(bc)
        g.set_options(dt=1e-3, linear_solver=femgpu.LINEAR_SOLVER_LU)
        assert g.step(1) == femgpu.FEM_OK
        g.set_options(dt=1e-3, cg_tolerance=TOL)
        if entry == "host":
            got[kernels, wait] = g.apply_compliance(b.cpu().numpy().T).T
        else:
            out = torch.full_like(b, np.nan)
            torch.cuda.synchronize()
            (g.apply_compliance_device if entry == "device" else g.apply_compliance_device_noalloc)(
                b.data_ptr(), len(b), out.data_ptr())
            g.synchronize()
            got[kernels, wait] = out.cpu().numpy()
        g.close()
    want = got["fused", None]
    assert np.array_equal(got[None, "0"], want)
    assert not np.array_equal(got[None, None], want)
    assert np.linalg.norm(got[None, None] - want) <= BOUND * np.linalg.norm(want)
