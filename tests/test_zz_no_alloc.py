"""fem_apply_compliance_device_noalloc, the compliance entry point that allocates nothing, against
fem_apply_compliance_device (Physics/DeformableRepresentation.cpp:175-190 is what both restate).

Two calls in a row on one GPU share its fixed workspace, the second on a smaller mesh with fewer columns,
so stale contents of the first call must not leak into the second. In FP64 mode both entry points run the
same kernels (one-launch solves of the columns side by side at these sizes) in the same batches, so the results are
equal bit for bit; in the FP32 +
refinement mode the existing entry point sends a remainder of fewer than 5 columns through the FP32 step
solver, and the two agree to the CG tolerance (bound 1e-9 relative at tolerance 1e-12).
"""
import sys

import numpy as np
import pytest

from opensurgsim_amd import femgpu
from opensurgsim_amd import meshgen as mg

from helpers import make_gpu

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def _both(g, B):
    """(existing entry point's C B, allocation-free C B) for host columns B (ndof x m)."""
    import torch
    bd = torch.from_numpy(np.ascontiguousarray(B.T)).cuda()
    x_ref = torch.zeros_like(bd)
    x_na = torch.full_like(bd, np.nan)
    torch.cuda.synchronize()
    g.apply_compliance_device(bd.data_ptr(), B.shape[1], x_ref.data_ptr())
    g.synchronize()
    g.apply_compliance_device_noalloc(bd.data_ptr(), B.shape[1], x_na.data_ptr())
    g.synchronize()
    return x_ref.cpu().numpy().T, x_na.cpu().numpy().T


@pytest.mark.parametrize("precision", [femgpu.FP64, femgpu.FP32_REFINED])
def test_noalloc_compliance_matches_existing_entry_point(precision):
    big = mg.config_corotational((9, 7, 8), seed=5)
    small = mg.config_corotational((4, 3, 5), seed=6)
    say("noalloc compliance: precision", precision, "dofs", big.x0.size, "then", small.x0.size)
    results = []
    for cfg, ncols, seed in ((big, 11, 1), (small, 3, 2)):
        g = make_gpu(cfg, precision=precision, tol=1e-12)
        assert g.step(3) == femgpu.FEM_OK
        B = np.random.default_rng(seed).normal(size=(cfg.x0.size, ncols))
        X_ref, X_na = _both(g, B)
        say("  ncols", ncols, "max |diff|", float(np.max(np.abs(X_ref - X_na))))
        assert np.all(np.isfinite(X_na))
        if precision == femgpu.FP64:
            assert np.array_equal(X_na, X_ref)
        else:
            for j in range(ncols):
                assert np.linalg.norm(X_na[:, j] - X_ref[:, j]) <= 1e-9 * np.linalg.norm(X_ref[:, j])
        # boundary rows of the solutions are zero, as applyCompliance leaves them
        for n in cfg.bc_nodes:
            assert np.all(X_na[3 * n:3 * n + 3] == 0.0)
        results.append(X_na)
        g.close()
    assert results[1].shape == (small.x0.size, 3)


def test_noalloc_compliance_rejections():
    import torch
    cfg = mg.config_corotational((3, 3, 3), seed=4)
    g = make_gpu(cfg, tol=1e-12)
    bd = torch.zeros((1, cfg.x0.size), dtype=torch.float64, device="cuda")
    with pytest.raises(femgpu.FemError) as e:  # no system matrix before the first step
        g.apply_compliance_device_noalloc(bd.data_ptr(), 1, bd.data_ptr())
    assert e.value.code == femgpu.FEM_ERR_ORDER
    g.close()
    # a mesh beyond the workspace: 45^3 cubes, 97,336 nodes, 292,008 DOFs
    big = mg.config_corotational((45, 45, 45), seed=4)
    say("noalloc compliance: oversize mesh dofs", big.x0.size)
    g = femgpu.FemGpu(0)
    g.upload_mesh(big.kind, big.x0, big.conn, big.E, big.nu, big.rho)
    bd = torch.zeros((1, big.x0.size), dtype=torch.float64, device="cuda")
    with pytest.raises(femgpu.FemError) as e:
        g.apply_compliance_device_noalloc(bd.data_ptr(), 1, bd.data_ptr())
    assert e.value.code == femgpu.FEM_ERR_INVALID and "at most" in str(e.value)
    g.close()
