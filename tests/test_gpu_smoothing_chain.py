"""Smoothing chain of the matrix-free V-cycle (each patch kernel completes the
Chebyshev step before it): on both sides of the patch counts up to which it
runs (FP64 256, FP32 512) and for one, two and three smoothing steps, whose
buffers change places differently, the cycle is the per-element path's, and
its last step's rho starts a solve that converges to the true residual.  The
two paths differ by rounding alone, which the cycle (a smoothing operator)
does not amplify: 1e-13 in FP64 and 1e-5 in FP32 of the result's norm."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float((a.double() - b.double()).norm() / b.double().norm())


@pytest.mark.parametrize("cells,patches,degree", [((9, 1, 1), 1, 2), ((42, 13, 5), 256, 1), ((38, 9, 8), 257, 2),
                                                  ((60, 13, 7), 512, 3), ((57, 12, 8), 513, 3), ((60, 13, 7), 512, 2)])
def test_chain_is_the_per_element_cycle(cells, patches, degree):
    import torch
    from wnfea_amd.mesh.solid_generator import generate_c3d10_structured_block
    from wnfea_amd.solver.solid_solver import (MatrixFreeOperator, assemble_c3d10_bsr, build_amg, solve_mixed,
                                               true_residual)
    print(f"smoothing chain on {cells}, degree {degree}", flush=True)
    nx, ny, nz = cells
    m, _ = generate_c3d10_structured_block(0.025 * nx, 0.02 * ny, 0.02 * nz, nx, ny, nz, tip_load_total=-1000.0,
                                           tets_per_hex=6, load_direction="z")
    system = assemble_c3d10_bsr(m, want_fp64_equilibrated=True)
    amg = build_amg(system, storage=("fp64", "fp32"), autotune=False, level_degrees=[degree])
    op = MatrixFreeOperator(system)
    try:
        assert op.patch_info["patches"] == patches and op.patch_info["elems"] == 64
        op.attach_smoother(amg)
        rd = torch.as_tensor(np.random.default_rng(7).standard_normal(system.n_dofs), device="cuda")
        z64, z32 = amg.vcycle(rd), amg.vcycle(rd.float())
        assert torch.equal(amg.vcycle(rd), z64) and torch.equal(amg.vcycle(rd.float()), z32)
        for prec in ("fp64", "fp32"):
            u, _, _, rel, _ = solve_mixed(system, amg, tol=1e-8, amg_precision=prec, operator=op)
            assert rel <= 1e-8 and true_residual(system, u) <= 1.5e-8, prec
        op.set_patch(0)  # per-element products (re-attaches the hierarchy)
        assert _rel(z64, amg.vcycle(rd)) <= 1e-13
        assert _rel(z32, amg.vcycle(rd.float())) <= 1e-5
    finally:
        op.close()
        amg.close()
