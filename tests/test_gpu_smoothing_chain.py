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


@pytest.mark.parametrize("degree", [1, 2])
def test_nodes_of_no_element_take_the_node_kernels(degree):
    """A clamped node that belongs to no element, and so to no patch, amid the
    others and one at their end: the chain, whose patches store the steps of
    the nodes they hold, stays off, and the cycle is the per-element path's on
    every node, these two included."""
    import dataclasses

    import torch
    from wnfea_amd.mesh.solid_generator import generate_c3d10_structured_block
    from wnfea_amd.solver.solid_solver import (MatrixFreeOperator, assemble_c3d10_bsr, build_amg, solve_mixed,
                                               true_residual)
    print(f"nodes of no element, degree {degree}", flush=True)
    m, _ = generate_c3d10_structured_block(0.3, 0.04, 0.04, 12, 2, 2, tip_load_total=-1000.0, tets_per_hex=6,
                                           load_direction="z")
    n, k = len(m.mesh_nodes), 100
    m.mesh_nodes = np.vstack([m.mesh_nodes[:k], [[0.1, 0.1, 0.1]], m.mesh_nodes[k:], [[0.2, 0.1, 0.1]]])
    m.solid_elements = m.solid_elements + (m.solid_elements >= k)
    clamp = m.supports[0]
    for item in (*m.supports, *m.loads):
        item.node_id += int(item.node_id >= k)
    m.supports += [dataclasses.replace(clamp, node_id=i) for i in (k, n + 1)]
    system = assemble_c3d10_bsr(m, want_fp64_equilibrated=True)
    own = torch.tensor([3 * k, 3 * k + 1, 3 * k + 2, 3 * n + 3, 3 * n + 4, 3 * n + 5], device="cuda")
    assert bool(torch.as_tensor(system.fixed_mask, device="cuda")[own].all())
    amg = build_amg(system, storage=("fp64", "fp32"), autotune=False, level_degrees=[degree], coarse_size=400)
    op = MatrixFreeOperator(system)
    try:
        op.attach_smoother(amg)
        rd = torch.as_tensor(np.random.default_rng(7).standard_normal(system.n_dofs), device="cuda")
        z64, z32 = amg.vcycle(rd), amg.vcycle(rd.float())
        for prec in ("fp64", "fp32"):
            u, _, _, rel, _ = solve_mixed(system, amg, tol=1e-8, amg_precision=prec, operator=op)
            assert rel <= 1e-8 and true_residual(system, u) <= 1.5e-8, prec
        op.set_patch(0)
        z64e, z32e = amg.vcycle(rd), amg.vcycle(rd.float())
        assert _rel(z64, z64e) <= 1e-13 and _rel(z32, z32e) <= 1e-5
        assert _rel(z64[own], z64e[own]) <= 1e-13 and _rel(z32[own], z32e[own]) <= 1e-5
    finally:
        op.close()
        amg.close()
