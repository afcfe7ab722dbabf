"""Several load cases on a hierarchy whose coarse spaces hold the translations
alone (a system without node coordinates): its coarser levels and transfers
have 3x3 blocks, where those of the rigid-body modes have 6x6."""
import dataclasses

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("group", [4, 8])
def test_load_cases_without_coordinates(group):
    import torch
    from oracle import oracle as O
    from wnfea_amd.mesh.solid_generator import generate_c3d10_structured_block
    from wnfea_amd.solver.solid_solver import assemble_c3d10_bsr, build_amg, solve_multi
    m, _ = generate_c3d10_structured_block(1.0, 0.1, 0.1, 20, 2, 2, tip_load_total=-1000.0, tets_per_hex=6,
                                           load_direction="z")
    system = dataclasses.replace(assemble_c3d10_bsr(m), coords=None)
    amg = build_amg(system, storage=("fp32",), autotune=False, coarse_size=100)
    B = np.random.default_rng(3).standard_normal((system.n_dofs, 5))
    B[system.fixed_mask] = 0.0
    try:
        assert [lv.A.blocksize for lv in amg.levels] == [(3, 3)] * 3
        U, _, rels, _ = solve_multi(system, amg, torch.as_tensor(B, device="cuda"), tol=1e-8, group=group)
    finally:
        amg.close()
    E, nu = m.element_moduli()
    K, _ = O.assemble_csr(m.mesh_nodes, m.solid_elements, E, nu, m.fixed_dof_mask(3), m.load_vector(3))
    R = B - K @ U.cpu().numpy()
    # the solver's own residual, and the same with the oracle's matrix (its rounding is far below 1e-8)
    assert np.all(rels <= 1e-8)
    assert np.all(np.linalg.norm(R, axis=0) <= 2e-8 * np.linalg.norm(B, axis=0))
