"""CG whose cycle forms rho = r . (S z) in its last smoothing step, on
assembled 3- and 6-blocks: six iterations equal a numpy CG that applies the
same device cycle and forms rho itself.  FP64 cycles differ by the order of
the sums alone (1e-11 of the iterate after six steps); an FP32 cycle may round
its input the other way where r differs in the last bit (1e-5).  Row counts at
and off the 64-row slices."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _system(dpn, nx):
    import scipy.sparse as sp
    from wnfea_amd.solver.solid_solver import system_from_csr
    def lap(n):
        return sp.diags([-np.ones(n - 1), 2.0 * np.ones(n), -np.ones(n - 1)], [-1, 0, 1])
    I = sp.identity
    L = sp.kron(sp.kron(lap(nx), I(4)), I(4)) + sp.kron(sp.kron(I(nx), lap(4)), I(4)) \
        + sp.kron(sp.kron(I(nx), I(4)), lap(4))
    rng = np.random.default_rng(dpn)
    q = np.linalg.qr(rng.standard_normal((dpn, dpn)))[0]
    block = q @ np.diag(np.linspace(1.0, 5.0, dpn)) @ q.T
    n = nx * 16
    D = sp.diags(np.repeat(np.exp(rng.uniform(-1.0, 1.0, n)), dpn))
    K = (D @ sp.kron(L + 0.01 * I(n), block) @ D).tocsr()
    K = (0.5 * (K + K.T)).tocsr()
    xyz = np.stack(np.meshgrid(np.arange(nx), np.arange(4), np.arange(4), indexing="ij"), -1).reshape(-1, 3)
    f = rng.standard_normal(dpn * n)
    return K, f, system_from_csr(K, f, coords=xyz.astype(float), want_fp64_equilibrated=True, dpn=dpn)


@pytest.mark.parametrize("nx", [13, 16, 41])
@pytest.mark.parametrize("dpn", [3, 6])
@pytest.mark.parametrize("precision,cycle", [("fp64", "fp64"), ("fp64", "fp32"), ("fp64_equilibrated", "fp64")])
def test_cg_iterates(dpn, nx, precision, cycle):
    import torch
    from wnfea_amd.solver.solid_solver import build_amg, pcg_device
    print(f"cycle rho: {dpn}-blocks, {16 * nx} rows, {precision} with a {cycle} cycle", flush=True)
    K, f, system = _system(dpn, nx)
    amg = build_amg(system, storage=("fp64", "fp32"), autotune=False, coarse_size=150)
    assert len(amg.levels) >= 2
    x, it, _, _ = pcg_device(system, rtol=1e-30, max_iter=6, preconditioner="amg", precision=precision, amg=amg,
                             amg_precision=cycle)
    assert it == 6
    s = system.scale.cpu().numpy()
    dt = torch.float32 if cycle == "fp32" else torch.float64
    r, u, p, rho0 = f.copy(), np.zeros_like(f), 0.0, 1.0
    for k in range(6):
        z = s * amg.vcycle(torch.as_tensor(s * r, device="cuda").to(dt)).double().cpu().numpy()
        rho = r @ z
        p = z + (rho / rho0 if k else 0.0) * p
        q = K @ p
        a = rho / (p @ q)
        u, r, rho0 = u + a * p, r - a * q, rho
    err = np.linalg.norm(x.cpu().numpy() - u) / np.linalg.norm(u)
    assert err <= (1e-11 if cycle == "fp64" else 1e-5), err
    amg.close()
    system.K.close()


@pytest.mark.parametrize("dpn,cycle", [(3, "fp64"), (3, "fp32"), (6, "fp64"), (6, "fp32")])
def test_carried_finalisation_changes_nothing(dpn, cycle):
    """Chunks of one iteration finalise ||r||^2 in a launch of their own, longer
    ones in the next iteration's first kernel: the same sums in the same order,
    so the same bits and the same last iteration."""
    import torch
    from wnfea_amd.solver.solid_solver import build_amg, pcg_device
    print(f"carried finalisation: {dpn}-blocks, {cycle} cycle", flush=True)
    _, _, system = _system(dpn, 41)
    amg = build_amg(system, storage=("fp64", "fp32"), autotune=False, coarse_size=150)
    runs = [pcg_device(system, rtol=1e-9, preconditioner="amg", amg=amg, amg_precision=cycle, check_every=k)
            for k in (1, 2, 5, 16)]
    assert 5 < runs[0][1] < 200 and runs[0][2] <= 1e-9
    for x, it, rel, _ in runs[1:]:
        assert it == runs[0][1] and rel == runs[0][2] and torch.equal(x, runs[0][0])
    amg.close()
    system.K.close()


@pytest.mark.parametrize("cells,cycle", [((9, 1, 1), "fp64"), ((20, 4, 4), "fp32"), ((57, 12, 8), "fp32")])
def test_carried_finalisation_matrix_free(cells, cycle):
    import torch
    from wnfea_amd.mesh.solid_generator import generate_c3d10_structured_block
    from wnfea_amd.solver.solid_solver import MatrixFreeOperator, assemble_c3d10_bsr, build_amg, solve_mixed
    print(f"carried finalisation on a box of {cells} cells, {cycle} cycle", flush=True)
    nx, ny, nz = cells
    m, _ = generate_c3d10_structured_block(0.025 * nx, 0.02 * ny, 0.02 * nz, nx, ny, nz, tip_load_total=-1000.0,
                                           tets_per_hex=6, load_direction="z")
    system = assemble_c3d10_bsr(m, want_fp64_equilibrated=True)
    amg = build_amg(system, storage=("fp64", "fp32"), autotune=False, coarse_size=200)
    op = MatrixFreeOperator(system)
    op.attach_smoother(amg)
    runs = [solve_mixed(system, amg, tol=1e-8, amg_precision=cycle, operator=op, check_every=k) for k in (1, 3, 16)]
    for u, it, _, rel, _ in runs:
        assert it == runs[0][1] and rel == runs[0][3] <= 1e-8 and torch.equal(u, runs[0][0])
    op.close()
    amg.close()


@pytest.mark.timeout(120)
@pytest.mark.parametrize("nx", [5120, 5121])
def test_cg_iterates_where_the_rho_pass_returns(nx):
    """On both sides of the 2 560 partials (slices of 32 rows, padded to the 8
    XCDs) up to which the last product forms rho."""
    test_cg_iterates(3, nx, "fp64", "fp64")
