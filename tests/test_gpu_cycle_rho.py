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
