"""Dense coarsest product: by rows up to 32 MB of inverse, by packed symmetric
64 x 64 tiles beyond.  Hierarchies of one level on both sides of the line in
FP64 (2 048 rows) and FP32 (2 896), at sizes that leave a partial last tile and
a partial last round of a row; the cycle must be inv @ r, in FP32 of the
inverse rounded to FP32 with the sum in FP64 and the result rounded once."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells,rows", [((1, 1, 1), 81), ((16, 2, 2), 2475), ((20, 2, 2), 3075)])
def test_cycle_is_the_inverse_product(cells, rows):
    import torch
    from wnfea_amd.mesh.solid_generator import generate_c3d10_structured_block
    from wnfea_amd.solver.solid_solver import assemble_c3d10_bsr, build_amg
    print(f"coarsest product of {rows} rows", flush=True)
    m, _ = generate_c3d10_structured_block(1.0, 0.1, 0.1, *cells, tip_load_total=-1000.0, tets_per_hex=6,
                                           load_direction="z")
    amg = build_amg(assemble_c3d10_bsr(m, want_fp64_equilibrated=True), storage=("fp64", "fp32"), autotune=False)
    inv = amg.coarse_inv
    assert len(amg.levels) == 1 and inv.shape[0] == rows
    r = np.random.default_rng(rows).standard_normal(rows)
    z = amg.vcycle(torch.as_tensor(r, device="cuda")).cpu().numpy()
    # a sum of `rows` products in another order: rows * eps of the sum of magnitudes
    assert np.all(np.abs(z - inv @ r) <= rows * 2.3e-16 * (np.abs(inv) @ np.abs(r)))
    r32, inv32 = r.astype(np.float32), inv.astype(np.float32).astype(np.float64)
    z32 = amg.vcycle(torch.as_tensor(r32, device="cuda")).double().cpu().numpy()
    ref = inv32 @ r32.astype(np.float64)
    # one rounding of the result to FP32, plus the FP64 sum's as above
    mag = np.abs(inv32) @ np.abs(r32.astype(np.float64))
    assert np.all(np.abs(z32 - ref) <= 6.0e-8 * np.abs(ref) + rows * 2.3e-16 * mag)
    amg.close()


def test_captured_iterations_follow_the_coarse_precision():
    """Sixteen captured CG iterations with the FP32 cycle's coarsest product
    switched between the FP32 and the FP64 inverse: the bits of host launches
    at each setting, also where the iterations of another one were captured
    last."""
    import torch
    from wnfea_amd.mesh.solid_generator import generate_c3d10_structured_block
    from wnfea_amd.solver.solid_solver import assemble_c3d10_bsr, build_amg, pcg_device, set_graphs
    m, _ = generate_c3d10_structured_block(1.0, 0.1, 0.1, 20, 2, 2, tip_load_total=-1000.0, tets_per_hex=6,
                                           load_direction="z")
    system = assemble_c3d10_bsr(m, want_fp64_equilibrated=True)
    amg = build_amg(system, storage=("fp64", "fp32"), autotune=False, coarse_size=600)
    kw = dict(rtol=1e-30, max_iter=16, check_every=8, preconditioner="amg", precision="fp64", amg=amg,
              amg_precision="fp32")
    host, got = {}, []
    try:
        assert len(amg.levels) == 2
        for prec in ("fp32", "fp64"):
            amg.set_coarse_precision(prec)
            host[prec] = pcg_device(system, **kw)[0].cpu()
        assert not torch.equal(host["fp32"], host["fp64"])
        set_graphs(True)
        for prec in ("fp32", "fp64", "fp64", "fp32"):
            amg.set_coarse_precision(prec)
            x = pcg_device(system, **kw)[0]
            got.append((prec, x.data_ptr(), x.cpu()))
            del x  # the next call's solution takes its place
    finally:
        set_graphs(False)
        amg.close()
    assert len({p for _, p, _ in got}) == 1  # the same buffers throughout
    for prec, _, x in got:
        assert torch.equal(x, host[prec]), prec


@pytest.mark.parametrize("group", [4, 8])
@pytest.mark.parametrize("cells,rows", [((1, 1, 1), 81), ((3, 1, 1), 189), ((16, 2, 2), 2475), ((20, 2, 2), 3075)])
def test_columns_are_the_inverse_product(cells, rows, group):
    """Several columns on a hierarchy of one level, whose rows end inside a run
    of 32 columns and a block of 16 rows.  The first CG iterate of column k is
    alpha_k S z_k, z_k = inv32 (S b_k)_32 with the sum in FP64 and rounded
    once: alpha_k, one factor per column, is taken from the median entry,
    which adds that entry's own rounding."""
    import torch
    from wnfea_amd import _lib
    from wnfea_amd.mesh.solid_generator import generate_c3d10_structured_block
    from wnfea_amd.solver.solid_solver import _Solver, assemble_c3d10_bsr, build_amg
    print(f"coarsest product of {rows} rows, {group} columns", flush=True)
    m, _ = generate_c3d10_structured_block(0.05 * cells[0], 0.1, 0.1, *cells, tip_load_total=-1000.0, tets_per_hex=6,
                                           load_direction="z")
    system = assemble_c3d10_bsr(m)
    amg = build_amg(system, storage=("fp32",), autotune=False)
    assert len(amg.levels) == 1 and amg.coarse_inv.shape[0] == rows
    B = np.random.default_rng(rows).standard_normal((rows, group))
    Bd = torch.as_tensor(B, device="cuda")
    X = torch.empty_like(Bd)
    its, rel = (_lib.ctypes.c_int * group)(), (_lib.ctypes.c_double * group)()
    _lib.check(_lib.load().wnfea_pcg_multi(_Solver.get(), system.K.handle, amg.handle, 1, _lib.dptr(system.scale), group,
                                           _lib.dptr(Bd), _lib.dptr(X), 1e-30, 1, 1, its, rel, _lib.stream_of()), "pcg")
    assert list(its) == [1] * group
    S = system.scale.cpu().numpy()[:, None]
    r32 = (S * B).astype(np.float32).astype(np.float64)
    inv32 = amg.coarse_inv.astype(np.float32).astype(np.float64)
    z, mag = inv32 @ r32, np.abs(inv32) @ np.abs(r32)
    bound = 6.0e-8 * np.abs(z) + rows * 2.3e-16 * mag
    x = X.cpu().numpy() / S
    for k in range(group):
        j = np.argsort(np.abs(z[:, k]))[rows // 2]
        alpha = x[j, k] / z[j, k]
        assert alpha > 0.0
        slack = bound[j, k] / abs(z[j, k])
        assert np.all(np.abs(x[:, k] / alpha - z[:, k]) <= 1.01 * (bound[:, k] + slack * np.abs(z[:, k])))
    amg.close()


@pytest.mark.parametrize("cells,rows", [((1, 1, 1), 81), ((16, 2, 2), 2475), ((20, 2, 2), 3075)])
def test_fp32_cycle_on_the_fp64_inverse(cells, rows):
    """An FP32 cycle told to apply the FP64 inverse: by rows up to 2 048, by
    tiles beyond.  Only its input and its result are rounded to FP32."""
    import torch
    from wnfea_amd.mesh.solid_generator import generate_c3d10_structured_block
    from wnfea_amd.solver.solid_solver import assemble_c3d10_bsr, build_amg
    print(f"FP64 coarsest product of {rows} rows in an FP32 cycle", flush=True)
    m, _ = generate_c3d10_structured_block(1.0, 0.1, 0.1, *cells, tip_load_total=-1000.0, tets_per_hex=6,
                                           load_direction="z")
    amg = build_amg(assemble_c3d10_bsr(m, want_fp64_equilibrated=True), storage=("fp64", "fp32"), autotune=False)
    inv = amg.coarse_inv
    assert len(amg.levels) == 1 and inv.shape[0] == rows
    r32 = np.random.default_rng(rows).standard_normal(rows).astype(np.float32)
    rd = torch.as_tensor(r32, device="cuda")
    plain = amg.vcycle(rd)
    amg.set_coarse_precision("fp64")
    z = amg.vcycle(rd)
    amg.set_coarse_precision("fp32")
    assert torch.equal(amg.vcycle(rd), plain) and not torch.equal(z, plain)
    ref = inv @ r32.astype(np.float64)
    mag = np.abs(inv) @ np.abs(r32.astype(np.float64))
    err = np.abs(z.double().cpu().numpy() - ref)
    assert np.all(err <= 6.0e-8 * np.abs(ref) + rows * 2.3e-16 * mag)
    amg.close()
