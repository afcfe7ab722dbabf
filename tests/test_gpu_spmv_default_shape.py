"""The launch shape a matrix gets before anyone tunes it (by its blocks per
lane: rows below, at and above four) gives the products of every explicit
shape's matrix, for y given or not: each sum has another order only, n terms
of relative error eps each."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b,per_row,lanes", [(3, 3, 1), (3, 4, 1), (3, 16, 4), (3, 25, 4), (6, 7, 2), (6, 16, 4),
                                             (3, 9, 2), (3, 0, 1)])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_default_shape(b, per_row, lanes, precision):
    import torch
    from wnfea_amd.solver.bsr_matrix import DeviceBSR
    n = 150
    rng = np.random.default_rng(per_row)
    cols = np.concatenate([np.sort(rng.choice(n, per_row, replace=False)) for _ in range(n)]).astype(np.int32)
    m = DeviceBSR(b, b, n, n, np.arange(0, n * per_row + 1, max(per_row, 1), dtype=np.int32)[:n + 1] if per_row
                  else np.zeros(n + 1, np.int32), cols, 1024, lanes)
    vals = rng.standard_normal((len(cols), b, b))
    m.set_values(torch.as_tensor(vals.reshape(len(cols), b * b), device=m.device))
    dt, eps = (torch.float64, 2.3e-16) if precision == "fp64" else (torch.float32, 1.2e-7)
    x = torch.as_tensor(rng.standard_normal(n * b), device=m.device).to(dt)
    y0 = torch.full((n * b,), float("nan"), dtype=dt, device=m.device)
    y = m.spmv(x, precision=precision)
    assert torch.equal(m.spmv(x, y0, precision=precision), y)  # beta = 0 reads no y
    w = torch.ones_like(x)
    assert torch.equal(m.spmv(x, w.clone(), beta=0.5, precision=precision).isnan(), torch.zeros_like(w).bool())
    dense = np.zeros((n * b, n * b))
    for k, c in enumerate(cols):
        dense[k // per_row * b:k // per_row * b + b, c * b:c * b + b] = vals[k]
    mag = np.abs(dense) @ np.abs(x.double().cpu().numpy())
    ref = dense @ x.double().cpu().numpy()
    # products and values rounded to the precision, per_row * b terms
    tol = (per_row * b + 2) * eps * mag
    for shape in (None, (1, 1), (2, 2), (4, 1)):
        if shape:
            m.tune(shape[0], True, shape[1])
        assert np.all(np.abs(m.spmv(x, precision=precision).double().cpu().numpy() - ref) <= tol), shape
    m.close()
