"""The multi-column product at the edges of its lane split: one row, rows
without blocks, rows longer and shorter than the lanes per row, every layout
width, both column counts and value precisions, against scipy."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nrhs", [4, 8])
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("br,bc,n_rows,n_cols,lanes", [
    (3, 3, 1, 1, 1), (3, 3, 65, 65, 1), (3, 3, 203, 203, 4), (3, 3, 67, 90, 16), (3, 3, 9, 300, 64),
    (6, 6, 37, 37, 0), (6, 6, 130, 130, 8), (3, 6, 101, 17, 2), (6, 3, 17, 101, 32)])
def test_spmm_edges(br, bc, n_rows, n_cols, lanes, prec, nrhs):
    import torch
    from wnfea_amd import _lib
    from wnfea_amd.solver.bsr_matrix import DeviceBSR
    rng = np.random.default_rng([br, bc, n_rows, lanes, nrhs])
    # block counts per row from none to all columns, uneven inside a slice
    count = np.minimum(rng.integers(0, 40, n_rows), n_cols)
    count[0] = min(n_cols, 33)
    cols = [np.sort(rng.choice(n_cols, c, replace=False)) for c in count]
    rowptr = np.concatenate([[0], np.cumsum(count)]).astype(np.int32)
    colidx = np.concatenate(cols).astype(np.int32)
    vals = rng.standard_normal((len(colidx), br * bc))
    X = rng.standard_normal((n_cols * bc, nrhs))
    if prec == "fp32":
        vals, X = vals.astype(np.float32).astype(np.float64), X.astype(np.float32).astype(np.float64)
    A = DeviceBSR(br, bc, n_rows, n_cols, rowptr, colidx, lanes=lanes)
    A.set_values(torch.as_tensor(vals, device="cuda"), 3)
    dt = torch.float32 if prec == "fp32" else torch.float64
    Xd = torch.as_tensor(X, device="cuda").to(dt)
    Y = torch.full((n_rows * br, nrhs), float("nan"), dtype=dt, device="cuda")
    L = _lib.load()
    _lib.check(L.wnfea_bsr_spmm(A.handle, int(prec == "fp32"), nrhs, _lib.dptr(Xd), _lib.dptr(Y), _lib.stream_of()),
               "wnfea_bsr_spmm")
    S = sp.bsr_matrix((vals.reshape(-1, br, bc), colidx, rowptr), shape=(n_rows * br, n_cols * bc))
    # each output is a sum of k = bc blocks products: |error| <= k eps |A| |x|
    eps = np.finfo(np.float32 if prec == "fp32" else np.float64).eps
    k = bc * max(int(count.max()), 1)
    bound = k * eps * (abs(S) @ np.abs(X))
    assert np.all(np.abs(Y.double().cpu().numpy() - S @ X) <= bound)
    A.close()
