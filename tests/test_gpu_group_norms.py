"""Squared norms over groups of nodes against numpy: empty groups, one node,
chunk edges, interleaved owners, with and without the subtracted vector."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [[1], [0, 5, 0], [1023, 1024, 1025, 4097], [3] * 130])
@pytest.mark.parametrize("subtract", [False, True])
@pytest.mark.parametrize("dpn", [3, 6])
def test_group_norms2(sizes, subtract, dpn):
    import torch
    from wnfea_amd import _lib
    rng = np.random.default_rng(len(sizes) + dpn)
    owner = rng.permutation(np.repeat(np.arange(len(sizes)), sizes))
    n, chunk_nodes = len(owner), 1024
    a, b = rng.standard_normal((n, dpn)), rng.standard_normal((n, dpn))
    perm = np.argsort(owner, kind="stable")
    starts = np.concatenate([[0], np.cumsum(sizes)])
    nc = [-(-s // chunk_nodes) for s in sizes]
    chunk = np.concatenate([starts[g] + chunk_nodes * np.arange(nc[g]) for g in range(len(sizes))] + [starts[-1:]])
    t = lambda v: torch.as_tensor(np.ascontiguousarray(v, dtype=np.int32), device="cuda")  # noqa: E731
    d = t(np.concatenate([[0], np.cumsum(nc)])), t(chunk), t(perm)
    ad, bd = torch.as_tensor(a, device="cuda"), torch.as_tensor(b, device="cuda") if subtract else None
    part = torch.empty(max(sum(nc), 1), dtype=torch.float64, device="cuda")
    out = torch.full((len(sizes),), float("nan"), dtype=torch.float64, device="cuda")
    _lib.check(_lib.load().wnfea_group_norms2(len(sizes), sum(nc), dpn, *[_lib.dptr(v) for v in d], _lib.dptr(ad),
                                              _lib.dptr(bd), _lib.dptr(part), _lib.dptr(out), _lib.stream_of()),
               "wnfea_group_norms2")
    v = ((a - b if subtract else a) ** 2).sum(1)
    ref = np.array([v[owner == g].sum() for g in range(len(sizes))])
    # sums of at most dpn * max(sizes) positive terms: relative error <= terms * eps
    assert np.all(np.abs(out.cpu().numpy() - ref) <= dpn * max(sizes) * 2.3e-16 * ref)
