"""Node-wise beam forces where a node's elements overrun a workgroup (a hub of
300 and 513 beams), where workgroups hold one node or many, and on nodes
without elements, against the CPU oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _mesh(kind):
    rng = np.random.default_rng(7)
    if kind == "single":
        X, C = rng.standard_normal((2, 3)), np.array([[1, 0]])
    elif kind == "chain":  # one node in 70 carries no beam
        X = np.cumsum(rng.uniform(0.2, 1.0, (701, 3)), axis=0)
        C = np.array([[i, i + 1] for i in range(700) if i % 70 not in (68, 69)])
    else:  # a hub: every spoke starts or ends at node 5
        n = int(kind)
        X = rng.standard_normal((n + 6, 3))
        spokes = np.concatenate([np.arange(5), np.arange(6, n + 1)])
        C = np.array([[5, k] if k % 2 else [k, 5] for k in spokes])
    return X, C.astype(np.int32)


@pytest.mark.parametrize("accumulate", [0, 1])
@pytest.mark.parametrize("kind", ["single", "chain", "300", "513"])
def test_node_forces_match_oracle(kind, accumulate):
    import torch
    from oracle import beam_oracle as B
    from wnfea_amd import _lib
    L = _lib.load()
    X, C = _mesh(kind)
    n, M = len(X), len(C)
    rng = np.random.default_rng(3)
    props = np.column_stack([rng.uniform(5e10, 2e11, M), rng.uniform(2e10, 8e10, M)]
                            + [rng.uniform(1e-6, 1e-4, M) for _ in range(4)])
    U = 1e-2 * rng.standard_normal((n, 6))
    ptr, inc = np.zeros(n + 1, dtype=np.int32), np.zeros(2 * M, dtype=np.int32)
    _lib.check(L.wnfea_node_incidence(n, M, 2, _lib.hptr(C), _lib.hptr(ptr), _lib.hptr(inc)), "incidence")
    d = [torch.as_tensor(a, device="cuda") for a in (C, X, props, U, ptr, inc)]
    F0 = rng.standard_normal(6 * n)
    F = torch.as_tensor(F0, device="cuda") if accumulate else torch.full((6 * n,), float("nan"), dtype=torch.float64,
                                                                         device="cuda")
    fe = torch.empty((M, 12), dtype=torch.float64, device="cuda")
    _lib.check(L.wnfea_beam_forces(M, n, *[_lib.dptr(t) for t in d], _lib.dptr(fe), _lib.dptr(F), accumulate,
                                   _lib.stream_of()), "wnfea_beam_forces")
    ref = B.corot_forces(X, C, props, U.ravel()) + (F0 if accumulate else 0.0)
    # a few hundred FP64 roundings per element, at most 513 elements per node
    assert np.abs(F.cpu().numpy() - ref).max() <= 1e-12 * np.abs(ref).max()
