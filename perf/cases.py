"""The work that users of this package have it do, as timed cases.

Each case is one call (or the few calls of one step) through the public entry
points, on the meshes of the benchmark and the tests: the C3D10 I-beam (3 mm
... 3 m of it: 300 layers are its 1 054 755 DOF), cantilever boxes of the
batch benchmark's range, and the co-rotational beam lattice.  ``prepare``
makes what a user's program holds before the call (mesh, assembled system,
hierarchy, operator, seeded loads or fields on the GPU), ``run`` is the call.

Kinds:

* ``solve``     one load case of a resident system to 1e-8 (``solve_mixed``),
  the V-cycle in FP32 (the default) or FP64, CG and the finest smoothing
  matrix-free or on the assembled matrix;
* ``multi``     several load cases of one system (``solve_multi``);
* ``batch``     many uneven boxes as one system (``BatchedSolids.solve``);
* ``adjoint``   compliance and its gradient with respect to every element's
  modulus, at the two designs of a line search (forward and backward of
  ``C3D10Adjoint.compliance``: reassembly, solve, sensitivities);
* ``newton``    one Newton correction of the beam lattice (residual, tangent,
  FP64 CG with the FP32 V-cycle);
* ``spmv``      y = K x with the 3x3 block matrix, FP64 or FP32 values;
* ``apply``     y = K x matrix-free, on straight or curved elements;
* ``stress``    the stress fields of a solution, returned to the host as the
  post-processing takes them;
* ``forces``    internal forces of a model on the device, 6 DOF per node (the
  call inside a caller's own Newton-Krylov loop);
* ``assemble``  new element moduli assembled into a resident system.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from wnfea_amd.mesh.lattice import beam_props, generate_beam_lattice
from wnfea_amd.mesh.rcm import apply_rcm_to_model
from wnfea_amd.mesh.solid_generator import (generate_c3d10_ibeam, generate_c3d10_structured_block,
                                            ibeam_tip_load_cases)
from wnfea_amd.solver.adjoint import C3D10Adjoint
from wnfea_amd.solver.batch import BatchedSolids, generate_box_batch
from wnfea_amd.solver.beam_solver import BeamSystem
from wnfea_amd.solver.residual import compute_internal_forces
from wnfea_amd.solver.solid_solver import (MatrixFreeOperator, assemble_c3d10_bsr, build_amg,
                                           compute_c3d10_stress_field, mesh_to_device, pcg_device,
                                           reassemble_c3d10_values, solve_mixed, solve_multi)

TOL = 1e-8
DEV = "cuda"
#: the I-beam's strength thresholds in the benchmark; boxes take the library's defaults
IBEAM_AMG = {"theta": 0.1, "theta_decay": 0.5}


def listed():
    return [
        # the small box of the benchmark and the smoke run: launches and latency count
        {"name": "solve-box-40x4x4", "kind": "solve", "mesh": "box", "nx": 40, "nyz": 4, "precision": "fp32",
         "operator": "matrix_free"},
        # the headline workload: 1 054 755 DOF to 1e-8
        {"name": "solve-ibeam-300", "kind": "solve", "mesh": "ibeam", "layers": 300, "precision": "fp32",
         "operator": "matrix_free"},
        # an ordinary model solved all in FP64 on the assembled matrix, as the drop-in entry points do
        {"name": "solve-fp64-ibeam-41", "kind": "solve", "mesh": "ibeam", "layers": 41, "precision": "fp64",
         "operator": "assembled"},
        # a set of load cases that does not fill its last group
        {"name": "multi-ibeam-60x12", "kind": "multi", "layers": 60, "columns": 12},
        # uneven boxes in one system
        {"name": "batch-24-boxes", "kind": "batch", "boxes": 24, "mesh_seed": 1},
        # design optimisation: value and gradient at two designs
        {"name": "adjoint-ibeam-20", "kind": "adjoint", "layers": 20},
        # the inner step of the geometrically nonlinear frame solver
        {"name": "newton-lattice-32", "kind": "newton", "cells": 32},
        # the benchmark's SpMV figure
        {"name": "spmv-fp32-ibeam-300", "kind": "spmv", "layers": 300, "precision": "fp32"},
        # a mesh with curved elements, as second-order mesh files hold
        {"name": "apply-curved-ibeam-75", "kind": "apply", "layers": 75, "curved": True},
        # post-processing of a solution
        {"name": "stress-ibeam-100", "kind": "stress", "layers": 100},
        # the smallest call: a small frame's forces inside a caller's Krylov loop
        {"name": "forces-lattice-12", "kind": "forces", "mesh": "lattice", "cells": 12},
        # new moduli of a design step
        {"name": "assemble-ibeam-100", "kind": "assemble", "layers": 100},
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["solve", "solve", "multi", "batch", "adjoint", "newton", "spmv", "apply", "stress", "forces",
                       "assemble"])
    if kind == "solve":
        c = {"kind": kind, "precision": rng.choice(["fp32", "fp32", "fp64"]),
             "operator": rng.choice(["matrix_free", "matrix_free", "assembled"])}
        if rng.random() < 0.5:
            return {**c, "mesh": "box", "nx": rng.randint(10, 60), "nyz": rng.randint(3, 8)}
        return {**c, "mesh": "ibeam", "layers": size(5, 150)}
    if kind == "multi":
        return {"kind": kind, "layers": size(5, 60), "columns": size(2, 20)}
    if kind == "batch":
        return {"kind": kind, "boxes": rng.randint(6, 28), "mesh_seed": rng.randint(2, 9999)}
    if kind == "adjoint":
        return {"kind": kind, "layers": size(5, 40)}
    if kind == "newton":
        return {"kind": kind, "cells": rng.randint(7, 32)}
    if kind == "spmv":
        return {"kind": kind, "layers": size(4, 250), "precision": rng.choice(["fp64", "fp32"])}
    if kind == "apply":
        return {"kind": kind, "layers": size(4, 150), "curved": rng.random() < 0.5}
    if kind == "stress":
        return {"kind": kind, "layers": size(4, 150)}
    if kind == "forces":
        if rng.random() < 0.5:
            return {"kind": kind, "mesh": "lattice", "cells": rng.randint(4, 40)}
        return {"kind": kind, "mesh": "ibeam", "layers": size(4, 100)}
    return {"kind": kind, "layers": size(4, 100)}


# ------------------------------------------------------------------ inputs
def _rng(case, seed):
    return np.random.default_rng([int(seed), sum(map(ord, case["kind"]))])


def _solid(case):
    """(RCM-ordered model, tip nodes, amg keywords) of a solid case."""
    if case.get("mesh", "ibeam") == "ibeam":
        n = case["layers"]
        model, meta = generate_c3d10_ibeam(n_layers=n, length=3.0 * n / 300)
        model, _, o2n = apply_rcm_to_model(model)
        return model, o2n[meta["tip_nodes"]], dict(IBEAM_AMG)
    nx, k = case["nx"], case["nyz"]
    model, meta = generate_c3d10_structured_block(nx / 40.0, k / 40.0, k / 40.0, nx, k, k, tip_load_total=-1000.0,
                                                  tets_per_hex=6, load_direction="z")
    tip = np.array([ld.node_id for ld in model.loads])
    model, _, o2n = apply_rcm_to_model(model)
    return model, o2n[tip], {}


def _tip_loads(case, model, tip, columns, seed):
    """Seeded forces and moments on the tip, (n_dofs, columns) on the host."""
    if case.get("mesh", "ibeam") == "ibeam":
        B = ibeam_tip_load_cases(model.mesh_nodes, tip, n_cases=columns, seed=int(seed))
    else:
        f = _rng(case, seed).normal(0.0, 1000.0, (3, columns)) / len(tip)
        B = np.zeros((3 * len(model.mesh_nodes), columns))
        for c in range(3):
            B[3 * tip + c] = f[c]
    B[model.fixed_dof_mask(3)] = 0.0
    return B


def _curve(model, amplitude=0.08):
    """The model with its midside nodes moved off the edge midpoints by a smooth
    field of `amplitude` cell sizes (a function of the node alone, so shared
    nodes move together and every element keeps a positive volume)."""
    X, T = model.mesh_nodes.copy(), model.solid_elements
    mid = np.unique(T[:, 4:])
    h = 0.01
    p = X[mid]
    X[mid] += amplitude * 0.006 * np.column_stack([np.sin(p[:, 1] / h), np.sin(p[:, 2] / h), np.sin(p[:, 0] / h)])
    model.mesh_nodes = X
    return model


def _displacement(model, seed, case):
    """A bent, twisted and locally perturbed displacement field, (n, 3)."""
    r = _rng(case, seed)
    X = model.mesh_nodes
    L = max(float(X[:, 0].max()), 1e-9)
    a = r.normal(0.0, 1e-3, 4)
    s = X[:, 0] / L
    u = np.column_stack([1e-2 * a[0] * X[:, 2] * s, a[1] * s**2 + a[3] * s * X[:, 2], a[2] * s**2 - a[3] * s * X[:, 1]])
    u += 1e-6 * r.normal(size=u.shape)
    u[model.fixed_dof_mask(3).reshape(-1, 3)] = 0.0
    return u


def _lattice_field(model, seed, case):
    """Translations and rotations of a swaying, compressed frame, (n, 6)."""
    r = _rng(case, seed)
    X = model.mesh_nodes
    H = max(float(X[:, 2].max()), 1.0)
    a = r.normal(0.0, 1.0, 3)
    s = X[:, 2] / H
    U = np.zeros((len(X), 6))
    U[:, 0], U[:, 1], U[:, 2] = 0.02 * a[0] * s**2, 0.02 * a[1] * s**2, -0.002 * (1 + abs(a[2])) * s
    U[:, 3], U[:, 4] = -0.04 * a[1] * s / H, 0.04 * a[0] * s / H
    U += 1e-5 * r.normal(size=U.shape)
    U[model.fixed_dof_mask(6).reshape(-1, 6)] = 0.0
    return U.reshape(-1)


def _moduli(case, seed, M):
    return 210e9 * (0.2 + 0.8 * _rng(case, seed).uniform(size=M))


def _tensor(a):
    return torch.as_tensor(np.ascontiguousarray(a), device=DEV)


# ------------------------------------------------------------------ prepare
def prepare(case, seed):
    kind = case["kind"]
    if kind in ("newton", "forces") and case.get("mesh", "lattice") == "lattice":
        model, _ = generate_beam_lattice(case["cells"], seed=int(seed) % 100003)
        model, _, _ = apply_rcm_to_model(model)
        U = _tensor(_lattice_field(model, seed, case))
        if kind == "forces":
            return {"kind": kind, "model": model, "U": U}
        frame = BeamSystem(model)
        frame.assemble_tangent(torch.zeros_like(U))
        frame.build_amg()
        return {"kind": kind, "frame": frame, "U": U}
    if kind == "batch":
        r = _rng(case, seed)
        models = [m for m, _ in generate_box_batch(case["boxes"], seed=case["mesh_seed"])]
        for m in models:
            f = r.normal(0.0, 1000.0, 3) / len(m.loads)
            for ld in m.loads:
                ld.fx, ld.fy, ld.fz = (float(v) for v in f)
        return {"kind": kind, "boxes": BatchedSolids(models)}
    model, tip, amg_kw = _solid(case)
    M = len(model.solid_elements)
    if kind == "forces":
        U = np.zeros((len(model.mesh_nodes), 6))
        U[:, :3] = _displacement(model, seed, case)
        return {"kind": kind, "model": model, "U": _tensor(U.reshape(-1))}
    if kind == "stress":
        return {"kind": kind, "model": model, "mesh": mesh_to_device(model),
                "U": _tensor(_displacement(model, seed, case).reshape(-1))}
    if kind == "adjoint":
        E = _moduli(case, seed, M)
        model.solid_E, model.solid_nu = E, np.full(M, 0.3)
        B = _tip_loads(case, model, tip, 1, seed)[:, 0].reshape(-1, 3)
        for ld in model.loads:
            ld.fx, ld.fy, ld.fz = (float(v) for v in B[ld.node_id])
        problem = C3D10Adjoint(model)
        problem.set_moduli(E)
        step = _rng(case, seed + 1).uniform(-0.01, 0.01, (2, M))
        return {"kind": kind, "problem": problem, "designs": [_tensor(E * (1 + d)) for d in step]}
    if kind == "apply" and case["curved"]:
        model = _curve(model)
    system = assemble_c3d10_bsr(model, want_fp64_equilibrated=case.get("precision") == "fp64" and kind == "solve",
                                keep_plan=kind == "assemble")
    state = {"kind": kind, "system": system}
    if kind == "assemble":
        state["E"] = _tensor(_moduli(case, seed, M))
    elif kind == "spmv":
        state["precision"] = case["precision"]
        x = _displacement(model, seed, case).reshape(-1)
        if case["precision"] == "fp32":  # the FP32 values are those of the equilibrated matrix
            x = (_tensor(x) / system.scale).float()
        state["x"] = x if isinstance(x, torch.Tensor) else _tensor(x)
    elif kind == "apply":
        state["operator"] = MatrixFreeOperator(system)
        state["x"] = _tensor(_displacement(model, seed, case).reshape(-1))
    else:
        B = _tensor(_tip_loads(case, model, tip, case.get("columns", 1), seed))
        if kind == "multi":
            state["B"] = B
        else:
            system.F = B[:, 0].contiguous()
        state["precision"] = case.get("precision", "fp32")
        state["amg"] = build_amg(system, storage=(state["precision"],), **amg_kw)
        state["operator"] = None
        if case.get("operator") == "matrix_free":
            state["operator"] = MatrixFreeOperator(system)
            state["operator"].attach_smoother(state["amg"])
    return state


# ------------------------------------------------------------------ run
def run(state):
    kind = state["kind"]
    if kind == "solve":
        return solve_mixed(state["system"], state["amg"], tol=TOL, amg_precision=state["precision"],
                           operator=state["operator"])[0]
    if kind == "multi":
        return solve_multi(state["system"], state["amg"], state["B"], tol=TOL)[0]
    if kind == "batch":
        return state["boxes"].solve(TOL)[0]
    if kind == "adjoint":
        out = []
        for E in state["designs"]:
            E = E.detach().requires_grad_()
            C = state["problem"].compliance(E)
            C.backward()
            out += [C.detach(), E.grad]
        return out
    if kind == "newton":
        frame, U = state["frame"], state["U"]
        R = frame.residual(U, 0.5)
        frame.assemble_tangent(U)
        dU = pcg_device(frame.system, b=-R, rtol=TOL, max_iter=500, preconditioner="amg", precision="fp64",
                        amg=frame.amg, amg_precision="fp32")[0]
        return {"R": R, "dU": dU}
    if kind == "spmv":
        return state["system"].K.spmv(state["x"], precision=state["precision"])
    if kind == "apply":
        return state["operator"].apply(state["x"])
    if kind == "stress":
        return list(compute_c3d10_stress_field(state["model"], state["U"], mesh=state["mesh"]))
    if kind == "forces":
        return compute_internal_forces(state["model"], state["U"])
    s = reassemble_c3d10_values(state["system"], E=state["E"])
    return {"K": s.K.get_values(), "diag": s.diag, "scale": s.scale}


# ------------------------------------------------------------------ work
def _counts(case):
    """(nodes, elements, 3x3 blocks) of a solid case; the blocks to a few per cent."""
    if case["kind"] == "batch":
        r = np.random.default_rng(case["mesh_seed"])
        n = m = got = 0
        while got < case["boxes"]:
            nx, ny = int(r.integers(10, 61)), int(r.integers(3, 9))
            k = (2 * nx + 1) * (2 * ny + 1) ** 2
            if 2000 <= 3 * k <= 60000:
                n, m, got = n + k, m + 6 * nx * ny * ny, got + 1
    elif case.get("mesh", "ibeam") == "ibeam":
        n, m = 1170 * case["layers"] + 585, 696 * case["layers"]
    else:
        n = (2 * case["nx"] + 1) * (2 * case["nyz"] + 1) ** 2
        m = 6 * case["nx"] * case["nyz"] ** 2
    return n, m, int(25.1 * n)


#: CG iterations that a smoothed-aggregation cycle needs here (22 to 48 over the cases)
_ITERATIONS = 30


def work(case):
    """Bytes and operations of one pass.  Solves: per iteration, the operator in
    its smallest form (connectivity and geometry of each element, or blocks
    for a frame) once in FP64 for CG and four times in the cycle's precision
    (its smoothing steps and defect), and the vectors those read and write."""
    kind = case["kind"]
    if kind in ("newton", "forces") and case.get("mesh", "lattice") == "lattice":
        c = case["cells"]
        n, beams = (c + 1) ** 3, 3 * c * (c + 1) ** 2
        force = {"bytes": 56 * beams + n * (24 + 2 * 48), "flops": 600 * beams}
        if kind == "forces":
            return force
        blocks = n + 2 * beams
        it = 2 * _ITERATIONS
        return {"bytes": force["bytes"] + 288 * blocks + it * (blocks * (292 + 4 * 148) + n * 6 * (7 * 8 + 20 * 4)),
                "flops": force["flops"] + 16000 * beams + it * 72 * 5 * blocks}
    n, m, nnzb = _counts(case)
    if kind == "spmv":
        s = 4 if case["precision"] == "fp32" else 8
        return {"bytes": nnzb * (9 * s + 4) + 6 * n * s, "flops": 18 * nnzb}
    if kind == "apply":
        return {"bytes": m * (40 + 16 + (320 if case["curved"] else 80)) + 48 * n, "flops": 2160 * m}
    if kind == "stress":
        return {"bytes": m * (40 + 16 + 56) + n * (24 + 24 + 8), "flops": 1800 * m}
    if kind == "forces":
        return {"bytes": m * 56 + n * (24 + 96), "flops": 4000 * m}
    if kind == "assemble":
        return {"bytes": m * 56 + 24 * n + nnzb * (72 + 36 + 72 + 4), "flops": 12000 * m}
    s = 8 if case.get("precision") == "fp64" else 4
    columns = case.get("columns", 1)
    element = m * (20 + 80 + 16)
    cycle = 4 * (m * (20 + 12 * s) + columns * 3 * n * 7 * s)
    per = element + columns * 3 * n * 7 * 8 + cycle
    flops = columns * 5 * 700 * m
    groups = -(-columns // 8)
    solves = {"adjoint": 2}.get(kind, 1)
    total = {"bytes": _ITERATIONS * (per + (groups - 1) * (element + cycle // 8)), "flops": _ITERATIONS * flops}
    if kind == "adjoint":
        total["bytes"] += m * 56 + 24 * n + nnzb * 108
        total["flops"] += 12000 * m
    return {k: solves * v for k, v in total.items()}


# ------------------------------------------------------------------ exact
def _gauss():
    a, b = (5 - 5 ** 0.5) / 20, (5 + 3 * 5 ** 0.5) / 20
    out = np.zeros((4, 3, 10))
    for g, (x, y, z) in enumerate([(a, a, a), (b, a, a), (a, b, a), (a, a, b)]):
        L = (1 - x - y - z, x, y, z)
        dL = np.zeros((4, 10))
        for k in range(4):
            dL[k, k] = 4 * L[k] - 1
        for e, (p, q) in enumerate([(0, 1), (1, 2), (2, 0), (0, 3), (1, 3), (2, 3)]):
            dL[p, 4 + e], dL[q, 4 + e] = 4 * L[q], 4 * L[p]
        out[g] = dL[1:] - dL[0]
    return torch.as_tensor(out, device=DEV)


class _Plain:
    """The C3D10 mesh in plain torch: shape gradients, weights and moduli."""

    def __init__(self, model, E=None):
        self.T = torch.as_tensor(np.asarray(model.solid_elements, dtype=np.int64), device=DEV)
        self.X = _tensor(np.asarray(model.mesh_nodes, dtype=np.float64))
        Em, nu = model.element_moduli()
        E = _tensor(Em) if E is None else E
        nu = _tensor(nu)
        self.lam, self.mu = E * nu / ((1 + nu) * (1 - 2 * nu)), E / (2 * (1 + nu))
        self.fixed = torch.as_tensor(model.fixed_dof_mask(3), device=DEV)
        J = torch.einsum("gki,mic->mgkc", _gauss(), self.X[self.T])
        self.w = torch.linalg.det(J) / 24
        self.g = torch.einsum("mgck,gki->mgci", torch.linalg.inv(J), _gauss())

    def stress(self, u):
        """(elements, 4, 3, 3) Gauss-point stresses of u (n, 3)."""
        H = torch.einsum("mai,mgja->mgij", u[self.T], self.g)
        tr = torch.diagonal(H, dim1=2, dim2=3).sum(-1)
        eye = torch.eye(3, dtype=H.dtype, device=DEV)
        return (self.mu[:, None, None, None] * (H + H.transpose(2, 3))
                + (self.lam[:, None] * tr)[..., None, None] * eye)

    def apply(self, u, bcs=True):
        v = u.clone()
        if bcs:
            v[self.fixed] = 0
        S = self.stress(v.view(-1, 3)) * self.w[..., None, None]
        f = torch.einsum("mgij,mgja->mai", S, self.g).reshape(-1, 3)
        y = torch.zeros_like(u).view(-1, 3).index_add_(0, self.T.reshape(-1), f).view(-1)
        if bcs:
            y[self.fixed] = u[self.fixed]
        return y

    def blocks(self):
        """(3x3 block values, rows, columns) in row-major block order, supports applied."""
        n = len(self.X)
        gg = torch.einsum("mgia,mgjb,mg->mabij", self.g, self.g, self.w)
        Ke = (self.lam[:, None, None, None, None] * gg + self.mu[:, None, None, None, None] * gg.transpose(3, 4))
        tr = self.mu[:, None, None] * torch.diagonal(gg, dim1=3, dim2=4).sum(-1)
        for c in range(3):
            Ke[..., c, c] += tr
        del gg, tr
        a, b = self.T[:, :, None].expand(-1, -1, 10).reshape(-1), self.T[:, None, :].expand(-1, 10, -1).reshape(-1)
        clamped = self.fixed.view(-1, 3).all(1)
        keep = ~((clamped[a] | clamped[b]) & (a != b))
        keys, at = torch.unique((a * n + b)[keep], return_inverse=True)
        V = torch.zeros((len(keys), 3, 3), dtype=torch.float64, device=DEV)
        V.index_add_(0, at, Ke.reshape(-1, 3, 3)[keep])
        r, c = keys // n, keys % n
        f = self.fixed.view(-1, 3)
        V[f[r][:, :, None] | f[c][:, None, :]] = 0
        k = torch.arange(3, device=DEV)
        on = (r == c)[:, None, None] & (k[:, None] == k[None, :]) & f[r][:, :, None]
        V[on.expand_as(V)] = 1
        return V, r, c

    def dense(self):
        V, r, c = self.blocks()
        n = len(self.X)
        A = torch.zeros((n, 3, n, 3), dtype=torch.float64, device=DEV)
        A[r, :, c, :] = V
        return A.view(3 * n, 3 * n)


def _dense_solve(A, B):
    L = torch.linalg.cholesky(A)
    x = torch.cholesky_solve(B, L)
    for _ in range(2):
        x = x + torch.cholesky_solve(B - A @ x, L)
    return x


def _frame_forces(model, U):
    """Co-rotational beam forces of U (n, 6), plain torch."""
    C = torch.as_tensor(np.asarray(model.mesh_elements, dtype=np.int64), device=DEV)
    X = _tensor(np.asarray(model.mesh_nodes, dtype=np.float64))
    E, G, A, Iy, Iz, J = _tensor(beam_props(model)).T
    dot = lambda a, b: (a * b).sum(1, keepdim=True)  # noqa: E731
    unit = lambda a: a / a.norm(dim=1, keepdim=True)  # noqa: E731
    cross = lambda a, b: torch.linalg.cross(a, b, dim=1)  # noqa: E731
    v0 = X[C[:, 1]] - X[C[:, 0]]
    L0 = v0.norm(dim=1, keepdim=True)
    e1 = v0 / L0
    up = torch.zeros_like(e1)
    up[:, 2] = (e1[:, 2].abs() < 0.9).double()
    up[:, 1] = 1 - up[:, 2]
    e2 = unit(cross(up, e1))
    u = U.view(-1, 6)
    du, t1, t2 = u[C[:, 1], :3] - u[C[:, 0], :3], u[C[:, 0], 3:], u[C[:, 1], 3:]
    v = v0 + du
    L = v.norm(dim=1, keepdim=True)
    r1 = v / L
    cr, cphi = cross(e1, r1), dot(e1, r1)
    r2 = cphi * e2 + cross(cr, e2) + dot(cr, e2) / (1 + cphi) * cr
    tw = 0.5 * dot(t1 + t2, r1)
    r2 = torch.cos(tw) * r2 + torch.sin(tw) * cross(r1, r2)
    r2 = unit(r2 - dot(r2, r1) * r1)
    r3 = unit(cross(r1, r2))
    ul = (2 * dot(v0, du) + dot(du, du)) / (L + L0)
    y1, z1 = dot(r2, t1) + dot(r3, du) / L, dot(r3, t1) - dot(r2, du) / L
    y2, z2 = dot(r2, t2) + dot(r3, du) / L, dot(r3, t2) - dot(r2, du) / L
    k = lambda a: (a / L0[:, 0])[:, None]  # noqa: E731
    N, T = k(E * A) * ul, k(G * J) * dot(r1, t2 - t1)
    My1, My2 = k(E * Iy) * (4 * y1 + 2 * y2), k(E * Iy) * (2 * y1 + 4 * y2)
    Mz1, Mz2 = k(E * Iz) * (4 * z1 + 2 * z2), k(E * Iz) * (2 * z1 + 4 * z2)
    f1 = -N * r1 - (My1 + My2) / L * r3 + (Mz1 + Mz2) / L * r2
    m1, m2 = -T * r1 + My1 * r2 + Mz1 * r3, T * r1 + My2 * r2 + Mz2 * r3
    F = torch.zeros_like(u)
    F.index_add_(0, C[:, 0], torch.cat([f1, m1], 1))
    F.index_add_(0, C[:, 1], torch.cat([-f1, m2], 1))
    return F.view(-1)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("newton", "forces") and case.get("mesh", "lattice") == "lattice":
        model, _ = generate_beam_lattice(case["cells"], seed=int(seed) % 100003)
        model, _, _ = apply_rcm_to_model(model)
        U = _tensor(_lattice_field(model, seed, case))
        F = _frame_forces(model, U)
        if kind == "forces":
            return F
        fixed = torch.as_tensor(model.fixed_dof_mask(6), device=DEV)
        R = F - 0.5 * _tensor(model.load_vector(6))
        R[fixed] = U[fixed]
        return {"R": R, "dU": None}
    if kind in ("batch", "adjoint"):
        return None
    if kind in ("solve", "multi") and 3 * _counts(case)[0] > 25000:
        return None  # a dense factorisation would be too large
    model, tip, _ = _solid(case)
    if kind in ("solve", "multi"):
        x = _dense_solve(_Plain(model).dense(), _tensor(_tip_loads(case, model, tip, case.get("columns", 1), seed)))
        return x if kind == "multi" else x[:, 0]
    if kind == "assemble":
        V, r, c = _Plain(model, E=_tensor(_moduli(case, seed, len(model.solid_elements)))).blocks()
        diag = torch.diagonal(V[r == c], dim1=1, dim2=2).reshape(-1)
        return {"K": V.reshape(-1, 9), "diag": diag, "scale": 1 / torch.sqrt(diag.abs())}
    if kind == "apply" and case["curved"]:
        model = _curve(model)
    u = _displacement(model, seed, case)
    P = _Plain(model)
    if kind == "spmv":
        x = _tensor(u.reshape(-1))
        if case["precision"] == "fp64":
            return P.apply(x)
        V, r, c = P.blocks()
        S = 1 / torch.sqrt(torch.diagonal(V[r == c], dim1=1, dim2=2).reshape(-1).abs())
        del V
        return S * P.apply(S * (x / S).float().double())
    if kind == "apply":
        return P.apply(_tensor(u.reshape(-1)))
    if kind == "forces":
        F = torch.zeros((len(u), 6), dtype=torch.float64, device=DEV)
        F[:, :3] = P.apply(_tensor(u.reshape(-1)), bcs=False).view(-1, 3)
        return F.view(-1)
    s = P.stress(_tensor(u))
    six = torch.stack([s[..., 0, 0], s[..., 1, 1], s[..., 2, 2], s[..., 0, 1], s[..., 1, 2], s[..., 0, 2]], -1)
    vm = torch.sqrt(0.5 * ((six[..., 0] - six[..., 1]) ** 2 + (six[..., 1] - six[..., 2]) ** 2
                           + (six[..., 2] - six[..., 0]) ** 2 + 6 * (six[..., 3:] ** 2).sum(-1))).mean(1)
    total, count = torch.zeros(len(u), dtype=torch.float64, device=DEV), torch.zeros(len(u), device=DEV)
    at = P.T.reshape(-1)
    total.index_add_(0, at, vm[:, None].expand(-1, 10).reshape(-1))
    count.index_add_(0, at, torch.ones(len(at), device=DEV))
    return [six.mean(1), vm, total / count.clamp(min=1)]
