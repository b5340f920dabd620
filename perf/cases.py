"""What the performance of the numeric LDLᵀ is measured on: factorisations and solves through the package's public
entry points, from the smallest plate, where latency and launches count, to the 1.5M-DOF plate of the benchmark.

Three kinds of case:

  statics    new stiffness values into a matrix that lies on the device, then factorise and solve to a backward error
             of `target` (one step of a design loop or of an implicit time integration: one structure, many values)
  solve      solves with a factor kept on the device (load cases that arrive one after the other)
  buckling   S·(K − σG)·S formed on the device, factorised in indefinite mode (its Sturm count) and a block solved: one
             shift of a buckling analysis

The mesh, its order and its symbolic factor are the program's fixed part and are made once per geometry. The seed gives
what changes from one analysis to the next: each node's stiffness factor (K ← diag(g)·K·diag(g), g within ±30 %), the
loads and, for buckling, the shift.
"""

import functools
import math

import numpy as np
import torch

from o_o_solver_amd import (FactorOptions, FactorSolve, Plan, Precision, SupernodalFactor, SymbolicFactor, SymmetricCsc,
                            models)
from o_o_solver_amd.pencil import ShiftedPencil

DEVICE = "cuda:0"
PRECISIONS = {"fp64": Precision.FP64, "fp32": Precision.FP32}


def _statics(name, model, nx, ny, nz=0, rhs=1, precision="fp64", target=1e-10, tuned=False):
    return {"name": name, "kind": "statics", "model": model, "nx": nx, "ny": ny, "nz": nz, "rhs": rhs,
            "precision": precision, "target": target, "tuned": tuned}


def _solve(name, model, nx, ny, nz=0, rhs=1, refined=False):
    return {"name": name, "kind": "solve", "model": model, "nx": nx, "ny": ny, "nz": nz, "rhs": rhs,
            "precision": "fp64", "target": 1e-10, "refined": refined}


def _buckling(name, circ, axial, rhs):
    return {"name": name, "kind": "buckling", "model": "cylinder", "nx": circ, "ny": axial, "nz": 0, "rhs": rhs}


def listed():
    return [
        # The smallest statics analysis the tests pin against the reference: nothing but latency and launches.
        _statics("plate24_k1", "plate", 24, 24),
        # Plain statics of one load case on the 100 × 100 plate (58,806 DOF).
        _statics("plate100_k1", "plate", 100, 100),
        # An ordinary part, odd in every size: 137 × 91 elements, five load cases.
        _statics("plate137x91_k5", "plate", 137, 91, rhs=5),
        # The benchmark: 500 × 500 elements (1,494,006 DOF), 16 load cases, on a tuned plan.
        _statics("plate500_k16", "plate", 500, 500, rhs=16, tuned=True),
        # FP32 fronts on a shell, refined by conjugate gradients to what an FP64 factor gives.
        _statics("plate300x220_fp32_k16", "plate", 300, 220, rhs=16, precision="fp32", target=1e-13),
        # A solid in FP64: few, large and dense fronts.
        _statics("hex24_k4", "hex", 24, 24, 24, rhs=4),
        # A solid of the size from which FP32 fronts are the selector's choice.
        _statics("hex40_fp32_k4", "hex", 40, 40, 40, rhs=4, precision="fp32", target=1e-12, tuned=True),
        # A design study: 32 independent plates of 20 to 80 elements a side, factorised as one matrix.
        _statics("batch32_k1", "batch", 32, 0),
        # One load case at a time against a factor kept on the device.
        _solve("solve_plate200_k1", "plate", 200, 200),
        # A block of 33 load cases (not a whole number of 16-column tiles), refined.
        _solve("solve_plate210x130_k33", "plate", 210, 130, rhs=33, refined=True),
        # Buckling shifts of a stiffened cylinder: a small one, and the benchmark's (429,840 DOF).
        _buckling("buckling48x20_k2", 48, 20, 2),
        _buckling("buckling360x200_k2", 360, 200, 2),
    ]


def _between(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["statics", "statics", "statics", "solve", "buckling"])
    if kind == "buckling":
        case = _buckling("", _between(rng, 24, 200), _between(rng, 12, 120), rng.randint(1, 6))
    else:
        model = rng.choice(["plate", "plate", "hex", "batch"])
        rhs = _between(rng, 1, 40)
        if model == "plate":
            shape = (_between(rng, 16, 400), _between(rng, 16, 400), 0)
        elif model == "hex":
            shape = (_between(rng, 6, 32), _between(rng, 6, 32), _between(rng, 6, 32))
        else:
            shape = (_between(rng, 2, 32), 0, 0)
        if kind == "statics":
            precision = rng.choice(["fp64", "fp64", "fp32"])
            case = _statics("", model, *shape, rhs=rhs, precision=precision,
                            target={"fp64": 1e-10, "fp32": 1e-12 if model == "hex" else 1e-13}[precision],
                            tuned=rng.random() < 0.3)
        else:
            case = _solve("", model, *shape, rhs=rhs, refined=rng.random() < 0.5)
    del case["name"]
    return case


@functools.lru_cache(maxsize=3)
def _geometry(model, nx, ny, nz):
    """The workload, analysed: its mesh, symbolic factor and stiffness matrix in the factor's order."""
    if model == "plate":
        w = models.plate(nx, ny, width=ny / nx, jitter=0.2, seed=20261203, thickness=(1e-3, 4e-3),
                         thickness_mode="log-uniform")
    elif model == "hex":
        w = models.hex_block(nx, ny, nz, size=(1.0, ny / nx, nz / nx), seed=20261204, sigma=1.5)
    elif model == "batch":
        w = models.plate_batch_c4(nx)
    else:
        w = models.cylinder(nx, ny, stringer_every=max(1, nx // 24))
    w.analyse()
    return w


def _workload(case):
    return _geometry(case["model"], case["nx"], case["ny"], case["nz"])


def _structure(s):
    """The symbolic factor again, without the plans made with it: each state has its own plan."""
    return SymbolicFactor(s.n, s.first_column, s.column_count, s.parent, s.row_start, s.rows_all, s.node_order,
                          s.flop_count, s.panel_value_count, s.factor_entry_count)


def _factors(w, seed):
    """Each equation's stiffness factor g (one per node)."""
    members = getattr(w, "members", [w])
    per_node = np.full(w.n // members[0].dof_per_node, members[0].dof_per_node)
    return np.repeat(np.random.default_rng(seed).uniform(0.7, 1.3, per_node.size), per_node)


def _scaled(matrix, g):
    columns = np.repeat(np.arange(matrix.n, dtype=np.int32), np.diff(matrix.offsets))
    return SymmetricCsc(matrix.n, matrix.offsets, matrix.rows, matrix.values * g[matrix.rows] * g[columns])


def _loads(case, w, seed):
    if case["kind"] == "buckling":
        return np.random.default_rng(seed + 1).standard_normal((w.n, case["rhs"]))
    return w.loads("top" if case["model"] == "hex" else "random", nrhs=case["rhs"], seed=seed + 1)


def _shift(case, seed):
    """A shift near the first buckling factors, which lie close together: from about 94 on for 120 elements round the
    cylinder and more, higher on coarser meshes."""
    return float(np.random.default_rng(seed + 2).uniform(0.9, 1.05)) * max(94.0, 1e4 / case["nx"])


def _on_device(b):
    return torch.from_numpy(np.ascontiguousarray(b.T)).to(DEVICE).T


def prepare(case, seed):
    w = _workload(case)
    g = _factors(w, seed)
    b = _on_device(_loads(case, w, seed))
    matrix = _scaled(w.matrix, g)
    symbolic = _structure(w.symbolic)
    state = {"case": case, "b": b}
    if case["kind"] == "buckling":
        geometric = w.geometric()
        load = _scaled(SymmetricCsc(geometric.n, geometric.offsets, geometric.rows, -geometric.values), g)
        state["pencil"] = ShiftedPencil(symbolic, matrix, load, transform="buckling")
        state["shift"] = _shift(case, seed)
        return state
    plan = Plan(symbolic)
    state["matrix"] = plan.matrix(matrix)
    if case["kind"] == "statics":
        state["values"] = torch.from_numpy(matrix.values).to(DEVICE)
        state["options"] = FactorOptions(precision=PRECISIONS[case["precision"]])
        if case["tuned"]:
            plan.autotune(state["matrix"], PRECISIONS[case["precision"]])
    else:
        state["factor"] = SupernodalFactor.factorise(symbolic, None, device_matrix=state["matrix"])
    return state


def run(state):
    case = state["case"]
    if case["kind"] == "buckling":
        pencil = state["pencil"]
        shifted = pencil.factorise(state["shift"])
        x = pencil.solve(shifted, state["b"])
        inertia = shifted.inertia
        return {"x": x, "inertia": [inertia.positive, inertia.negative, inertia.zero]}
    if case["kind"] == "statics":
        matrix = state["matrix"]
        matrix.set_values_device(state["values"])
        factor, x, _ = SupernodalFactor.factorise_and_solve(matrix.plan.symbolic, None, state["b"], state["options"],
                                                            device_matrix=matrix, target=case["target"], max_steps=40)
        inertia = factor.inertia
        return {"x": x, "inertia": [inertia.positive, inertia.negative, inertia.zero]}
    solve = FactorSolve(state["factor"])
    if case["refined"]:
        return solve.solve_refined(state["b"], target=case["target"])[0]
    return solve.solve(state["b"].clone())  # solved in place where the columns are contiguous


def work(case):
    """The factorisation's flops by the symbolic factor's own count and the multiplications and additions of one solve;
    the matrix and the loads read once, the factor written once and read once by the solve, the solutions written
    once."""
    w = _workload(case)
    entries, rhs = w.symbolic.factor_entry_count, case["rhs"]
    vectors = 2 * 8 * w.n * rhs
    solve = 4.0 * entries * rhs
    if case["kind"] == "solve":
        return {"bytes": 8.0 * entries + vectors, "flops": solve}
    size = 4 if case.get("precision") == "fp32" else 8
    matrices = 2 if case["kind"] == "buckling" else 1
    return {"bytes": 12.0 * w.matrix.rows.size * matrices + 2.0 * size * entries + vectors,
            "flops": w.symbolic.flop_count + solve}


def tolerance(case):
    """About four times the largest error seen over the range, against `exact` and against a correction by the
    residual: the conditioning times the rounding of 64 bits, or what the target leaves after conjugate gradients."""
    if case["kind"] == "buckling":
        rel = 1e-6
    elif case.get("precision") == "fp32":
        rel = 1e-7
    else:
        rel = 1e-11 if case["model"] == "hex" else 1e-8
    return {"rel": rel, "max": 10 * rel, "differ": 0.0}


def exact(case, seed):
    """The solutions by block elimination in 64 bits in the mesh's own numbering, where the matrix is block
    tridiagonal with blocks as wide as its bandwidth, and one correction by the residual in extended precision; the
    inertia of a positive definite matrix."""
    w = _workload(case)
    g = _factors(w, seed)
    matrix = _scaled(w.matrix, g)
    values = matrix.values
    if case["kind"] == "buckling":
        values = values + _shift(case, seed) * _scaled(w.geometric(), g).values
    members = getattr(w, "members", [w])
    dofs = members[0].dof_per_node
    natural = (w.symbolic.node_order.astype(np.int64)[:, None] * dofs + np.arange(dofs)).reshape(-1)
    columns = np.repeat(np.arange(w.n, dtype=np.int64), np.diff(matrix.offsets))
    i, j = natural[matrix.rows], natural[columns]
    i, j = np.maximum(i, j), np.minimum(i, j)
    width = int(np.max(i - j))
    blocks = -(-w.n // width)
    # About 20 seconds for the elimination and for the residual.
    if blocks * 3.0 * width ** 3 > 5e12 or 2.0 * values.size * case["rhs"] > 4e8:
        return None
    loads = np.zeros((w.n, case["rhs"]))
    loads[natural] = _loads(case, w, seed)
    solve = _block_elimination(w.n, width, i, j, values)
    x = solve(loads).astype(np.longdouble)
    x = x + solve((loads - _product(w.n, i, j, values, x)).astype(np.float64))
    x = torch.from_numpy(x.astype(np.float64)[natural])
    if case["kind"] == "solve":
        return x
    return {"x": x, "inertia": None if case["kind"] == "buckling" else [w.n, 0, 0]}


def _product(n, i, j, values, x):
    """A·x in the precision of x, A given by its lower triangle's entries."""
    off = i != j
    rows = np.concatenate([i, j[off]])
    order = np.argsort(rows, kind="stable")
    columns = np.concatenate([j, i[off]])[order]
    values = np.concatenate([values, values[off]])[order].astype(x.dtype)
    starts = np.searchsorted(rows[order], np.arange(n))
    return np.stack([np.add.reduceat(values * x[columns, h], starts) for h in range(x.shape[1])], axis=1)


def _block_elimination(n, width, i, j, values):
    """The solves with a symmetric matrix of bandwidth `width`, by block elimination (LU of each diagonal block)."""
    blocks = -(-n // width)
    order = np.argsort(j // width, kind="stable")
    i, j, values = (torch.from_numpy(a[order]).to(DEVICE) for a in (i, j, values))
    ends = torch.searchsorted(j // width, torch.arange(blocks + 1, device=DEVICE)).tolist()

    def size(q):
        return min(width, n - q * width)

    def entries(q):
        at = slice(ends[q], ends[q + 1])
        r, c, v = i[at] - q * width, j[at] - q * width, values[at]
        below = r >= width
        diagonal = torch.zeros(size(q), size(q), dtype=torch.float64, device=DEVICE)
        diagonal[r[~below], c[~below]] = v[~below]
        diagonal = torch.tril(diagonal) + torch.tril(diagonal, -1).T
        if q + 1 == blocks:
            return diagonal, None
        coupling = torch.zeros(size(q + 1), size(q), dtype=torch.float64, device=DEVICE)
        coupling[r[below] - width, c[below]] = v[below]
        return diagonal, coupling

    kept, carried = [], None
    for q in range(blocks):
        diagonal, coupling = entries(q)
        if carried is not None:
            diagonal = diagonal - carried
        lu, pivots = torch.linalg.lu_factor(diagonal)
        transfer = None
        if coupling is not None:
            transfer = torch.linalg.lu_solve(lu, pivots, coupling.T.contiguous())
            carried = coupling @ transfer
        kept.append((lu, pivots, transfer))

    def solve(rhs):
        rhs = torch.from_numpy(rhs).to(DEVICE)
        y = [rhs[q * width:q * width + size(q)] for q in range(blocks)]
        for q in range(blocks - 1):
            y[q + 1] = y[q + 1] - kept[q][2].T @ y[q]
        for q in range(blocks - 1, -1, -1):
            lu, pivots, transfer = kept[q]
            y[q] = torch.linalg.lu_solve(lu, pivots, y[q].contiguous())
            if transfer is not None:
                y[q] = y[q] - transfer @ y[q + 1]
        return torch.cat(y).cpu().numpy()

    return solve
