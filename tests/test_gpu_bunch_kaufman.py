"""Bunch–Kaufman pivoting on the GPU (indefinite mode) against the compiled reference's own indefinite factor
(MultifrontalDriver::eliminatePivoted, MultifrontalDriver.cpp:346-436) and the oracle's dense Bunch–Kaufman
(DenseBlockKernels.cpp:448-580): the same inertia, the same pivots (D per equation, 2 × 2 and delayed counts) where
the pivot tests are not within rounding of their thresholds, and solutions with a small backward error."""

import numpy as np
import pytest

import _oracle
from _problems import graph_matrix
from o_o_solver_amd import FactorOptions, FactorSolve, PivotingMode, SupernodalFactor, SymbolicFactor, SymmetricCsc, \
    models
from o_o_solver_amd.pencil import combine, pencil_scale_of, scale_symmetric

pytestmark = pytest.mark.gpu

INDEFINITE = FactorOptions(pivoting=PivotingMode.INDEFINITE)


def backward_error(a, x, b):
    r = b - a.multiply(x)
    norm = np.max(np.sum(np.abs(a.to_dense()), axis=1)) if a.n <= 3000 else None
    if norm is None:
        # ‖A‖∞ from the lower CSC: row sums of |a_ij| over both triangles.
        cols = np.repeat(np.arange(a.n), np.diff(a.offsets))
        sums = np.zeros(a.n)
        np.add.at(sums, a.rows, np.abs(a.values))
        np.add.at(sums, cols, np.where(a.rows != cols, np.abs(a.values), 0.0))
        norm = np.max(sums)
    return np.max(np.abs(r)) / (norm * np.max(np.abs(x)) + np.max(np.abs(b)))


def reference_indefinite(graph, order, matrix, b):
    """The compiled reference's indefinite factor and solve on the same structure: (inertia, counts, D by equation,
    x)."""
    h, _, _, _ = _oracle.ref_symbolic(graph[0], graph[1], graph[2], order=np.array(order, np.int32))
    try:
        x = np.array(b, order="F", copy=True)
        rc, msg, inertia, counts, _, _, diag = _oracle.ref_factor_solve(h, matrix, b=x, pivoting=1)
    finally:
        _oracle.reference().ref_sym_free(h)
    assert rc == 0, msg
    return inertia, counts, diag, x


def plate_pencil(nx, fraction, seed=3):
    """S·(K − σM)·S of a jittered plate with a lumped mass (1 on translations, 1e-4 on rotations), σ a fraction of the
    median diagonal ratio K_jj / M_jj."""
    w = models.plate(nx, jitter=0.2, seed=seed, thickness=(1e-3, 4e-3), thickness_mode="log-uniform")
    sym = w.analyse()
    k = w.matrix
    cols = np.repeat(np.arange(k.n), np.diff(k.offsets))
    diag = k.rows == cols
    mv = np.where(diag, np.where((k.rows % 6) < 3, 1.0, 1e-4), 0.0)
    mass = SymmetricCsc(k.n, k.offsets, k.rows, mv)
    dk, dm = k.values[diag], mv[diag]
    shift = fraction * np.median(dk / dm)
    return w, sym, scale_symmetric(combine(1.0, k, -shift, mass), pencil_scale_of(k))


@pytest.mark.parametrize("nx,fraction", [(12, 0.01), (12, 1.0), (30, 1e-3), (30, 1.0), (60, 0.5)])
def test_plate_pencil_pivots_match_the_reference(gpu_device, reference_lib, nx, fraction):
    w, sym, a = plate_pencil(nx, fraction)
    b = np.random.default_rng(nx).standard_normal((a.n, 3))
    inertia, counts, diag, x_ref = reference_indefinite((w.graph_offsets, w.adjacency, w.weights), sym.node_order, a,
                                                        b)
    f = SupernodalFactor.factorise(sym, a, INDEFINITE)
    got = [f.inertia.positive, f.inertia.negative, f.inertia.zero]
    print(f"plate {nx} σ-fraction {fraction}: inertia {got} (reference {inertia.tolist()}), delayed "
          f"{f.delayed_pivot_count} ({counts[0]}), 2x2 {f.two_by_two_pivot_count} ({counts[1]})", flush=True)
    assert got == inertia.tolist()
    # The same pivot sequence as the reference's (the same delayed columns and 2 × 2 pivots), so D per equation
    # agrees to rounding.
    assert (f.delayed_pivot_count, f.two_by_two_pivot_count) == (int(counts[0]), int(counts[1]))
    scale = np.maximum(np.abs(diag), 1e-300)
    assert np.max(np.abs(f.diagonal() - diag) / scale) <= 1e-8
    x = FactorSolve(f).solve(b)
    assert backward_error(a, x, b) <= 1e-12
    assert np.max(np.abs(x - x_ref)) <= 1e-6 * np.max(np.abs(x_ref))


def clique_graph(groups, links):
    """Scalar nodes in cliques (lists of nodes), plus the edges between groups listed in `links` (every node of one
    group to every node of the other)."""
    n = sum(len(g) for g in groups)
    adjacency = [set() for _ in range(n)]
    for g in groups:
        for a in g:
            adjacency[a].update(v for v in g if v != a)
    for i, j in links:
        for a in groups[i]:
            for v in groups[j]:
                adjacency[a].add(v)
                adjacency[v].add(a)
    offsets = np.cumsum([0] + [len(s) for s in adjacency]).astype(np.int64)
    nb = np.concatenate([sorted(s) for s in adjacency]).astype(np.int32)
    return offsets, nb, np.ones(n, np.int32)


@pytest.mark.parametrize("sizes,seed", [((5, 7, 6), 1), ((20, 30, 16), 2), ((70, 90, 40), 3), ((150, 130, 110), 4)])
def test_weak_children_delay_their_columns_to_the_parent(gpu_device, reference_lib, sizes, seed):
    # Two cliques A and B joined only through a separator S (order A, B, S: supernodes A and B, parent S). A's and B's
    # own couplings are tiny against their couplings to S, so their columns fail the pivot tests and are delayed
    # into S's front, where they are eliminated with S's columns.
    a_n, b_n, s_n = sizes
    groups = [list(range(a_n)), list(range(a_n, a_n + b_n)), list(range(a_n + b_n, a_n + b_n + s_n))]
    graph = clique_graph(groups, [(0, 2), (1, 2)])
    order = np.arange(a_n + b_n + s_n, dtype=np.int32)
    sym = SymbolicFactor.analyse(graph[0], graph[1], graph[2], order)
    rng = np.random.default_rng(seed)
    n = a_n + b_n + s_n
    group_of = np.repeat([0, 1, 2], sizes)
    values = {}

    def coupling(u, v):
        if (u, v) not in values:
            weak = group_of[u] == group_of[v] and group_of[u] < 2
            values[(u, v)] = rng.standard_normal() * (1e-4 if weak else 1.0)
        return values[(u, v)]

    diagonal = np.where(group_of < 2, 1e-5, 1.0) * rng.standard_normal(n)
    m = graph_matrix(sym, graph[0], graph[1], diagonal, coupling)
    b = rng.standard_normal((n, 2))
    inertia, counts, diag, x_ref = reference_indefinite(graph, order, m, b)
    f = SupernodalFactor.factorise(sym, m, INDEFINITE)
    got = [f.inertia.positive, f.inertia.negative, f.inertia.zero]
    print(f"cliques {sizes}: inertia {got} ({inertia.tolist()}), delayed {f.delayed_pivot_count} ({counts[0]}), "
          f"2x2 {f.two_by_two_pivot_count} ({counts[1]})", flush=True)
    assert got == inertia.tolist()
    assert counts[0] > 0 and f.delayed_pivot_count > 0
    assert f.delayed_pivot_count == counts[0] and f.two_by_two_pivot_count == counts[1]
    assert np.max(np.abs(f.diagonal() - diag) / np.maximum(np.abs(diag), 1e-300)) <= 1e-8
    # The parent's panel holds the delayed equations among its rows.
    root = sym.supernode_count - 1
    values_root, rows_root = f.panel(root)
    assert values_root.shape == (n - sum(f.panel(s)[0].shape[1] for s in range(root)), values_root.shape[1])
    assert len(set(rows_root.tolist())) == len(rows_root)
    x = FactorSolve(f).solve(b)
    assert backward_error(m, x, b) <= 1e-12
    assert np.max(np.abs(x - x_ref)) <= 1e-8 * np.max(np.abs(x_ref))


@pytest.mark.parametrize("n,seed", [(3, 1), (40, 2), (130, 3), (257, 4)])
def test_dense_front_matches_the_oracle_bunch_kaufman(gpu_device, n, seed):
    # A complete graph is one supernode, its front the whole matrix: the GPU's elimination by panels against the
    # oracle's column by column (the reference's order), pivot for pivot.
    graph = clique_graph([list(range(n))], [])
    sym = SymbolicFactor.analyse(graph[0], graph[1], graph[2], np.arange(n, dtype=np.int32))
    assert sym.supernode_count == 1
    rng = np.random.default_rng(seed)
    dense = rng.standard_normal((n, n))
    dense = dense + dense.T
    dense[np.arange(n), np.arange(n)] *= 1e-3  # small diagonals: 2 × 2 pivots and interchanges
    assert np.array_equal(sym.node_order, np.arange(n))
    rows = np.concatenate([np.arange(j, n) for j in range(n)]).astype(np.int32)
    offsets = np.concatenate([[0], np.cumsum(np.arange(n, 0, -1))]).astype(np.int64)
    m = SymmetricCsc(n, offsets, rows, np.concatenate([dense[j:, j] for j in range(n)]))
    f = SupernodalFactor.factorise(sym, m, INDEFINITE)
    a = np.array(np.tril(dense), order="F")
    perm = np.zeros(n, np.int64)
    sub = np.zeros(n)
    e = _oracle.oracle().orc_bunch_kaufman(_oracle.P(a), n, n, n, _oracle.P(perm), _oracle.P(sub))
    assert e == n
    values, rows = f.panel(0)
    assert rows.tolist() == perm.tolist()
    assert np.allclose(f.subdiagonal(0), sub, rtol=1e-9, atol=0)
    scale = np.max(np.abs(a))
    assert np.max(np.abs(np.tril(values, -1) - np.tril(a, -1))) <= 1e-9 * max(1.0, np.max(np.abs(np.tril(a, -1))))
    assert np.max(np.abs(np.diag(values) - np.diag(a))) <= 1e-10 * scale
    b = rng.standard_normal((n, 2))
    x = FactorSolve(f).solve(b)
    assert np.max(np.abs(dense @ x - b)) <= 1e-9 * (np.max(np.abs(dense)) * np.max(np.abs(x)) + np.max(np.abs(b)))


def dense_problem(dense):
    """One supernode whose front is the whole matrix: (symbolic factor, matrix)."""
    n = dense.shape[0]
    sym = SymbolicFactor(n, [0], [n], [-1], [0, 0], np.zeros(0, np.int32))
    rows = np.concatenate([np.arange(j, n) for j in range(n)]).astype(np.int32)
    offsets = np.concatenate([[0], np.cumsum(np.arange(n, 0, -1))]).astype(np.int64)
    return sym, SymmetricCsc(n, offsets, rows, np.concatenate([dense[j:, j] for j in range(n)]))


@pytest.mark.parametrize("n,diagonal", [(1, 1.0), (16, 1e-3), (17, 30.0), (64, 10.0), (512, 50.0), (513, 1e-3),
                                        (1025, 50.0)])
def test_panel_edges_match_the_oracle_bunch_kaufman(gpu_device, n, diagonal):
    # The steps' panels at the edges of their register layouts (16 columns; 256, 512 and 1024 rows), with diagonals
    # that make almost every pivot 2 × 2 (1e-3) or pass most tests and interchange some columns (10 to 50): the oracle's
    # pivots exactly. Values: n·eps·(growth of the pivots, up to 1e3 here) is below 1e-9.
    rng = np.random.default_rng(n)
    dense = rng.standard_normal((n, n))
    dense = dense + dense.T
    dense[np.arange(n), np.arange(n)] *= diagonal
    sym, m = dense_problem(dense)
    f = SupernodalFactor.factorise(sym, m, INDEFINITE)
    a = np.array(np.tril(dense), order="F")
    perm, sub = np.zeros(n, np.int64), np.zeros(n)
    assert _oracle.oracle().orc_bunch_kaufman(_oracle.P(a), n, n, n, _oracle.P(perm), _oracle.P(sub)) == n
    values, rows = f.panel(0)
    assert rows.tolist() == perm.tolist()
    assert np.array_equal(f.subdiagonal(0) != 0, sub != 0)
    assert np.max(np.abs(np.tril(values, -1) - np.tril(a, -1))) <= 1e-9 * max(1.0, np.max(np.abs(np.tril(a, -1))))
    assert np.max(np.abs(np.diag(values) - np.diag(a))) <= 1e-9 * np.max(np.abs(np.diag(a)))


@pytest.mark.parametrize("columns,rows", [(20, 1030), (3, 2046), (33, 4090), (5, 4100)])
def test_tall_fronts_keep_their_inertia(gpu_device, columns, rows):
    # A supernode of few columns over many rows and its parent, at the row counts where the panel takes another layout
    # (1024, 2048, 4096 rows) or the columns go through memory (more): a diagonal that dominates with random signs is
    # its own pivot order (no interchange), and its signs are the inertia.
    n = columns + rows
    sym = SymbolicFactor(n, [0, columns], [columns, rows], [1, -1], [0, rows, rows],
                         np.arange(columns, n, dtype=np.int32))
    rng = np.random.default_rng(n)
    dense = np.tril(rng.uniform(-1.0, 1.0, (n, n)), -1)
    signs = np.where(rng.random(n) < 0.3, -1.0, 1.0)
    dense[np.arange(n), np.arange(n)] = signs * n
    _, m = dense_problem(dense)
    f = SupernodalFactor.factorise(sym, m, INDEFINITE)
    assert [f.inertia.positive, f.inertia.negative, f.inertia.zero] == [int(np.sum(signs > 0)), int(np.sum(signs < 0)),
                                                                      0]
    assert f.panel(0)[1].tolist() == list(range(n)) and f.two_by_two_pivot_count == 0
    b = rng.standard_normal((n, 2))
    x = FactorSolve(f).solve(b)
    full = dense + np.tril(dense, -1).T
    assert np.max(np.abs(full @ x - b)) <= 1e-13 * (np.max(np.sum(np.abs(full), 1)) * np.max(np.abs(x)) +
                                                     np.max(np.abs(b)))


def tall_problem(columns, rows, zero):
    """A supernode of `columns` candidates over `rows` rows and its parent: candidates that interchange and pair among
    themselves, four that a weak diagonal delays, four that are pivoted alone over a larger row below and, with `zero`,
    one column of zeros; (symbolic factor, matrix, the supernode's front)."""
    n = columns + rows
    sym = SymbolicFactor(n, [0, columns], [columns, rows], [1, -1], [0, rows, rows],
                         np.arange(columns, n, dtype=np.int32))
    rng = np.random.default_rng(n)
    own = np.tril(rng.standard_normal((columns, columns)))
    own[np.arange(columns), np.arange(columns)] *= rng.choice([1e-3, 1.0, 10.0], columns)
    below = 1e-3 * rng.standard_normal((rows, columns))
    special = rng.permutation(columns)[:8]
    own[special] *= 1e-5
    own[:, special] *= 1e-5
    own[special, special] = np.where(np.arange(8) < 4, 1e-5, 0.5)
    below[:, special] = rng.standard_normal((rows, 8))
    if zero:
        at = columns // 2 if columns // 2 not in special else int(np.setdiff1d(np.arange(columns), special)[0])
        own[at] = own[:, at] = 0.0
        below[:, at] = 0.0
    diagonal = 100.0 * np.where(rng.random(rows) < 0.3, -1.0, 1.0)
    starts = np.concatenate([[0], np.cumsum(np.concatenate([np.arange(n, rows, -1), np.ones(rows, np.int64)]))])
    index = np.concatenate([np.arange(j, n) for j in range(columns)] + [np.arange(columns, n)]).astype(np.int32)
    values = np.concatenate([np.concatenate([own[j:, j], below[:, j]]) for j in range(columns)] + [diagonal])
    front = np.zeros((n, n), order="F")
    front[:columns, :columns] = own
    front[columns:, :columns] = below
    return sym, SymmetricCsc(n, starts.astype(np.int64), index, values), front


@pytest.mark.parametrize("columns,rows,zero", [(40, 2100, True), (60, 2020, False), (50, 4040, False), (45, 4200, False),
                                               (40, 4200, True)])
def test_tall_fronts_match_the_oracle_bunch_kaufman(gpu_device, columns, rows, zero):
    # Every branch of the pivot tests where a thread holds eight rows of eight columns (2,049 to 4,096 rows; from 2,048
    # rows on, four rows of sixteen) and where the columns go through memory (more): the oracle's pivots exactly.
    # Values: the growth of the multipliers (4/0.5 and 1/0.36 a column) over a few columns, times eps, is below 1e-9.
    sym, m, front = tall_problem(columns, rows, zero)
    n = columns + rows
    perm, sub = np.zeros(columns, np.int64), np.zeros(columns)
    e = _oracle.oracle().orc_bunch_kaufman(_oracle.P(front), n, n, columns, _oracle.P(perm), _oracle.P(sub))
    pivots = np.diag(front)[:e]
    assert columns - e == 4 and np.count_nonzero(sub[:e]) >= 4 and np.count_nonzero(pivots == 0.0) == int(zero)
    assert not np.array_equal(perm, np.arange(columns))
    f = SupernodalFactor.factorise(sym, m, INDEFINITE)
    values, index = f.panel(0)
    assert f.delayed_pivot_count == columns - e and values.shape == (n, e)
    assert index.tolist() == perm.tolist() + list(range(columns, n))
    assert np.allclose(f.subdiagonal(0), sub[:e], rtol=1e-9, atol=0)
    lower = np.tril(front[:, :e], -1)
    assert np.max(np.abs(np.tril(values, -1) - lower)) <= 1e-9 * max(1.0, np.max(np.abs(lower)))
    assert np.max(np.abs(np.diag(values) - pivots)) <= 1e-9 * np.max(np.abs(pivots))
    assert f.inertia.zero == int(zero)
    if not zero:
        b = np.random.default_rng(rows).standard_normal((n, 2))
        x = FactorSolve(f).solve(b)
        assert backward_error(m, x, b) <= 1e-12


@pytest.mark.parametrize("sizes,seed", [((5, 7, 6), 1), ((70, 90, 40), 3), ((300, 420, 200), 5)])
def test_delayed_columns_keep_the_inertia(gpu_device, sizes, seed):
    # Two cliques whose own couplings are tiny against those to a separator: their columns are delayed into its front
    # (passes that eliminate nothing, fronts that grow). The inertia is that of the dense eigenvalues, which lie far
    # from zero.
    groups = np.split(np.arange(sum(sizes)), np.cumsum(sizes)[:-1])
    graph = clique_graph([g.tolist() for g in groups], [(0, 2), (1, 2)])
    n = sum(sizes)
    sym = SymbolicFactor.analyse(graph[0], graph[1], graph[2], np.arange(n, dtype=np.int32))
    assert sym.node_order.tolist() == list(range(n))
    rng = np.random.default_rng(seed)
    group_of = np.repeat([0, 1, 2], sizes)
    dense = np.tril(rng.standard_normal((n, n)))
    weak = (group_of[:, None] == group_of[None, :]) & (group_of[:, None] < 2)
    dense = np.where(weak, 1e-4 * dense, dense)
    dense[np.arange(n), np.arange(n)] *= np.where(group_of < 2, 0.1, 1.0)
    dense[(group_of[:, None] + group_of[None, :]) == 1] = 0.0  # the two cliques do not touch
    offsets, rows, values = [0], [], []
    for j in range(n):
        below = [j] + [int(i) for i in graph[1][graph[0][j]:graph[0][j + 1]] if i > j]
        rows += below
        values += dense[below, j].tolist()
        offsets.append(len(rows))
    m = SymmetricCsc(n, np.array(offsets), np.array(rows, np.int32), np.array(values))
    full = m.to_dense()
    f = SupernodalFactor.factorise(sym, m, INDEFINITE)
    eigenvalues = np.linalg.eigvalsh(full)
    assert f.delayed_pivot_count > 0
    assert (f.inertia.negative, f.inertia.positive) == (int(np.sum(eigenvalues < 0)), int(np.sum(eigenvalues > 0)))
    b = rng.standard_normal((n, 2))
    x = FactorSolve(f).solve(b)
    assert backward_error(m, x, b) <= 1e-12


@pytest.mark.parametrize("nx,k", [(8, 1), (30, 5), (60, 17)])
def test_interchanges_without_delays_solve_as_the_general_structure_does(gpu_device, nx, k):
    # A plate whose supernodes interchange among their own columns but delay none (couplings to the rows below 1e-3 of
    # those within), with seven equations of their own appended: with a strong block there no column of the factor is
    # delayed, and the sweeps' lists are the plan's; with a weak one its columns are, and the lists are derived anew.
    # The plate's equations see the same operations either way: the same panels, and solutions equal to the last bit.
    w = models.plate(nx)
    sym = w.analyse()
    p = w.matrix
    n, s = p.n, sym.supernode_count
    union = SymbolicFactor(n + 7, np.concatenate([sym.first_column, [n, n + 4]]),
                           np.concatenate([sym.column_count, [4, 3]]), np.concatenate([sym.parent, [s + 1, -1]]),
                           np.concatenate([sym.row_start, np.array([3, 3]) + sym.row_start[-1]]),
                           np.concatenate([sym.rows_all, [n + 4, n + 5, n + 6]]).astype(np.int32))
    rng = np.random.default_rng(nx)
    own = np.repeat(np.arange(s), sym.column_count)
    cols = np.repeat(np.arange(n), np.diff(p.offsets))
    values = rng.standard_normal(len(p.rows)) * np.where(own[p.rows] == own[cols], 1.0, 1e-3)
    block = np.tril(rng.standard_normal((7, 7)))
    b = rng.standard_normal((n + 7, k))
    solved = []
    for weak in (False, True):
        dense = block.copy()
        dense[:4, :4] *= 1e-6 if weak else 1e3
        m = SymmetricCsc(n + 7, np.concatenate([p.offsets, p.offsets[-1] + np.cumsum(np.arange(7, 0, -1))]),
                         np.concatenate([p.rows] + [np.arange(n + j, n + 7) for j in range(7)]).astype(np.int32),
                         np.concatenate([values] + [dense[j:, j] for j in range(7)]))
        f = SupernodalFactor.factorise(union, m, INDEFINITE)
        assert (f.delayed_pivot_count > 0) == weak
        x = FactorSolve(f).solve(b)
        assert backward_error(m, x, b) <= 1e-12
        solved.append((f, x))
    strong, general = solved[0][0], solved[1][0]
    moved = 0
    for q in range(s):
        (panel, rows), (other, other_rows) = strong.panel(q), general.panel(q)
        assert rows.tolist() == other_rows.tolist() and np.array_equal(panel, other)
        moved += rows.tolist() != sorted(rows.tolist())
    assert moved > s // 4
    assert np.array_equal(solved[0][1][:n], solved[1][1][:n])
