"""Panels of dense fronts at the edges of the blocked elimination's blocks and tiles, on the GPU against numpy's Cholesky
factor (L = C·diag(C)⁻¹, D = diag(C)²): a child of c columns over r rows and its parent of r columns, for c around the
16-column sub-panels and the 64-column blocks of a panel step, and where the triangle keeps its whole inverse (192
columns and more: the solves read it).

The matrices are symmetric with a dominating diagonal (condition below 4), so a backward-stable factor's entries differ
from the exact ones by a few times n·eps of their type: below 1e-12 in FP64 and 1e-4 in FP32 for n <= 1200."""

import numpy as np
import pytest

from o_o_solver_amd import FactorOptions, FactorSolve, Precision, SupernodalFactor, SymbolicFactor, SymmetricCsc

pytestmark = pytest.mark.gpu


def dense_front(c, r):
    n = c + r
    rng = np.random.default_rng(1000 * c + r)
    dense = rng.uniform(-1.0, 1.0, (n, n))
    dense = np.tril(dense) + np.tril(dense, -1).T
    dense[np.arange(n), np.arange(n)] = 2.0 * n * rng.uniform(0.8, 1.2, n)
    sym = SymbolicFactor(n, [0, c], [c, r], [1, -1], [0, r, r], np.arange(c, n, dtype=np.int32))
    rows = np.concatenate([np.arange(j, n) for j in range(n)]).astype(np.int32)
    offsets = np.concatenate([[0], np.cumsum(np.arange(n, 0, -1))]).astype(np.int64)
    return dense, sym, SymmetricCsc(n, offsets, rows, np.concatenate([dense[j:, j] for j in range(n)]))


@pytest.mark.parametrize("precision", [Precision.FP64, Precision.FP32])
@pytest.mark.parametrize("c,r", [(1, 97), (15, 100), (16, 100), (17, 100), (33, 90), (48, 130), (63, 65), (64, 64),
                                 (65, 64), (100, 1), (127, 33), (128, 128), (129, 100), (192, 40), (200, 150), (257, 130),
                                 (449, 70), (1090, 60)])
def test_panels_match_the_dense_factor(gpu_device, c, r, precision):
    dense, sym, matrix = dense_front(c, r)
    chol = np.linalg.cholesky(dense)
    d = np.diag(chol) ** 2
    lower = chol / np.diag(chol)
    factor = SupernodalFactor.factorise(sym, matrix, FactorOptions(precision=precision))
    tolerance = 1e-12 if precision == Precision.FP64 else 1e-4
    assert np.max(np.abs(factor.diagonal() - d) / d) <= tolerance
    if precision == Precision.FP64:
        for s, (first, count) in enumerate(((0, c), (c, r))):
            values, rows = factor.panel(s)
            assert rows.tolist() == list(range(first, c + r))
            expected = lower[first:, first:first + count]
            assert np.max(np.abs(np.tril(values, -1) - np.tril(expected, -1))) <= tolerance
            assert not np.any(np.triu(values, 1))
    b = np.random.default_rng(7).standard_normal((c + r, 3))
    x = FactorSolve(factor).solve(b)
    assert np.max(np.abs(x - np.linalg.solve(dense, b))) <= tolerance * np.max(np.abs(x))


@pytest.mark.parametrize("precision", [Precision.FP64, Precision.FP32])
@pytest.mark.parametrize("widths", [(1025,), (576, 1090), (1024, 512, 200), (40, 2113)])
def test_inverses_beside_the_panel_steps_give_the_same_bits(gpu_device, widths, precision):
    # Supernodes of one level over a common parent: on three streams the whole inverses of those with more than sixteen
    # blocks of 64 columns follow every sixteen blocks beside the panel steps, on one stream all levels' come last. The
    # products and their order are the same, so are the panels and (through the inverses) the solutions.
    rows = 40
    children = len(widths)
    n = sum(widths) + rows
    first = np.concatenate([[0], np.cumsum(widths)])
    sym = SymbolicFactor(n, first, list(widths) + [rows], [children] * children + [-1],
                         rows * np.minimum(np.arange(children + 2), children),
                         np.tile(np.arange(n - rows, n, dtype=np.int32), children))
    rng = np.random.default_rng(n)
    index = [np.concatenate([np.arange(j, first[s] + c), np.arange(n - rows, n)]) for s, c in enumerate(widths)
             for j in range(first[s], first[s] + c)] + [np.arange(j, n) for j in range(n - rows, n)]
    offsets = np.concatenate([[0], np.cumsum([i.size for i in index])]).astype(np.int64)
    values = rng.uniform(-1.0, 1.0, offsets[-1])
    values[offsets[:-1]] = 2.0 * n * rng.uniform(0.8, 1.2, n)
    plan = sym.plan()
    matrix = plan.matrix(SymmetricCsc(n, offsets, np.concatenate(index).astype(np.int32), values))
    options = FactorOptions(precision=precision)
    b = rng.standard_normal((n, 3))
    expected = None
    for mode in ("graph", "eager_streams", "graph_streams", "eager_streams"):
        plan.launch_mode(precision, mode)
        factor = SupernodalFactor.factorise(sym, None, options, device_matrix=matrix)
        got = [factor.panel(s)[0] for s in range(children + 1)] + [FactorSolve(factor).solve(b)]
        del factor
        expected = expected or got
        assert all(np.array_equal(x, y) for x, y in zip(got, expected)), mode
