"""The RCS factorization's 48-column diagonal blocks at their edges, through the block solves:
widths inside and across the three 16-column parts, blocks whose pivots the rules zero
(dense_ldlt.rs:164-256: also an earlier pivot's column of L, once a pivot 1e12 times larger
follows it in its 6x6 block; sparse_ldlt.rs:399-445), against the oracle.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float(np.max(np.abs(a - b)) / np.max(np.abs(b)))


def _coupled(nb, seed):
    """Dense, symmetric indefinite, every pivot of magnitude about 12 nb (diagonally dominant):
    condition number below 10, so two correct solves differ by rounding (1e-10 leaves 1e5)."""
    rng = np.random.default_rng(seed)
    n = 6 * nb
    A = rng.normal(size=(n, n))
    A = 0.5 * (A + A.T)
    return A + np.diag(rng.choice([-1.0, 1.0], n) * 6.0 * n), rng.normal(size=n)


def _isolate(A, k, block):
    """Block k without coupling to the others."""
    s = slice(6 * k, 6 * k + 6)
    A[s, :] = A[:, s] = 0.0
    A[s, s] = block


@pytest.mark.parametrize("nb", [1, 2, 3, 4, 5, 6, 7, 8, 9, 11, 16, 17])
def test_widths(sg, orc, nb):
    A, b = _coupled(nb, nb)
    want = orc.block_ldlt_solve_dense(A, [6] * nb, b)
    assert _rel(want, np.linalg.solve(A, b)) < 1e-10
    assert _rel(sg.block_ldlt_solve(A, b), want) < 1e-10
    assert _rel(sg.sparse_ldlt_solve(A, b), want) < 1e-10


@pytest.mark.parametrize("nb,k", [(1, 0), (4, 2), (8, 0), (8, 5), (9, 7), (10, 9)])
def test_zero_block(sg, orc, nb, k):
    """A block of zeros (a free pose without terms): its pivots are dropped and it solves to 0;
    the scalar rule's solve divides by them (NaN)."""
    A, b = _coupled(nb, 50 + nb)
    _isolate(A, k, np.zeros((6, 6)))
    want = orc.block_ldlt_solve_dense(A, [6] * nb, b)
    got = sg.block_ldlt_solve(A, b)
    s = slice(6 * k, 6 * k + 6)
    assert np.all(got[s] == 0.0)
    assert np.max(np.abs(got - want)) < 1e-10 * max(1.0, np.max(np.abs(want)))
    scalar = sg.sparse_ldlt_solve(A, b)
    assert np.all(np.isnan(scalar[s]))
    rest = np.r_[0:6 * k, 6 * k + 6:6 * nb]
    if rest.size:
        assert _rel(scalar[rest], want[rest]) < 1e-10


@pytest.mark.parametrize("nb,k", [(1, 0), (8, 3), (9, 8)])
def test_pivot_dropped_behind_a_larger_one(sg, orc, nb, k):
    """Pivots 1e-5, 1e9, 1e6...: the first is kept (above 1e-12 of 1), but at 1e-14 of the
    second its column of L is zeroed for the block's later rows, which changes the solution's
    other components by O(1).  The entries of L are below 2, and eliminating the 1e9 pivot
    leaves 1e9 x 1e-16 = 1e-7 in pivots of 1e6: those components agree to about 1e-13, and
    the bar is 1e-9."""
    A, b = _coupled(nb, 80 + nb)
    rng = np.random.default_rng(90 + nb)
    L = np.tril(rng.uniform(0.5, 1.5, (6, 6)), -1) + np.eye(6)
    d = np.array([1e-5, 1e9, 1e6, 2e6, 3e6, 4e6])
    block = L @ np.diag(d) @ L.T
    _isolate(A, k, 0.5 * (block + block.T))
    want = orc.block_ldlt_solve_dense(A, [6] * nb, b)
    got = sg.block_ldlt_solve(A, b)
    s = slice(6 * k, 6 * k + 6)
    rest = np.r_[6 * k + 1:6 * k + 6]  # the first component, b / 1e-5, would hide them
    assert _rel(got[s], want[s]) < 1e-10 and _rel(got[rest], want[rest]) < 1e-9
    if nb > 1:
        assert _rel(np.delete(got, np.r_[s]), np.delete(want, np.r_[s])) < 1e-10
    # the rule matters here: a solve that keeps the column is off
    assert _rel(np.linalg.solve(A, b)[rest], want[rest]) > 0.1
