"""The register LU panel at the edges of its workgroups (256 and 512 rows)
and column segments (16), m x w panels with every tie and non-finite rule,
against the oracle's getf2: pivots equal, factors within rounding."""
import numpy as np
import pytest

import atlas_amd as X
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("m,n", [(1, 1), (15, 15), (17, 16), (63, 33), (64, 64), (65, 47), (255, 64),
                                 (256, 64), (257, 64), (511, 31), (512, 64), (513, 64), (700, 130),
                                 (1025, 48), (4097, 64)])
def test_panel_shapes_vs_oracle(dt, m, n):
    rng = np.random.default_rng(m * 131 + n)
    # distinct magnitudes: no near ties, so the pivots are decided exactly
    A = np.asfortranarray(rng.uniform(-1, 1, (m, n)).astype(dt))
    L, Q = A.copy(order="F"), A.astype(np.float64).copy(order="F")
    info, piv = X.getrf(L)
    oinfo, opiv = O.getrf(Q)
    assert info == oinfo == 0
    if dt == np.float64:
        assert np.array_equal(piv, opiv)
    P = A.astype(np.float64).copy()
    for k, p in enumerate(piv):
        P[[k, p]] = P[[p, k]]
    k = min(m, n)
    Lf, Uf = np.tril(L[:, :k].astype(np.float64), -1) + np.eye(m, k), np.triu(L[:k].astype(np.float64))
    u = np.finfo(dt).eps
    # |P A - L U| <= gamma_k |L| |U| (Higham, Accuracy and Stability, Theorem 9.3)
    assert np.all(np.abs(P - Lf @ Uf) <= (k + 2) * u * (np.abs(Lf) @ np.abs(Uf)) + 1e-300)
    assert np.abs(Lf).max() <= 1.0


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("m", [40, 300, 600])
def test_panel_ties_take_the_lowest_row(dt, m):
    """all entries of the first column equal in magnitude: row 0, no swap;
    a tie between rows of different wavefronts and workgroups: the lower"""
    A = np.asfortranarray(np.ones((m, 3), dt))
    A[1::2, 0] = -1
    A[:, 1] = 0.25
    lo, hi = m // 3, m - 1
    A[lo, 1] = A[0, 1] * A[lo, 0] + 0.5 * 1
    A[hi, 1] = A[0, 1] * A[hi, 0] - 0.5 * 1
    A[:, 2] = np.arange(m) % 7 / dt(8)
    info, piv = X.getrf(A.copy(order="F"))
    _, opiv = O.getrf(A.astype(np.float64).copy(order="F"))
    assert piv[0] == 0 and np.array_equal(piv, opiv)


@pytest.mark.parametrize("m", [50, 400, 900])
def test_panel_nan_never_wins_and_rows_above_stay_finite(m):
    rng = np.random.default_rng(m)
    A = np.asfortranarray(rng.uniform(-1, 1, (m, 40)))
    A[m - 3:m - 1] *= 1e-6                       # not chosen among the first pivots
    A[m - 2, 20] = np.nan
    A[m - 3, 22] = np.inf
    L = A.copy(order="F")
    info, piv = X.getrf(L)
    assert piv[20] != m - 2 and (20 <= piv[20] < m)
    # the first 20 columns (their rows below 20 may end elsewhere) and the rows
    # chosen before the NaN's column are untouched by it
    B = A.copy(order="F")
    B[m - 2, 20] = B[m - 3, 22] = 0.5
    R = B.copy(order="F")
    X.getrf(R)
    rows = lambda M: sorted(map(tuple, M[20:, :20]))            # noqa: E731
    assert np.array_equal(L[:20, :20], R[:20, :20]) and rows(L) == rows(R)
    assert np.isfinite(L[:20]).all()


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("m,col", [(64, 0), (300, 17), (700, 63)])
def test_panel_zero_pivot_reports_its_column(dt, m, col):
    rng = np.random.default_rng(m)
    A = np.asfortranarray(rng.uniform(-1, 1, (m, 64)).astype(dt))
    A[:, col] = 0
    L = A.copy(order="F")
    info, piv = X.getrf(L)
    assert info == col + 1 and piv[col] == col
    assert np.all(L[:, col] == 0)
