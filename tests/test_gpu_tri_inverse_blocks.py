"""TRSM through the inverted 64 x 64 diagonal blocks: orders at the edges of
the block and of its 16- and 32-wide doubling levels, against a triangular
solve in higher precision, with the bound n u |inv(A)| |A| |x| (Higham,
Accuracy and Stability, section 8.1, times 8 for the products with inverted
blocks); an infinite or NaN entry must not reach solution rows that do not
depend on it."""
import numpy as np
import pytest

import atlas_amd as X

pytestmark = pytest.mark.gpu


def _tri(rng, n, uplo, diag, dt):
    A = rng.uniform(-1, 1, (n, n)) / max(n, 1) ** 0.5
    A[np.arange(n), np.arange(n)] = rng.uniform(1, 2, n) * rng.choice([-1, 1], n)
    return np.asfortranarray(A.astype(dt)), (np.tril if uplo == X.Lower else np.triu)


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("uplo", [X.Lower, X.Upper])
@pytest.mark.parametrize("diag", [X.Unit, X.NonUnit])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 31, 32, 33, 48, 49, 63, 64, 65, 97, 130])
def test_trsm_block_edges(dt, uplo, diag, n):
    rng = np.random.default_rng(n)
    A, keep = _tri(rng, n, uplo, diag, dt)
    B = np.asfortranarray(rng.uniform(-1, 1, (n, 300)).astype(dt))
    Y = X.trsm(X.Left, uplo, X.NoTrans, diag, 1.0, A, B.copy(order="F")).astype(np.float64)
    M = keep(A).astype(np.float64)
    if diag == X.Unit:
        M[np.arange(n), np.arange(n)] = 1.0
    ref = np.linalg.solve(M, B.astype(np.float64))
    u = np.finfo(dt).eps / 2
    bound = 8 * (n + 1) * u * (np.abs(np.linalg.inv(M)) @ (np.abs(M) @ np.abs(ref))) + 1e-300
    assert np.all(np.abs(Y - ref) <= bound)


@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_trsm_nonfinite_entry_stays_below_its_row(bad):
    rng = np.random.default_rng(3)
    n = 64
    A, _ = _tri(rng, n, X.Lower, X.NonUnit, np.float64)
    A[40, 7] = bad
    B = np.asfortranarray(rng.uniform(-1, 1, (n, 300)))
    Y = X.trsm(X.Left, X.Lower, X.NoTrans, X.NonUnit, 1.0, A, B.copy(order="F"))
    ref = np.linalg.solve(np.tril(A)[:40, :40], B[:40])
    assert np.allclose(Y[:40], ref, rtol=1e-11, atol=1e-13)
    assert not np.isfinite(Y[40]).any()


@pytest.mark.parametrize("dt,tiny,big", [(np.float64, 1e-300, 1e200), (np.float32, 1e-30, 1e20)])
@pytest.mark.parametrize("row", [20, 40])
def test_trsm_overflow_in_the_inverse_stays_below_its_row(dt, tiny, big, row):
    """A small diagonal entry and a large one below it overflow in the
    block's inverse: the rows above the large entry do not depend on it."""
    n = 64
    A, _ = _tri(np.random.default_rng(3), n, X.Lower, X.NonUnit, dt)
    A[5, 5], A[6:, 5], A[row, 5] = tiny, 0, big
    B = np.asfortranarray(np.random.default_rng(4).uniform(-1, 1, (n, 300)).astype(dt))
    B[5] = tiny
    Y = X.trsm(X.Left, X.Lower, X.NoTrans, X.NonUnit, 1.0, A, B.copy(order="F"))
    ref = np.linalg.solve(np.tril(A)[:row, :row].astype(np.float64), B[:row])
    M = np.abs(np.tril(A)[:row, :row].astype(np.float64))
    M[:, 5] = M[5] = 0
    M[5, 5] = 1          # row 5 and column 5 stand apart
    bound = 8 * (n + 1) * np.finfo(dt).eps * (np.abs(np.linalg.inv(M)) @ (M @ np.abs(ref))) + 1e-30
    assert np.all(np.abs(Y[:row] - ref) <= bound)
