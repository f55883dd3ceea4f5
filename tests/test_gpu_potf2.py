"""The Cholesky of one 128-wide diagonal block (and through it potrf): orders
at the edges of its 32-column panels and 64-wide inverses, both triangles,
against |A - L L^T| <= 8 (n + 1) u |L| |L|^T (Higham, Accuracy and Stability,
Theorem 10.3; 8 for the products with the blocks' inverses, whose condition
is below 8 here), the other triangle untouched, and the first failing minor
at every panel and block edge."""
import numpy as np
import pytest

import atlas_amd as X

pytestmark = pytest.mark.gpu


def _spd(rng, n):
    B = rng.standard_normal((n, n))
    return B @ B.T / n + np.eye(n)


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("uplo", [X.Lower, X.Upper])
@pytest.mark.parametrize("n", [1, 16, 17, 31, 32, 33, 48, 63, 64, 65, 95, 96, 97, 127, 128, 129, 160,
                               193, 257, 300])
def test_potrf_block_edges(dt, uplo, n):
    rng = np.random.default_rng(n)
    S = _spd(rng, n).astype(dt)
    S = np.tril(S) + np.tril(S, -1).T
    A = np.asfortranarray(S)
    junk = rng.standard_normal((n, n)).astype(dt)
    keep, other = (np.tril, lambda M: np.triu(M, 1)) if uplo == X.Lower else \
        (np.triu, lambda M: np.tril(M, -1))
    A = np.asfortranarray(keep(A) + other(junk))
    assert X.potrf(A, uplo) == 0
    assert np.array_equal(other(A), other(junk))
    L = keep(A).astype(np.float64)
    L = L if uplo == X.Lower else L.T
    u = np.finfo(dt).eps / 2
    assert np.all(np.abs(S.astype(np.float64) - L @ L.T) <= 8 * (n + 1) * u * (np.abs(L) @ np.abs(L).T))


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("uplo", [X.Lower, X.Upper])
@pytest.mark.parametrize("col", [1, 16, 32, 33, 64, 65, 96, 97, 128, 129, 200])
def test_potrf_first_failing_minor(dt, uplo, col):
    rng = np.random.default_rng(col)
    A = np.asfortranarray(_spd(rng, 200).astype(dt))
    A[col - 1, col - 1] = -1
    assert X.potrf(A, uplo) == col


@pytest.mark.parametrize("dt,scale", [(np.float64, 1e-290), (np.float64, 1e290),
                                      (np.float32, 1e-33), (np.float32, 1e33)])
@pytest.mark.parametrize("uplo", [X.Lower, X.Upper])
def test_potrf_pivots_outside_the_short_square_root(dt, scale, uplo):
    """Pivots where the reciprocal square root's steps would over- or
    underflow: the block is done again with the library's square root."""
    n = 150
    S = (_spd(np.random.default_rng(5), n) * scale).astype(dt)
    A = np.asfortranarray(np.tril(S) if uplo == X.Lower else np.triu(np.tril(S).T))
    assert X.potrf(A, uplo) == 0
    L = np.tril(A).astype(np.float64) if uplo == X.Lower else np.triu(A).T.astype(np.float64)
    S = np.tril(S).astype(np.float64)
    u = np.finfo(dt).eps / 2
    E = np.abs(S / scale - np.tril((L / np.sqrt(scale)) @ (L / np.sqrt(scale)).T))
    La = np.abs(L / np.sqrt(scale))
    assert np.all(E <= 8 * (n + 1) * u * (La @ La.T))


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("uplo", [X.Lower, X.Upper])
@pytest.mark.parametrize("bad", [np.inf, np.nan])
@pytest.mark.parametrize("c", [0, 1, 14, 15, 16, 17, 31, 33, 50, 63])
def test_potrf_nonfinite_entry_stays_right_of_its_column(dt, uplo, bad, c):
    """A(70, c) not finite: info names row 70, and that row's entries left of
    column c are what they are without it."""
    n, r = 100, 70
    S = _spd(np.random.default_rng(11), n).astype(dt)
    S = np.tril(S) + np.tril(S, -1).T
    L = np.linalg.cholesky(S.astype(np.float64))
    A = np.asfortranarray(S)
    A[(r, c) if uplo == X.Lower else (c, r)] = bad
    assert X.potrf(A, uplo) == r + 1
    F = (A if uplo == X.Lower else A.T).astype(np.float64)
    tol = 64 * n * np.finfo(dt).eps          # c n u kappa(S) |L|, kappa(S) < 8
    assert np.abs(F[r, :c] - L[r, :c]).max(initial=0) <= tol
    others = [i for i in range(64, n) if i != r]
    assert np.abs(np.tril(F - L)[:64, :64]).max() <= tol
    assert np.abs((F - L)[others, :64]).max() <= tol


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("uplo", [X.Lower, X.Upper])
@pytest.mark.parametrize("n,col", [(20, 9), (100, 1), (100, 17), (100, 33), (100, 75), (128, 128)])
def test_potrf_failure_leaves_the_columns_before_it_factored(dt, uplo, n, col):
    """Within a block of 128: the columns before the failing one hold the
    factor in every row, the failing one and those after it are as given."""
    S = _spd(np.random.default_rng(col), n).astype(dt)
    S = np.tril(S) + np.tril(S, -1).T
    L = np.linalg.cholesky(S.astype(np.float64))
    S[col - 1, col - 1] = -1
    A = np.asfortranarray(S)
    assert X.potrf(A, uplo) == col
    F = A if uplo == X.Lower else A.T
    assert np.array_equal(F[:, col - 1:], S[:, col - 1:])
    # c n u kappa(S) |L|, kappa(S) < 8
    assert np.abs(np.tril(F.astype(np.float64) - L)[:, :col - 1]).max(initial=0) <= \
        64 * n * np.finfo(dt).eps


@pytest.mark.parametrize("dt,jitter", [(np.float64, 1e-6), (np.float64, 1e-13), (np.float32, 1e-5)])
@pytest.mark.parametrize("uplo", [X.Lower, X.Upper])
@pytest.mark.parametrize("n", [33, 64, 100, 128])
def test_potrf_block_backward_stable_on_kernel_matrices(dt, jitter, uplo, n):
    """|A - L L^T| <= 8 (n + 1) u |L| |L|^T whatever the condition of the
    32-column blocks: Gaussian kernel matrices, nearly singular."""
    x = np.sort(np.random.default_rng(n).uniform(0, 10, n))
    S = (np.exp(-0.5 * (x[:, None] - x) ** 2) + jitter * np.eye(n)).astype(dt)
    S = np.tril(S) + np.tril(S, -1).T
    A = np.asfortranarray(S)
    assert X.potrf(A, uplo) == 0
    L = (np.tril(A) if uplo == X.Lower else np.triu(A).T).astype(np.longdouble)
    u = np.finfo(dt).eps / 2
    assert np.all(np.abs(S - L @ L.T) <= 8 * (n + 1) * u * (np.abs(L) @ np.abs(L).T))
