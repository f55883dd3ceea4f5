"""The batched Cholesky factor + solve at the edges of its 32-column panels
and 32-row tiles, for every right-hand-side count, failing minors in every
part of a panel, and the largest order (where LDS holds no split diagonal
sum).  Bounds: |A - L L^T| <= c (n + 1) u |L| |L|^T elementwise (Higham,
Accuracy and Stability, Theorem 10.3; c = 8 for the products with the
diagonal blocks' inverses, whose condition is below 8 for these matrices),
||b - A x|| <= c n u ||A|| ||x|| in the infinity norm."""
import numpy as np
import pytest

import atlas_amd as X

pytestmark = pytest.mark.gpu


def _spd(rng, n):
    B = rng.standard_normal((n, n))
    return B @ B.T / n + np.eye(n)


def _check(torch, sizes, dt, nrhs, fails=()):
    rng = np.random.default_rng(sum(sizes) + nrhs)
    u = np.finfo(dt).eps / 2
    A0 = [_spd(rng, n).astype(dt) for n in sizes]
    for i, col in fails:
        A0[i][col - 1, col - 1] = -1.0
    up = [np.triu(rng.standard_normal(a.shape), 1).astype(dt) for a in A0]   # never read
    B0 = [rng.uniform(-1, 1, (n, nrhs)).astype(dt) for n in sizes]
    dev = lambda m: torch.tensor(np.ascontiguousarray(m.T), device="cuda")   # noqa: E731
    As, Bs = [dev(np.tril(a) + w) for a, w in zip(A0, up)], [dev(b) for b in B0]
    info = torch.full((len(sizes),), -7, dtype=torch.int32, device="cuda")
    with X.posv_batch(As, Bs if nrhs else [], info) as plan:
        plan.run()
        torch.cuda.synchronize()
    inf = info.cpu().numpy()
    bad = dict(fails)
    for i, n in enumerate(sizes):
        F = As[i].cpu().numpy().T
        assert np.array_equal(np.triu(F, 1), up[i]), n
        if i in bad:
            assert inf[i] == bad[i], (n, inf[i])
            assert np.array_equal(Bs[i].cpu().numpy().T, B0[i]) if nrhs else True
            continue
        assert inf[i] == 0, (n, inf[i])
        L, A = np.tril(F).astype(np.float64), A0[i].astype(np.float64)
        A = np.tril(A) + np.tril(A, -1).T
        assert np.all(np.abs(A - L @ L.T) <= 8 * (n + 1) * u * (np.abs(L) @ np.abs(L).T)), n
        if nrhs:
            x, b = Bs[i].cpu().numpy().T.astype(np.float64), B0[i].astype(np.float64)
            bound = 8 * n * u * np.abs(A).sum(1).max() * np.abs(x).max(0) + 1e-300
            assert np.all(np.abs(b - A @ x).max(0) <= bound), n


EDGES = [1, 2, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65, 95, 96, 97, 127, 129, 191, 193, 257]


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("nrhs", [0, 1, 3, 5, 8])
def test_posv_panel_and_tile_edges(dt, nrhs):
    import torch
    X.use_torch_stream()
    _check(torch, EDGES, dt, nrhs)


@pytest.mark.parametrize("dt", [np.float64, np.float32])
def test_posv_first_failing_minor(dt):
    import torch
    X.use_torch_stream()
    cols = [1, 16, 17, 32, 33, 48, 64, 65, 100]
    _check(torch, [100] * len(cols) + [40, 33], dt, 2, list(enumerate(cols)) + [(9, 40), (10, 33)])


def test_posv_largest_order():
    import torch
    X.use_torch_stream()
    n = X.lib().atlmx_batch_max_order(0, 1)
    _check(torch, [n, 70], np.float64, 8)


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
def test_posv_nonfinite_entry_stays_right_of_its_column(dt, bad):
    """A(70, c) not finite: the factorization stops at row 70, and that row's
    entries left of column c are what they are without it, as a substitution
    leaves them; every other row above the failing panel too."""
    import torch
    X.use_torch_stream()
    n, r = 100, 70
    cols = [0, 1, 7, 14, 15, 16, 17, 30, 31, 33, 47, 50, 63]
    rng = np.random.default_rng(11)
    S = _spd(rng, n).astype(dt)
    L = np.linalg.cholesky(np.tril(S).astype(np.float64) + np.tril(S, -1).T.astype(np.float64))
    As = []
    for c in cols:
        A = np.tril(S)
        A[r, c] = bad
        As.append(torch.tensor(np.ascontiguousarray(A.T), device="cuda"))
    info = torch.full((len(cols),), -7, dtype=torch.int32, device="cuda")
    with X.posv_batch(As, [], info) as plan:
        plan.run()
        torch.cuda.synchronize()
    assert info.cpu().tolist() == [r + 1] * len(cols)
    # |L - fl(L)| <= c n u kappa(S) |L| in norm; kappa(S) < 8 here
    tol = 64 * n * np.finfo(dt).eps
    for c, A in zip(cols, As):
        F = A.cpu().numpy().T.astype(np.float64)
        assert np.abs(F[r, :c] - L[r, :c]).max(initial=0) <= tol, c
        assert not np.isfinite(F[r, c]), c
        others = [i for i in range(64, n) if i != r]
        assert np.abs(np.tril(F - L)[:64, :64]).max() <= tol, c
        assert np.abs((F - L)[others, :64]).max() <= tol, c


def _cholesky_by_16(A):
    """batch of FP32 matrices: right-looking, 16 columns at a time, divisions
    and substitutions, every operation rounded (products fused)"""
    f = np.float32
    fma = lambda a, b, c: (a.astype(np.float64) * b + c).astype(f)     # noqa: E731
    A = np.tril(A)
    n = A.shape[1]
    for k in range(0, n, 16):
        e = min(n, k + 16)
        for j in range(k, e):
            A[:, j, j] = np.sqrt(A[:, j, j])
            A[:, j + 1:, j] /= A[:, j, j, None]
            A[:, j + 1:, j + 1:e] = fma(-A[:, j + 1:, j, None], A[:, None, j + 1:e, j],
                                        A[:, j + 1:, j + 1:e])
        S = np.zeros_like(A[:, e:, e:])
        for j in range(k, e):
            S = fma(A[:, e:, j, None], A[:, None, e:, j], S)
        A[:, e:, e:] -= S
    return np.tril(A)


@pytest.mark.parametrize("n,count", [(8, 2000), (20, 1000), (32, 1000), (64, 300), (100, 200)])
def test_posv_rounding_no_larger_than_by_substitution(n, count):
    """The mean error of the FP32 factors over a batch against that of the
    same batch by divisions and substitutions; 2% for the samples' spread."""
    import torch
    X.use_torch_stream()
    rng = np.random.default_rng(n)
    A = rng.uniform(-1, 1, (count, n, n))
    A = (A @ A.transpose(0, 2, 1) / n + 0.05 * np.eye(n)).astype(np.float32)
    A = np.tril(A) + np.tril(A, -1).transpose(0, 2, 1)
    L = np.linalg.cholesky(A.astype(np.float64))
    dev = torch.tensor(A, device="cuda")
    info = torch.zeros(count, dtype=torch.int32, device="cuda")
    with X.posv_batch(list(dev), [], info) as plan:
        plan.run()
        torch.cuda.synchronize()
    assert not info.any()
    err = lambda F: (np.linalg.norm(F - L, axis=(1, 2)) / np.linalg.norm(L, axis=(1, 2))).mean()  # noqa: E731
    F = np.tril(dev.cpu().numpy().transpose(0, 2, 1)).astype(np.float64)
    assert err(F) <= 1.02 * err(_cholesky_by_16(A).astype(np.float64))


def _kernel_matrix(rng, n, jitter, dt):
    """Gaussian kernel of sorted points, nearly singular but for the jitter"""
    x = np.sort(rng.uniform(0, 10, n))
    A = (np.exp(-0.5 * (x[:, None] - x) ** 2) + jitter * np.eye(n)).astype(dt)
    return np.tril(A) + np.tril(A, -1).T


@pytest.mark.parametrize("dt,jitter", [(np.float64, 1e-6), (np.float64, 1e-10),
                                       (np.float64, 1e-13), (np.float32, 1e-3),
                                       (np.float32, 1e-5)])
def test_posv_backward_stable_on_kernel_matrices(dt, jitter):
    """|A - L L^T| <= 8 (n + 1) u |L| |L|^T whatever the condition of the
    diagonal blocks (Higham, Accuracy and Stability, Theorem 10.3): a product
    with a block's inverse alone misses it by its condition."""
    import torch
    X.use_torch_stream()
    rng = np.random.default_rng(2)
    A0 = [_kernel_matrix(rng, n, jitter, dt) for n in (33, 40, 64, 100, 128, 200, 256)]
    As = [torch.tensor(a, device="cuda") for a in A0]
    Bs = [torch.tensor(rng.uniform(-1, 1, (2, len(a))).astype(dt), device="cuda") for a in A0]
    B0 = [b.cpu().numpy().T.astype(np.longdouble) for b in Bs]
    info = torch.full((len(A0),), -7, dtype=torch.int32, device="cuda")
    with X.posv_batch(As, Bs, info) as plan:
        plan.run()
        torch.cuda.synchronize()
    assert not info.any()
    u = np.finfo(dt).eps / 2
    for a, t, b, b0 in zip(A0, As, Bs, B0):
        n, A = len(a), a.astype(np.longdouble)
        L, x = np.tril(t.cpu().numpy().T).astype(np.longdouble), b.cpu().numpy().T
        assert np.all(np.abs(A - L @ L.T) <= 8 * (n + 1) * u * (np.abs(L) @ np.abs(L).T)), n
        # two triangular solves on top of the factor's bound
        bound = 24 * (n + 1) * u * (np.abs(L) @ np.abs(L).T) @ np.abs(x)
        assert np.all(np.abs(b0 - A @ x.astype(np.longdouble)) <= bound), n


def test_posv_rounding_on_a_graded_spectrum():
    """Eigenvalues from 1 to 1e-3: the Schur complements shrink, and a sum
    carried over all columns before it meets the entry rounds at the entry's
    first size.  The residual against that of updates 16 columns at a time;
    2% for the samples' spread."""
    import torch
    X.use_torch_stream()
    n, count = 256, 12
    rng = np.random.default_rng(8)
    q = np.linalg.qr(rng.standard_normal((count, n, n)))[0]
    A = ((q * 1e-3 ** (np.arange(n) / (n - 1))) @ q.transpose(0, 2, 1)).astype(np.float32)
    A = np.tril(A) + np.tril(A, -1).transpose(0, 2, 1)
    dev = torch.tensor(A, device="cuda")
    info = torch.zeros(count, dtype=torch.int32, device="cuda")
    with X.posv_batch(list(dev), [], info) as plan:
        plan.run()
        torch.cuda.synchronize()
    assert not info.any()

    def resid(F):
        F = np.tril(F).astype(np.float64)
        return np.linalg.norm(A - F @ F.transpose(0, 2, 1), axis=(1, 2)).mean()
    assert resid(dev.cpu().numpy().transpose(0, 2, 1)) <= 1.02 * resid(_cholesky_by_16(A))
