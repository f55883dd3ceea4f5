"""The batched LU factor + solve with one panel row per thread (orders up to
256): edges of its 32-column panels, 16-column strips and 32-row tiles, every
right-hand-side count, zero pivots in every part of a panel, the transposed
solve, and a batch one order above, which takes the other kernel.  Pivots
equal the oracle's; |P A - L U| <= gamma_n |L| |U| (Higham, Accuracy and
Stability, Theorem 9.3, doubled for the 4 x 4 inverses); the solve by its
normwise backward error, c n u with c the growth observed (<= 64)."""
import numpy as np
import pytest

import atlas_amd as X
import oracle as O

pytestmark = pytest.mark.gpu


def _run(torch, sizes, dt, nrhs, zeros=(), trans=False):
    rng = np.random.default_rng(sum(sizes) * 3 + nrhs)
    u = np.finfo(dt).eps / 2
    A0 = [rng.uniform(-1, 1, (n, n)).astype(dt) for n in sizes]
    for i, col in zeros:
        A0[i][:, col] = 0
    B0 = [rng.uniform(-1, 1, (n, nrhs)).astype(dt) for n in sizes]
    dev = lambda m: torch.tensor(np.ascontiguousarray(m.T), device="cuda")   # noqa: E731
    As, Bs = [dev(a) for a in A0], [dev(b) for b in B0]
    piv = [torch.full((n,), -1, dtype=torch.int32, device="cuda") for n in sizes]
    info = torch.full((len(sizes),), -7, dtype=torch.int32, device="cuda")
    mk = X.gesv_t_batch if trans else X.gesv_batch
    with mk(As, piv, Bs if nrhs else [], info) as plan:
        plan.run()
        torch.cuda.synchronize()
    inf, zero = info.cpu().numpy(), dict(zeros)
    for i, n in enumerate(sizes):
        F, p = As[i].cpu().numpy().T.astype(np.float64), piv[i].cpu().numpy()
        A = A0[i].astype(np.float64)
        if dt == np.float64:
            assert np.array_equal(p, O.getrf(A.copy(order="F"))[1]), n
        P = A.copy()
        for k, q in enumerate(p):
            assert k <= q < n
            P[[k, q]] = P[[q, k]]
        L, U = np.tril(F, -1) + np.eye(n), np.triu(F)
        assert np.all(np.abs(P - L @ U) <= 4 * (n + 1) * u * (np.abs(L) @ np.abs(U)) + 1e-300), n
        assert np.abs(np.tril(F, -1)).max(initial=0) <= 1.0
        if i in zero:
            assert inf[i] == zero[i] + 1
            continue
        assert inf[i] == 0
        if nrhs:
            x, b = Bs[i].cpu().numpy().T.astype(np.float64), B0[i].astype(np.float64)
            M = A.T if trans else A
            r = np.abs(b - M @ x).max(0) / (np.abs(M).sum(1).max() * np.abs(x).max(0))
            assert np.all(r <= 64 * max(n, 8) * u), (n, r.max() / (n * u))


EDGES = [1, 2, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65, 79, 81, 95, 97, 127, 129, 160, 191,
         193, 224, 255, 256]


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("nrhs", [0, 1, 3, 5, 8])
def test_gesv_panel_strip_and_tile_edges(dt, nrhs):
    import torch
    X.use_torch_stream()
    _run(torch, EDGES, dt, nrhs)


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("nrhs", [1, 8])
def test_gesv_transposed(dt, nrhs):
    import torch
    X.use_torch_stream()
    _run(torch, EDGES, dt, nrhs, trans=True)


@pytest.mark.parametrize("dt", [np.float64, np.float32])
def test_gesv_zero_pivots(dt):
    import torch
    X.use_torch_stream()
    cols = [0, 15, 16, 31, 32, 47, 63, 99]
    _run(torch, [100] * len(cols) + [64], dt, 2, list(enumerate(cols)))


def test_gesv_above_the_one_row_orders():
    import torch
    X.use_torch_stream()
    _run(torch, [257, 40, 300], np.float64, 2)


@pytest.mark.parametrize("dt,e", [(np.float64, -1060), (np.float64, 1000), (np.float32, -140),
                                  (np.float32, 120)])
@pytest.mark.parametrize("trans", [False, True])
@pytest.mark.parametrize("nrhs", [1, 8])
def test_gesv_pivots_without_a_normal_reciprocal(dt, e, trans, nrhs):
    """U of small integers times 2^e, its diagonal powers of two: the solution
    is integers and every step exact, so it must come out bit for bit, though
    1 / U(i, i) over- or underflows."""
    import torch
    X.use_torch_stream()
    rng = np.random.default_rng(nrhs)
    A0, B0, X0 = [], [], []
    for n in (1, 7, 40, 100):
        U = np.triu(rng.integers(-1, 2, (n, n)), 1) * (rng.random((n, n)) < 2.0 / n)
        U = U + np.diag(rng.choice([1, 2, 4], n) * rng.choice([-1, 1], n))
        x = rng.integers(-3, 4, (n, nrhs))
        A0.append(np.ldexp(U.astype(np.float64), e).astype(dt))
        B0.append(np.ldexp(((U.T if trans else U) @ x).astype(np.float64), e).astype(dt))
        X0.append(x)
    dev = lambda m: torch.tensor(np.ascontiguousarray(m.T), device="cuda")   # noqa: E731
    As, Bs = [dev(a) for a in A0], [dev(b) for b in B0]
    piv = [torch.zeros(len(a), dtype=torch.int32, device="cuda") for a in A0]
    info = torch.full((len(A0),), -7, dtype=torch.int32, device="cuda")
    with (X.gesv_t_batch if trans else X.gesv_batch)(As, piv, Bs, info) as plan:
        plan.run()
        torch.cuda.synchronize()
    assert not info.any()
    for b, x in zip(Bs, X0):
        assert np.array_equal(b.cpu().numpy().T, x.astype(dt))


def _lu_by_16(A):
    """batch of FP32 matrices: LU by divisions, substitutions and updates 16
    columns at a time, every operation rounded (products fused); the factors
    and the row order"""
    f = np.float32
    fma = lambda a, b, c: (a.astype(np.float64) * b + c).astype(f)     # noqa: E731
    A = A.copy()
    b, n, _ = A.shape
    rows, idx = np.tile(np.arange(n), (b, 1)), np.arange(b)
    for k in range(0, n, 16):
        e = min(n, k + 16)
        for j in range(k, e):
            p = j + np.argmax(np.abs(A[:, j:, j]), axis=1)
            for M in (A, rows):
                M[idx, j], M[idx, p] = M[idx, p], M[idx, j]
            A[:, j + 1:, j] /= A[:, j, j, None]
            A[:, j + 1:, j + 1:e] = fma(-A[:, j + 1:, j, None], A[:, None, j, j + 1:e],
                                        A[:, j + 1:, j + 1:e])
        for j in range(k, e):
            A[:, j + 1:e, e:] = fma(-A[:, j + 1:e, j, None], A[:, None, j, e:], A[:, j + 1:e, e:])
        S = np.zeros_like(A[:, e:, e:])
        for j in range(k, e):
            S = fma(A[:, e:, j, None], A[:, None, j, e:], S)
        A[:, e:, e:] -= S
    return A, rows


@pytest.mark.parametrize("n,count", [(8, 2000), (20, 1000), (32, 1000), (64, 400), (100, 300)])
def test_gesv_rounding_no_larger_than_by_substitution(n, count):
    """The mean residual of the FP32 factors over a batch against that of the
    same batch by divisions and substitutions; 2% for the samples' spread."""
    import torch
    X.use_torch_stream()
    A = np.random.default_rng(n).uniform(-1, 1, (count, n, n)).astype(np.float32)
    dev = torch.tensor(np.ascontiguousarray(A.transpose(0, 2, 1)), device="cuda")
    piv = torch.zeros(count, n, dtype=torch.int32, device="cuda")
    info = torch.zeros(count, dtype=torch.int32, device="cuda")
    with X.gesv_batch(list(dev), list(piv), [], info) as plan:
        plan.run()
        torch.cuda.synchronize()
    assert not info.any()
    F, p = dev.cpu().numpy().transpose(0, 2, 1), piv.cpu().numpy()
    rows, idx = np.tile(np.arange(n), (count, 1)), np.arange(count)
    for j in range(n):
        rows[idx, j], rows[idx, p[:, j]] = rows[idx, p[:, j]], rows[idx, j]

    def resid(F, rows):
        P = np.take_along_axis(A, rows[:, :, None], 1).astype(np.float64)
        E = P - (np.tril(F, -1).astype(np.float64) + np.eye(n)) @ np.triu(F).astype(np.float64)
        return (np.linalg.norm(E, axis=(1, 2)) / np.linalg.norm(P, axis=(1, 2))).mean()
    assert resid(F, rows) <= 1.02 * resid(*_lu_by_16(A))


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_gesv_nonfinite_entry_stays_below_its_row(dt, bad):
    """An entry right of the first panel, in the row that becomes pivot row j,
    is not finite: its column's entries above row j, and every other column's
    top 32 rows, are what they are without it, as a substitution leaves them."""
    import torch
    X.use_torch_stream()
    n, tops = 100, [1, 2, 3, 6, 14, 15, 16, 19, 29, 31]
    S = np.random.default_rng(4).uniform(-1, 1, (n, n)).astype(dt)

    def run(mats):
        As = [torch.tensor(np.ascontiguousarray(a.T), device="cuda") for a in mats]
        piv = [torch.zeros(n, dtype=torch.int32, device="cuda") for _ in mats]
        info = torch.zeros(len(mats), dtype=torch.int32, device="cuda")
        with X.gesv_batch(As, piv, [], info) as plan:
            plan.run()
            torch.cuda.synchronize()
        return [a.cpu().numpy().T for a in As], [p.cpu().numpy() for p in piv]
    (R,), (p,) = run([S])
    rows = np.arange(n)
    for k, q in enumerate(p):
        rows[[k, q]] = rows[[q, k]]
    cols = [32 + (7 * j) % 60 for j in tops]
    mats = []
    for j, c in zip(tops, cols):
        M = S.copy()
        M[rows[j], c] = bad
        mats.append(M)
    F, piv = run(mats)
    # the same sums in another order: c n u |L| |U|, both below 8 here
    tol = 64 * n * np.finfo(dt).eps
    for j, c, f, q in zip(tops, cols, F, piv):
        assert np.array_equal(q[:32], p[:32])
        keep = [i for i in range(n) if i != c]
        assert np.abs(f[:32, keep] - R[:32, keep]).max() <= tol, (j, c)
        assert np.abs(f[:j, c] - R[:j, c]).max() <= tol, (j, c)
        assert not np.isfinite(f[j, c])


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("trans", [False, True])
def test_gesv_backward_stable_where_l11_is_ill_conditioned(dt, trans):
    """Vandermonde and Gaussian kernel matrices: |P A - L U| <= 4 (n + 1) u
    |L| |U| (Higham, Accuracy and Stability, Theorem 9.3, with the reciprocals
    and 4 x 4 inverses) and the solve within twice that more; U12 as a product
    with inv(L11) misses it by 1e5 here."""
    import torch
    X.use_torch_stream()
    A0 = []
    for n in (40, 64, 100, 200, 256):
        x = np.sort(np.random.default_rng(n).uniform(0, 10, n))
        A0 += [np.vander(np.linspace(-1, 1, n), n).astype(dt),
               (np.exp(-0.5 * (x[:, None] - x) ** 2) + 1e-5 * np.eye(n)).astype(dt)]
    B0 = [np.random.default_rng(1).uniform(-1, 1, (len(a), 2)).astype(dt) for a in A0]
    dev = lambda m: torch.tensor(np.ascontiguousarray(m.T), device="cuda")   # noqa: E731
    As, Bs = [dev(a) for a in A0], [dev(b) for b in B0]
    piv = [torch.zeros(len(a), dtype=torch.int32, device="cuda") for a in A0]
    info = torch.full((len(A0),), -7, dtype=torch.int32, device="cuda")
    with (X.gesv_t_batch if trans else X.gesv_batch)(As, piv, Bs, info) as plan:
        plan.run()
        torch.cuda.synchronize()
    u = np.finfo(dt).eps / 2
    tiny = np.finfo(dt).tiny                       # products may underflow
    for i, (a, t, p, b, b0) in enumerate(zip(A0, As, piv, Bs, B0)):
        n, F = len(a), t.cpu().numpy().T.astype(np.longdouble)
        P, rows = a.astype(np.longdouble), np.arange(n)
        for k, q in enumerate(p.cpu().numpy()):
            rows[[k, q]] = rows[[q, k]]
        P = P[rows]
        L, U = np.tril(F, -1) + np.eye(n), np.triu(F)
        LU = np.abs(L) @ np.abs(U)
        assert np.all(np.abs(P - L @ U) <= 4 * (n + 1) * u * LU + n * tiny), n
        x, b0 = b.cpu().numpy().T.astype(np.longdouble), b0.astype(np.longdouble)
        if int(info[i]) or not np.isfinite(x).all():   # FP32: numerically singular
            continue
        r = np.abs(b0 - P.T @ x[rows]) if trans else np.abs(b0[rows] - P @ x)
        bound = LU.T @ np.abs(x[rows]) if trans else LU @ np.abs(x)
        assert np.all(r <= 12 * (n + 1) * u * bound + n * tiny * (1 + np.abs(x).max())), n
