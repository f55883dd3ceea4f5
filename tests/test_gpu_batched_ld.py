"""The batched factor + solve kernels and the Cholesky adjoint at leading
dimensions above the order, through the C plan entry points: bit for bit the
result at leading dimension n, and nothing written between the columns' ends
and the next ones' beginnings.  Orders at the edges of the 32-column panels,
16-column strips and 32-row tiles; LU orders above 256 take the other kernel."""
import ctypes as C

import numpy as np
import pytest

import atlas_amd as X

pytestmark = pytest.mark.gpu
PAD = -7.0
EDGES = [1, 2, 15, 16, 17, 31, 32, 33, 47, 48, 49, 64, 65, 97, 129, 200, 256]


class _Mats:
    """column-major matrices at their own leading dimensions on the GPU"""

    def __init__(self, mats, extra, torch):
        self.shape = [m.shape for m in mats]
        self.ld = [max(m.shape[0] + e, 1) for m, e in zip(mats, extra)]
        self.t = []
        for m, ld in zip(mats, self.ld):
            h = np.full((m.shape[1], ld), PAD, m.dtype)
            h[:, :m.shape[0]] = m.T
            self.t.append(torch.tensor(h, device="cuda"))
        self.ptrs = torch.tensor([t.data_ptr() for t in self.t], dtype=torch.int64, device="cuda")

    def args(self):
        return C.c_void_p(self.ptrs.data_ptr()), (C.c_int * len(self.ld))(*self.ld)

    def get(self):
        """the matrices, after a look at the padding"""
        out = []
        for t, (r, c), ld in zip(self.t, self.shape, self.ld):
            h = t.cpu().numpy()
            assert np.all(h[:, r:] == PAD), (r, c, ld)
            out.append(h[:, :r].T.copy())
        return out


def _run(kind, sizes, dt, nrhs, pads, torch):
    rng = np.random.default_rng(nrhs + len(sizes))
    pre, L = "d" if dt == np.float64 else "s", X.lib()
    A = [rng.uniform(-1, 1, (n, n)) for n in sizes]
    if kind in ("posv", "posv_adjoint"):
        A = [a @ a.T / len(a) + np.eye(len(a)) for a in A]
    rhs = lambda: [rng.uniform(-1, 1, (n, nrhs)).astype(dt) for n in sizes]    # noqa: E731
    pad = lambda k: [(3 * k + i) % 5 + 1 if pads else 0 for i in range(len(sizes))]   # noqa: E731
    As, Bs = _Mats([a.astype(dt) for a in A], pad(0), torch), _Mats(rhs(), pad(1), torch)
    n = (C.c_int * len(sizes))(*sizes)
    info = torch.full((len(sizes),), -7, dtype=torch.int32, device="cuda")
    piv = torch.full((sum(sizes),), -1, dtype=torch.int32, device="cuda")
    off = np.concatenate([[0], np.cumsum(sizes)[:-1]]) * 4 + piv.data_ptr()
    pp = torch.tensor(off, dtype=torch.int64, device="cuda")
    pA, lda = As.args()
    pB, ldb = Bs.args()
    f = getattr(L, "atlmx_%s%s_batch_plan" % (pre, kind))
    f.restype = C.c_void_p
    ptr = lambda t: C.c_void_p(t.data_ptr())                                   # noqa: E731
    out = [As, Bs]
    if kind == "posv":
        h = f(len(sizes), n, pA, lda, nrhs, pB, ldb, ptr(info))
    elif kind == "posv_adjoint":
        Bb, G = _Mats(rhs(), pad(1), torch), _Mats(A if dt == np.float64 else
                                                   [a.astype(dt) for a in A], pad(2), torch)
        pG, ldg = G.args()
        h = f(len(sizes), n, pA, lda, nrhs, pB, Bb.args()[0], ldb, pG, ldg, None)
        out += [Bb, G]
    else:
        h = f(len(sizes), n, pA, lda, ptr(pp), nrhs, pB, ldb, ptr(info))
    assert h
    L.atlmx_batch_run(C.c_void_p(h))
    torch.cuda.synchronize()
    L.atlmx_batch_destroy(C.c_void_p(h))
    return [m for o in out for m in o.get()] + [info.cpu().numpy(), piv.cpu().numpy()]


@pytest.mark.parametrize("kind", ["posv", "gesv", "gesv_t", "posv_adjoint"])
@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("nrhs", [1, 8])
@pytest.mark.parametrize("above", [False, True])
def test_leading_dimensions_above_the_order(kind, dt, nrhs, above):
    import torch
    X.use_torch_stream()
    sizes = EDGES + ([257, 300] if above else [])
    plain = _run(kind, sizes, dt, nrhs, False, torch)
    padded = _run(kind, sizes, dt, nrhs, True, torch)
    for i, (a, b) in enumerate(zip(plain, padded)):
        assert np.array_equal(a, b), i
    if kind != "posv_adjoint":
        assert not plain[-2].any()


def test_largest_lu_orders_and_a_width_from_a_smaller_plan():
    """The largest orders run, with 8 right-hand sides; and an order whose
    panel of 32 columns does not fit runs after a smaller one of its size
    class has been timed."""
    import torch
    X.use_torch_stream()
    L = X.lib()
    for dt, dbl in ((np.float64, 1), (np.float32, 0)):
        for sizes in ([L.atlmx_batch_max_order(1, dbl)], [300], [500]):
            rng = np.random.default_rng(sizes[0])
            A, B = rng.uniform(-1, 1, (sizes[0],) * 2), rng.uniform(-1, 1, (sizes[0], 8))
            As, Bs = _Mats([A.astype(dt)], [0], torch), _Mats([B.astype(dt)], [0], torch)
            piv = [torch.zeros(sizes[0], dtype=torch.int32, device="cuda")]
            info = torch.full((1,), -7, dtype=torch.int32, device="cuda")
            with X.gesv_batch(As.t, piv, Bs.t, info) as plan:
                plan.run()
                torch.cuda.synchronize()
            x = Bs.get()[0].astype(np.float64)
            r = np.abs(B.astype(dt) - A.astype(dt).astype(np.float64) @ x).max()
            assert int(info) == 0
            assert r <= 64 * sizes[0] * np.finfo(dt).eps * np.abs(A).sum(1).max() * np.abs(x).max()
