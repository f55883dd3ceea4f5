"""The work this library is measured on: calls a user's program makes, through
the public device-pointer C ABI (ctypes), the batched plans and the autograd
functions, on operands that already lie in GPU memory.

Matrices are column-major, held as the row-major transpose (a tensor of shape
(columns, rows)), as everywhere in atlas_amd.  Routines that work in place run
on a working copy that `run` refills from the pristine input first, as a
program that factors a fresh matrix each time fills its array.
"""
import math

import numpy as np
import torch

import atlas_amd as X

DT = {"d": torch.float64, "s": torch.float32, "z": torch.complex128}
ESZ = {"d": 8, "s": 4, "z": 16}


def listed():
    return [
        # one block of a small product inside a host loop: latency and the launch decide
        dict(name="dgemm_small", kind="gemm", p="d", ta="N", tb="N", m=96, n=80, k=112,
             alpha=1.0, beta=0.0),
        # the plain DGEMM configuration: C <- A B + C/2 at 2048
        dict(name="dgemm_2048", kind="gemm", p="d", ta="N", tb="N", m=2048, n=2048, k=2048,
             alpha=1.0, beta=0.5),
        # single precision, transposed left operand, no size a multiple of a tile
        dict(name="sgemm_ragged", kind="gemm", p="s", ta="T", tb="N", m=1511, n=777, k=4001,
             alpha=-1.0, beta=1.0),
        # an ordinary small dense solve, one right-hand side
        dict(name="dgesv_500", kind="gesv", p="d", n=500, nrhs=1),
        # the FP64 LU configuration with 64 right-hand sides
        dict(name="dgesv_8192", kind="gesv", p="d", n=8192, nrhs=64),
        # the FP64 Cholesky at an odd order, one right-hand side (normal equations)
        dict(name="dposv_4001", kind="posv", p="d", uplo="L", n=4001, nrhs=1),
        # complex general solve (a frequency-domain system)
        dict(name="zgesv_1024", kind="gesv", p="z", n=1024, nrhs=8),
        # the headline: FP64-accurate solve from an FP32 LU, kappa 1e6 (GMRES refinement)
        dict(name="mixed_16384", kind="mixed", n=16384, nrhs=1, kappa=1e6),
        # the same at an ordinary size and condition, 16 right-hand sides (plain refinement)
        dict(name="mixed_6000", kind="mixed", n=6000, nrhs=16, kappa=1e4),
        # many uneven small SPD systems: Cholesky factor and solve
        dict(name="batch_dposv", kind="bposv", p="d", count=4000, lo=8, hi=512, nrhs=1),
        # many uneven small general systems: LU factor and solve
        dict(name="batch_dgesv", kind="bgesv", p="d", count=4000, lo=8, hi=256, nrhs=1),
        # a differentiated layer of SPD solves: forward, backward
        dict(name="adjoint_dposv", kind="adjoint", count=512, n=256, nrhs=8),
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["gemm", "gemm", "gesv", "posv", "mixed", "bposv", "bgesv", "bgemm",
                       "adjoint"])
    if kind == "gemm":
        m, n, k = size(16, 8192), size(16, 8192), size(16, 8192)
        return dict(kind=kind, p=rng.choice("ds"), ta=rng.choice("NT"), tb=rng.choice("NT"),
                    m=m, n=n, k=k, alpha=1.0, beta=rng.choice([0.0, 0.5, 1.0]))
    if kind == "gesv":
        p = rng.choice("ddz")
        return dict(kind=kind, p=p, n=size(32, 8192 if p == "d" else 1500),
                    nrhs=size(1, 64))
    if kind == "posv":
        return dict(kind=kind, p=rng.choice("dds"), uplo=rng.choice("LU"), n=size(32, 8192),
                    nrhs=size(1, 64))
    if kind == "mixed":
        return dict(kind=kind, n=size(500, 16384), nrhs=rng.choice([1, 1, 16]),
                    kappa=rng.choice([1e2, 1e4, 1e6]))
    if kind in ("bposv", "bgesv"):
        hi = size(32, 512 if kind == "bposv" else 256)
        return dict(kind=kind, p=rng.choice("ds") if kind == "bposv" else "d",
                    count=size(500, 4000), lo=8, hi=hi, nrhs=rng.choice([1, 1, 4]))
    if kind == "bgemm":
        return dict(kind=kind, p=rng.choice("ds"), count=size(500, 4000), lo=16,
                    hi=size(32, 384))
    return dict(kind=kind, count=size(64, 512), n=size(32, 256), nrhs=rng.choice([1, 4, 8]))


# ---- inputs ---------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _uniform(shape, dt, g, lo=-1.0, hi=1.0):
    if dt.is_complex:
        re = torch.rand(shape, dtype=torch.float64, device="cuda", generator=g)
        im = torch.rand(shape, dtype=torch.float64, device="cuda", generator=g)
        return torch.complex(re * (hi - lo) + lo, im * (hi - lo) + lo)
    return torch.rand(shape, dtype=dt, device="cuda", generator=g) * (hi - lo) + lo


def _spd(n, dt, g):
    """B B^T / n + I, B standard normal, exactly symmetric"""
    B = torch.randn(n, n, dtype=torch.float64, device="cuda", generator=g)
    S = B @ B.T
    S /= n
    S = (S + S.T) * 0.5
    S.diagonal().add_(1.0)
    return S.to(dt)


def _haar(n, g):
    Q, R = torch.linalg.qr(torch.randn(n, n, dtype=torch.float64, device="cuda", generator=g))
    Q *= torch.sign(torch.diagonal(R))
    return Q


def _conditioned(n, kappa, g):
    """U diag(sigma) V^T, U and V Haar, sigma geometric from 1 to 1/kappa"""
    sigma = kappa ** (-torch.arange(n, dtype=torch.float64, device="cuda") / max(n - 1, 1))
    return (_haar(n, g) * sigma) @ _haar(n, g).T


def _sizes(case, seed):
    """the orders of a batch come from the case alone; its values from the seed"""
    r = np.random.default_rng(case["count"] * 1009 + case["hi"])
    return [int(v) for v in r.integers(case["lo"], case["hi"] + 1, case["count"])]


def _triples(case):
    r = np.random.default_rng(case["count"] * 1009 + case["hi"])
    return [[int(v) for v in r.integers(case["lo"], case["hi"] + 1, case["count"])]
            for _ in range(3)]


def _cut(buf, shapes):
    out, o = [], 0
    for s in shapes:
        w = math.prod(s)
        out.append(buf[o:o + w].view(*s))
        o += w
    return out


def _batch_inputs(case, seed):
    g, dt, ns = _gen(seed), DT[case["p"]], _sizes(case, seed)
    big = _uniform(sum(n * n for n in ns), dt, g)
    if case["kind"] == "bposv":
        normal = torch.empty_like(big).normal_(generator=g)
        for S, B in zip(_cut(big, [(n, n) for n in ns]), _cut(normal, [(n, n) for n in ns])):
            torch.mm(B, B.T, out=S)
            S.mul_(1.0 / S.shape[0])
            S.diagonal().add_(1.0)
    rhs = _uniform(sum(ns) * case["nrhs"], dt, g)
    return ns, big, rhs


# ---- prepare ----------------------------------------------------------------
def prepare(case, seed):
    kind = case["kind"]
    X.lib()
    X.use_torch_stream()
    g = _gen(seed)
    if kind == "gemm":
        dt, m, n, k = DT[case["p"]], case["m"], case["n"], case["k"]
        A = _uniform((k, m) if case["ta"] == "N" else (m, k), dt, g, -0.5, 0.5)
        B = _uniform((n, k) if case["tb"] == "N" else (k, n), dt, g, -0.5, 0.5)
        C = _uniform((n, m), dt, g, -0.5, 0.5)
        return dict(case=case, A=A, B=B, C=C, W=torch.empty_like(C))
    if kind == "gesv":
        dt, n = DT[case["p"]], case["n"]
        A, B = _uniform((n, n), dt, g), _uniform((case["nrhs"], n), dt, g)
        return dict(case=case, A=A, B=B, LU=torch.empty_like(A), Y=torch.empty_like(B),
                    ipiv=torch.zeros(n, dtype=torch.int32, device="cuda"))
    if kind == "posv":
        dt, n = DT[case["p"]], case["n"]
        A, B = _spd(n, dt, g), _uniform((case["nrhs"], n), dt, g)
        return dict(case=case, A=A, B=B, L=torch.empty_like(A), Y=torch.empty_like(B))
    if kind == "mixed":
        X.set_refine_stop(True)          # LAPACK dsgesv's stopping test
        A, B = _conditioned(case["n"], case["kappa"], g), _uniform(
            (case["nrhs"], case["n"]), torch.float64, g)
        return dict(case=case, A=A, B=B, Y=torch.empty_like(B))
    if kind in ("bposv", "bgesv"):
        ns, big, rhs = _batch_inputs(case, seed)
        F, Y = torch.zeros_like(big), torch.zeros_like(rhs)
        info = torch.zeros(len(ns), dtype=torch.int32, device="cuda")
        As, Bs = _cut(F, [(n, n) for n in ns]), _cut(Y, [(case["nrhs"], n) for n in ns])
        st = dict(case=case, big=big, rhs=rhs, F=F, Y=Y, info=info)
        if kind == "bposv":
            st["plan"] = X.posv_batch(As, Bs, info)
        else:
            st["ipiv"] = torch.zeros(sum(ns), dtype=torch.int32, device="cuda")
            st["plan"] = X.gesv_batch(As, _cut(st["ipiv"], [(n,) for n in ns]), Bs, info)
        return st
    if kind == "bgemm":
        dt = DT[case["p"]]
        ms, ns, ks = _triples(case)
        A = _uniform(sum(m * k for m, k in zip(ms, ks)), dt, g, -0.5, 0.5)
        B = _uniform(sum(k * n for k, n in zip(ks, ns)), dt, g, -0.5, 0.5)
        C = torch.zeros(sum(m * n for m, n in zip(ms, ns)), dtype=dt, device="cuda")
        plan = X.gemm_batch(X.NoTrans, X.NoTrans, 1.0, _cut(A, list(zip(ks, ms))),
                            _cut(B, list(zip(ns, ks))), 0.0, _cut(C, list(zip(ns, ms))))
        return dict(case=case, A=A, B=B, C=C, plan=plan)
    b, n = case["count"], case["n"]
    R = torch.randn(b, n, n, dtype=torch.float64, device="cuda", generator=g)
    A = R @ R.transpose(1, 2).contiguous() / n
    A.diagonal(dim1=1, dim2=2).add_(1.0)
    B = torch.randn(b, n, case["nrhs"], dtype=torch.float64, device="cuda", generator=g)
    W = torch.randn(b, n, case["nrhs"], dtype=torch.float64, device="cuda", generator=g)
    return dict(case=case, A=A.requires_grad_(True), B=B.requires_grad_(True), W=W)


# ---- run ----------------------------------------------------------------------
def run(state):
    case = state["case"]
    kind = case["kind"]
    L = X.lib()
    if kind == "gemm":
        A, B, W = state["A"], state["B"], state["W"]
        if case["beta"] != 0.0:
            W.copy_(state["C"])
        getattr(L, "atlmx_%sgemm" % case["p"])(
            X.NoTrans if case["ta"] == "N" else X.Trans,
            X.NoTrans if case["tb"] == "N" else X.Trans, case["m"], case["n"], case["k"],
            case["alpha"], X.dptr(A), A.shape[1], X.dptr(B), B.shape[1], case["beta"],
            X.dptr(W), case["m"])
        return W
    if kind == "gesv":
        n, nrhs, LU, Y, ipiv = case["n"], case["nrhs"], state["LU"], state["Y"], state["ipiv"]
        LU.copy_(state["A"])
        Y.copy_(state["B"])
        if case["p"] == "z":
            info = L.clapack_zgesv(X.ColMajor, n, nrhs, X.dptr(LU), n, X.dptr(ipiv), X.dptr(Y), n)
        else:
            info = L.atlmx_dgetrf(n, n, X.dptr(LU), n, X.dptr(ipiv))
            L.atlmx_dgetrs(X.NoTrans, n, nrhs, X.dptr(LU), n, X.dptr(ipiv), X.dptr(Y), n)
        return dict(LU=LU, ipiv=ipiv, X=Y, info=info)
    if kind == "posv":
        n, nrhs, F, Y = case["n"], case["nrhs"], state["L"], state["Y"]
        uplo = X.Lower if case["uplo"] == "L" else X.Upper
        F.copy_(state["A"])
        Y.copy_(state["B"])
        info = getattr(L, "atlmx_%spotrf" % case["p"])(uplo, n, X.dptr(F), n)
        getattr(L, "atlmx_%spotrs" % case["p"])(uplo, n, nrhs, X.dptr(F), n, X.dptr(Y), n)
        return dict(F=F, X=Y, info=info)
    if kind == "mixed":
        info, st = X.dsgesv_dev(state["A"], state["B"], state["Y"])
        return dict(X=state["Y"], info=info, fallback=st.fallback)
    if kind in ("bposv", "bgesv"):
        state["F"].copy_(state["big"])
        state["Y"].copy_(state["rhs"])
        state["plan"].run()
        out = dict(F=state["F"], X=state["Y"], info=state["info"])
        if kind == "bgesv":
            out["ipiv"] = state["ipiv"]
        return out
    if kind == "bgemm":
        state["plan"].run()
        return state["C"]
    from atlas_amd.autograd import CholeskySolve
    A, B = state["A"], state["B"]
    Y = CholeskySolve.apply(A, B)
    dA, dB = torch.autograd.grad((Y * state["W"]).sum(), (A, B))
    return dict(X=Y.detach(), dA=dA, dB=dB)


# ---- what one pass cannot do without ---------------------------------------------
def work(case):
    kind = case["kind"]
    if kind == "gemm":
        m, n, k, e = case["m"], case["n"], case["k"], ESZ[case["p"]]
        return {"bytes": e * (m * k + k * n + m * n * (2 if case["beta"] else 1)),
                "flops": 2.0 * m * n * k}
    if kind in ("gesv", "posv"):
        n, r, e = case["n"], case["nrhs"], ESZ[case["p"]]
        c = 4.0 if case["p"] == "z" else 1.0
        f = (2.0 / 3.0 if kind == "gesv" else 1.0 / 3.0) * n ** 3 + 2.0 * n * n * r
        tri = 2.0 if kind == "gesv" else 1.0
        return {"bytes": e * (tri * n * n + 2 * n * r), "flops": c * f}
    if kind == "mixed":
        n, r = case["n"], case["nrhs"]
        return {"bytes": 8.0 * (n * n + 2 * n * r), "flops": 2.0 / 3.0 * n ** 3 + 2.0 * n * n * r}
    if kind in ("bposv", "bgesv"):
        ns, r, e = _sizes(case, 0), case["nrhs"], ESZ[case["p"]]
        c, tri = (1.0 / 3.0, 1.0) if kind == "bposv" else (2.0 / 3.0, 2.0)
        return {"bytes": e * sum(tri * n * n + 2 * n * r for n in ns),
                "flops": sum(c * n ** 3 + 2.0 * n * n * r for n in ns)}
    if kind == "bgemm":
        t = list(zip(*_triples(case)))
        return {"bytes": ESZ[case["p"]] * sum(m * k + k * n + m * n for m, n, k in t),
                "flops": sum(2.0 * m * n * k for m, n, k in t)}
    b, n, r = case["count"], case["n"], case["nrhs"]
    # two factorizations are the autograd function's contract (L is recomputed), then
    # L-bar, L^T L-bar and two triangular solves with n right-hand sides
    return {"bytes": 8.0 * b * (2.5 * n * n + 5 * n * r),
            "flops": b * (2.0 / 3.0 * n ** 3 + 2.0 * n ** 3 + 12.0 * n * n * r)}


def tolerance(case):
    kind = case["kind"]
    single = case.get("p") == "s"
    if kind in ("gemm", "bgemm"):
        return {"rel": 2e-6 if single else 4e-15}
    if kind == "gesv" or kind == "bgesv":
        # the 2^-53 kappa of the worst uniform matrix (heavy-tailed: ~1e-10 is common);
        # pivots are integers and must agree
        return {"rel": 1e-8, "differ": 0.0}
    if kind == "mixed":
        # kappa times the residual that the stopping test leaves
        return {"rel": 4.0 * case["kappa"] * math.sqrt(case["n"]) * 2.0 ** -53}
    # kappa of B B^T / n + I is about 5
    return {"rel": 1e-5 if single else 1e-13}


# ---- the same in plain torch, 64 bits ----------------------------------------------
def exact(case, seed):
    kind = case["kind"]
    st = _inputs_only(case, seed)
    if kind == "gemm":
        a = st["A"].double() if case["ta"] == "T" else st["A"].double().T
        b = st["B"].double() if case["tb"] == "T" else st["B"].double().T
        C = case["alpha"] * (a @ b)
        if case["beta"] != 0.0:
            C += case["beta"] * st["C"].double().T
        return C.T.contiguous()
    if kind == "gesv":
        # LAPACK on the host: its complex pivot rule (|Re| + |Im|) is this library's
        LU, piv = torch.linalg.lu_factor(st["A"].cpu().T)
        Y = torch.linalg.lu_solve(LU, piv, st["B"].cpu().T)
        return dict(LU=LU.T.contiguous(), ipiv=(piv - 1).to(torch.int32),
                    X=Y.T.contiguous(), info=0)
    if kind == "posv":
        A = st["A"].double()
        F = torch.linalg.cholesky(A)
        Y = torch.cholesky_solve(st["B"].double().T, F)
        # column-major lower = the row-major tensor's upper triangle
        F = (F.T.triu() + A.tril(-1)) if case["uplo"] == "L" else (F + A.triu(1))
        return dict(F=F.contiguous(), X=Y.T.contiguous(), info=0)
    if kind == "mixed":
        Y = torch.linalg.solve(st["A"].T, st["B"].T)
        return dict(X=Y.T.contiguous(), info=0, fallback=0)
    if kind in ("bposv", "bgesv"):
        return _exact_batch(case, *st)
    if kind == "bgemm":
        ms, ns, ks = _triples(case)
        out = [(b.double() @ a.double()).reshape(-1) for a, b in
               zip(_cut(st["A"], list(zip(ks, ms))), _cut(st["B"], list(zip(ns, ks))))]
        return torch.cat(out)
    A, B, W = st["A"].detach(), st["B"].detach(), st["W"]
    F = torch.linalg.cholesky(A)
    Y, dB = torch.cholesky_solve(B, F), torch.cholesky_solve(W, F)
    S = -(dB @ Y.transpose(1, 2).contiguous())
    S = S + S.transpose(1, 2)
    dA = S.tril() - torch.diag_embed(S.diagonal(dim1=1, dim2=2)) * 0.5
    return dict(X=Y, dA=dA, dB=dB)


def _inputs_only(case, seed):
    if case["kind"] in ("bposv", "bgesv"):
        return _batch_inputs(case, seed)
    if case["kind"] == "bgemm":
        g, dt = _gen(seed), DT[case["p"]]
        ms, ns, ks = _triples(case)
        return dict(A=_uniform(sum(m * k for m, k in zip(ms, ks)), dt, g, -0.5, 0.5),
                    B=_uniform(sum(k * n for k, n in zip(ks, ns)), dt, g, -0.5, 0.5))
    return prepare(case, seed)


def _exact_batch(case, ns, big, rhs):
    r = case["nrhs"]
    big, rhs = big.cpu().double(), rhs.cpu().double()
    F, Y, piv = torch.empty_like(big), torch.empty_like(rhs), torch.empty(sum(ns), dtype=torch.int32)
    shapes, rows = [(n, n) for n in ns], [(r, n) for n in ns]
    for A, B, G, Z, p in zip(_cut(big, shapes), _cut(rhs, rows), _cut(F, shapes), _cut(Y, rows),
                             _cut(piv, [(n,) for n in ns])):
        if case["kind"] == "bposv":
            C = torch.linalg.cholesky(A)
            G.copy_(C.T + A.tril(-1))
            Z.copy_(torch.cholesky_solve(B.T, C).T)
        else:
            LU, pv = torch.linalg.lu_factor(A.T)
            G.copy_(LU.T)
            Z.copy_(torch.linalg.lu_solve(LU, pv, B.T).T)
            p.copy_(pv - 1)
    out = dict(F=F, X=Y, info=torch.zeros(len(ns), dtype=torch.int32))
    if case["kind"] == "bgesv":
        out["ipiv"] = piv
    return out
