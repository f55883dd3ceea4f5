"""The GEMM's smaller tiles (64 and 32, with the K slices split over one,
two or four wavefront groups): sizes at the edges of the tiles, K at the
edges of the slices and of the groups' shares, operands at odd leading
dimensions and odd element offsets (vector loads off 16-byte alignment).
Small integers make every partial sum exact in both precisions, so the
result must equal the integer product bit for bit, and nothing outside the
M x N block may change."""
import itertools

import numpy as np
import pytest

import atlas_amd as X

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (31, 33, 7), (32, 32, 64), (33, 65, 65), (64, 64, 129), (65, 31, 1023),
          (96, 200, 1025), (32, 40, 0), (1000, 1000, 64), (1000, 1000, 130), (1500, 1500, 127),
          (2100, 2100, 200)]


def _odd(host, dt, torch):
    """column-major host matrix on the GPU at an odd ld and an odd offset"""
    r, c = host.shape
    ld = (r + 2) | 1
    buf = torch.full((c * ld + 1,), -7.0, dtype=dt, device="cuda")
    buf[1:].view(c, ld)[:, :r] = torch.tensor(host.T.copy(), dtype=dt, device="cuda")
    return buf, buf[1:], ld


@pytest.mark.parametrize("p", ["d", "s"])
@pytest.mark.parametrize("ta,tb", list(itertools.product([X.NoTrans, X.Trans], repeat=2)))
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_gemm_tiles_integer_exact_unaligned(p, ta, tb, M, N, K):
    import torch
    dt = torch.float64 if p == "d" else torch.float32
    rng = np.random.default_rng(M * 7 + N * 3 + K)
    A = rng.integers(-4, 5, (M, K) if ta == X.NoTrans else (K, M)).astype(np.float64)
    B = rng.integers(-4, 5, (K, N) if tb == X.NoTrans else (N, K)).astype(np.float64)
    C = rng.integers(-50, 51, (M, N)).astype(np.float64)
    X.use_torch_stream()
    (_, a, lda), (_, b, ldb), (cb, c, ldc) = (_odd(m, dt, torch) for m in (A, B, C))
    before = cb.clone()
    getattr(X.lib(), "atlmx_%sgemm" % p)(ta, tb, M, N, K, 2.0, X.dptr(a), lda, X.dptr(b), ldb,
                                         -3.0, X.dptr(c), ldc)
    ref = 2 * ((A if ta == X.NoTrans else A.T) @ (B if tb == X.NoTrans else B.T)) - 3 * C
    view = before[1:].view(N, ldc)
    view[:, :M] = torch.tensor(ref.T.copy(), dtype=dt, device="cuda")
    assert torch.equal(cb, before)
