"""GPU: the standalone amgpcg entry point at the sizes where its tile and
one-workgroup kernels change: the coarsest sides 2 and 3 alone, one level in
the tail, the tail's largest side (64), the first tiled sides, sides that are
not multiples of a tile, odd sides with odd coarse levels."""
import numpy as np
import pytest

import oracle_bind as ob
import uaamg_amd as U

pytestmark = pytest.mark.gpu


def _rhs(N):
    rng = np.random.default_rng(N)
    b = np.zeros((N + 2, N + 2))
    t = np.pi * np.arange(1, N + 1) / (N + 1)
    b[1:-1, 1:-1] = 20.0 * np.outer(np.sin(t), np.sin(2 * t)) + rng.standard_normal((N, N))
    return b.reshape(-1)


# FP64: the V-cycle rounds as the oracle's does and only the order of the dot
# products differs, so the iterates agree to the repository's FP64 bar (1e-9
# of max|x|).  FP32: both solve A x = b to |r| < 1e-4 |b|; the smallest
# eigenvalue of A is about 2 pi^2, |b| <= max|b| (N + 2), so the two x differ
# by at most 2e-4 (N + 2) max|b| / 19 and, x being smooth, in practice by the
# residual's smooth part: 1e-3 of max|x|, also far above FP32 rounding
# (6e-8 x 4 N^2 / (2 pi^2) = 1e-3 at N = 280).
@pytest.mark.parametrize("N", [2, 3, 4, 5, 6, 7, 9, 31, 63, 64, 65, 66, 95, 127, 128, 130, 131, 257, 280])
@pytest.mark.parametrize("prec", [U.FP64, U.FP32])
def test_amgpcg_tile_edges(gpu, N, prec):
    b = _rhs(N)
    tol = (1e-10 if prec == U.FP64 else 1e-4) * float(np.linalg.norm(b))
    print(f"[amgpcg] N={N} precision={prec}", flush=True)
    xo, ito = ob.amgpcg(N, b, 300, tol)
    x, it = gpu.amgpcg(N, b, 300, tol, prec)
    assert abs(it - ito) <= 1 and it < 300, (it, ito)
    assert np.abs(x - xo).max() <= (1e-9 if prec == U.FP64 else 1e-3) * np.abs(xo).max()


def test_amgpcg_stops_at_max_iter(gpu):
    """Neither a chunk boundary nor the queue of iterations moves the limit."""
    b = _rhs(100)
    for mi in (0, 1, 3, 4, 5):
        xo, ito = ob.amgpcg(100, b, mi, 1e-30)
        x, it = gpu.amgpcg(100, b, mi, 1e-30, U.FP64)
        assert it == ito == mi
        assert np.abs(x - xo).max() <= 1e-9 * max(np.abs(xo).max(), 1.0)
