"""GPU: amgpcg at sides with more partial sums than a workgroup has threads
(operator 256, level-0 down 512) and at the first sides whose partials are
folded by a launch of their own.  The CG iterates of a fixed count equal the
oracle's to the repository's FP64 bar (1e-9 of max|x|); FP32 runs the same
launches and is held to the FP32 rounding of r over the smallest eigenvalue,
6e-8 x 4 N^2 / (2 pi^2)."""
import numpy as np
import pytest

import oracle_bind as ob
import uaamg_amd as U
from test_gpu_amgpcg import _rhs
from test_zz_no_alloc import _noalloc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [545, 700, 1024, 1025, 1100])
def test_fixed_count(gpu, N):
    b = _rhs(N)
    print(f"[amgpcg large] N={N}", flush=True)
    xo, ito = ob.amgpcg(N, b, 5, 1e-300)
    for prec in (U.FP64, U.FP32):
        x, it = gpu.amgpcg(N, b, 5, 1e-300, prec)
        assert it == ito == 5
        bar = 1e-9 if prec == U.FP64 else 6e-8 * 4 * N * N / (2 * np.pi ** 2)
        assert np.abs(x - xo).max() <= bar * np.abs(xo).max()


def test_folded_without_allocation(gpu):
    """The folded sums lie in the room of the fixed array too (FP32, N = 1040)."""
    b = _rhs(1040)
    print("[amgpcg large] noalloc N=1040", flush=True)
    for k in (3, 6):
        x, it = gpu.amgpcg(1040, b, k, 1e-300, U.FP32)
        y, iy = _noalloc(gpu, 1040, b, k, 1e-300, U.FP32, None)
        assert it == iy == k
        np.testing.assert_array_equal(x, y)
