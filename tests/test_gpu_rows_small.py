"""GPU: level-0 rows of 129 to 256 cells in windows of two cells a lane (FP32,
grids whose tiles of 4 planes fit the chip at once) at the widths where the
windows change, chunks of 2 planes with odd and even numbers of planes, and
record levels on the row kernels with such chunks (level 1 of more than 512
tiles of 4 x 4 rows, 65 to 128 cells wide).  Bars are the repository's: V-cycle
2e-5 (FP32; FP64 1e-12), 5e-2 (BF16 levels) of the oracle's, pressures 2e-5."""
import numpy as np
import pytest

import cases
import oracle_bind as ob
import uaamg_amd as U
from test_gpu_rows_wide import BAR

pytestmark = pytest.mark.gpu


def _problem(n, wall):
    pb = ob.Problem(n, tuple(v / 64.0 for v in n), None, wall)
    s = np.zeros(pb.shape[::-1], np.uint8)
    rng = np.random.default_rng(sum(n))
    for i in list(rng.integers(2, n[0], 8)) + [n[0] // 2 - 1, n[0] // 3, 2 * n[0] // 3]:   # anywhere, and where windows meet
        j, k = int(rng.integers(2, n[1] - 2)), int(rng.integers(2, n[2] - 2))
        s[k:k + 2, j:j + 3, i:i + 2] = 1
    pb.solid = s.reshape(-1)
    return pb


def _check(prec, n, wall, iters):
    pb = _problem(n, wall)
    print(f"[rows small] precision={prec} n={n} wall={wall}", flush=True)
    c = U.Context(precision=prec, tol_mode=U.TOL_REL)
    c.set_grid(pb.n, pb.h, pb.solid, pb.wall)
    m = pb.fluid_interior_mask()
    r = cases.random_rhs(pb, np.random.default_rng(5)) * m
    z, zo = c.apply(r), ob.uaamg_apply(pb, r)
    assert np.abs(z[m] - zo[m]).max() <= BAR[prec] * np.abs(zo[m]).max()
    if iters:
        po, _ = ob.pcg(pb, r, 400, 1e-6, tol_mode=1)
        p, st = c.solve(r, 400, 1e-6)
        assert st.status == 0 and st.forms_used & U.FORM_ROWS and st.kernel_set == 2
        a, b = p[m], po[m]
        if wall is None:
            a, b = a - a.mean(), b - b.mean()
        assert np.abs(a - b).max() <= 2e-5 * np.abs(b).max()
    c.close()


@pytest.mark.parametrize("wall", [None, [1, 1, 0, 1, 0, 0]], ids=["neumann", "dirichlet"])
@pytest.mark.parametrize("n", [(129, 18, 9), (130, 17, 10), (131, 16, 11), (151, 33, 14), (251, 19, 8), (252, 15, 13), (253, 20, 9), (256, 18, 12)],
                         ids=lambda n: "x".join(map(str, n)))
def test_narrow_windows(gpu, n, wall):
    for prec in (U.FP32, U.MIXED_BF16R):
        _check(prec, n, wall, True)


@pytest.mark.parametrize("n", [(40, 33, 9), (64, 18, 11), (128, 35, 6), (97, 16, 34)], ids=lambda n: "x".join(map(str, n)))
def test_two_plane_chunks(gpu, n):
    for prec in (U.FP32, U.FP64, U.MIXED_F64):
        _check(prec, n, None, True)


@pytest.mark.parametrize("n", [(256, 131, 98), (202, 130, 140)], ids=lambda n: "x".join(map(str, n)))
def test_record_rows(gpu, n):
    for prec in (U.FP32, U.MIXED_BF16):
        _check(prec, n, None, False)
