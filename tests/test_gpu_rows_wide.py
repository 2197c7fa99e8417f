"""GPU: level-0 row kernels on rows cut into windows (FP32: more than 256
cells, FP64: more than 128) at the widths where the windows change: one more
cell than a whole row, the largest row of two windows and one more, windows
that end on a cell pair or inside one, Dirichlet walls and solids at window
borders.  Bars are the repository's: V-cycle 1e-12 (FP64), 2e-5 (FP32), 5e-2
(BF16 levels) of the oracle's; FP64 PCG iterations within one.  (After 70 and
more iterations the FP64 pressure itself depends on the order of the dot
products: at nx = 129 it is 1.5e-9 of its maximum from the oracle's with these
kernels and with the march kernels, whose V-cycle equals the oracle's bit for
bit, so the pressure is held to the solve's accuracy only.)"""
import numpy as np
import pytest

import cases
import oracle_bind as ob
import uaamg_amd as U

pytestmark = pytest.mark.gpu

NY, NZ = 19, 9


def _problem(nx, wall):
    pb = ob.Problem((nx, NY, NZ), (nx / 64.0, NY / 64.0, NZ / 64.0), None, wall)
    s = np.zeros(pb.shape[::-1], np.uint8)
    rng = np.random.default_rng(nx)
    for i in rng.integers(2, nx, 12):                     # blocks anywhere along the row
        s[3:6, 4:9, i:i + 3] = 1
    for i in (nx // 2 - 1, nx // 3, 2 * nx // 3):         # and where windows of 2 or 3 meet
        s[2:5, 10:13, i:i + 2] = 1
    pb.solid = s.reshape(-1)
    return pb


def _ctx(pb, **kw):
    c = U.Context(tol_mode=U.TOL_REL, **kw)
    c.set_grid(pb.n, pb.h, pb.solid, pb.wall)
    return c


WIDTHS = {U.FP64: [129, 130, 131, 252, 253, 255, 256, 375],
          U.MIXED_F64: [130, 253],
          U.FP32: [257, 258, 260, 503, 504, 505, 512, 747],
          U.MIXED_BF16: [260, 505],
          U.MIXED_BF16R: [260, 505]}
BAR = {U.FP64: 1e-12, U.MIXED_F64: 2e-5, U.FP32: 2e-5, U.MIXED_BF16: 5e-2, U.MIXED_BF16R: 5e-2}


@pytest.mark.parametrize("wall", [None, [1, 1, 0, 1, 0, 0]], ids=["neumann", "dirichlet"])
@pytest.mark.parametrize("prec,nx", [(p, n) for p, ns in WIDTHS.items() for n in ns])
def test_wide_rows(gpu, prec, nx, wall):
    pb = _problem(nx, wall)
    print(f"[wide rows] precision={prec} nx={nx} wall={wall}", flush=True)
    c = _ctx(pb, precision=prec)
    rng = np.random.default_rng(5)
    r = cases.random_rhs(pb, rng) * pb.fluid_interior_mask()
    z, zo = c.apply(r), ob.uaamg_apply(pb, r)
    m = pb.fluid_interior_mask()
    assert np.abs(z[m] - zo[m]).max() <= BAR[prec] * np.abs(zo[m]).max()
    po, res = ob.pcg(pb, r, 400, 1e-6, tol_mode=1)
    p, st = c.solve(r, 400, 1e-6)
    c.close()
    assert st.status == 0 and st.forms_used & U.FORM_ROWS and st.kernel_set == 2
    a, b = p[m], po[m]
    if wall is None:
        a, b = a - a.mean(), b - b.mean()
    if prec == U.FP64:
        assert abs(st.iters - res.iters) <= 1, (st.iters, res.iters)
    assert np.abs(a - b).max() <= 2e-5 * np.abs(b).max()
