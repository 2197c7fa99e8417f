"""GPU: the 2D tile kernels (60 x 12 cells of a level per workgroup; level 0
up: 252 columns) at the sizes where tiles begin and end: one cell less, exactly one and
one more than a tile per axis, several tiles, odd sides, sides of 4 and 5
(hierarchies of one or two levels), Dirichlet walls, solids on the tile
borders.  Bars are the repository's: FP64 V-cycle 1e-12 and iterations within
one of the oracle's, pressure to the accuracy of a solve to relres 1e-8 (1e-7);
FP32 2e-5.  The fused CG passes equal the separate ones bit for bit."""
import numpy as np
import pytest

import cases
import oracle_bind as ob
import uaamg_amd as U

pytestmark = pytest.mark.gpu

SIZES = [(59, 11), (60, 12), (61, 13), (64, 16), (65, 17), (63, 15), (120, 24), (121, 25), (181, 49), (9, 130), (130, 9), (7, 6),
         (256, 150), (251, 21), (252, 22), (253, 23), (505, 40)]


def _problem(n, wall):
    pb = ob.Problem(n, (n[0] / 64.0, n[1] / 60.0), None, wall)
    s = np.zeros(pb.shape[::-1], np.uint8)
    rng = np.random.default_rng(n[0] * 1000 + n[1])
    if min(n) > 8:
        for i, j in zip(rng.integers(2, n[0], 6), rng.integers(2, n[1], 6)):
            s[j:j + 2, i:i + 3] = 1
        for i in range(60, n[0], 60):                  # where tiles meet
            s[2:4, i:i + 2] = 1
        for j in range(12, n[1], 12):
            s[j:j + 2, 3:5] = 1
    pb.solid = s.reshape(-1)
    return pb


@pytest.mark.parametrize("wall", [None, [1, 0, 0, 1, 0, 0]], ids=["neumann", "dirichlet"])
@pytest.mark.parametrize("n", SIZES, ids=lambda n: f"{n[0]}x{n[1]}")
@pytest.mark.parametrize("prec", [U.FP64, U.FP32, U.MIXED_F64], ids=["fp64", "fp32", "mixed64"])
def test_tile_levels_and_solve(gpu, prec, n, wall):
    pb = _problem(n, wall)
    print(f"[tile2d] precision={prec} n={n} wall={wall}", flush=True)
    c = U.Context(precision=prec, tol_mode=U.TOL_REL)
    c.set_grid(pb.n, pb.h, pb.solid, pb.wall)
    m = pb.fluid_interior_mask()
    r = 1e3 * cases.random_rhs(pb, np.random.default_rng(5)) * m
    z, zo = c.apply(r), ob.uaamg_apply(pb, r)
    assert np.abs(z[m] - zo[m]).max() <= (1e-12 if prec == U.FP64 else 2e-5) * np.abs(zo[m]).max()
    tol = 1e-8 if prec == U.FP64 else 1e-6
    po, res = ob.pcg(pb, r, 400, tol, tol_mode=1)
    p, st = c.solve(r, 400, tol)
    pf, sf = U.Context(precision=prec, tol_mode=U.TOL_REL, forms=U.FORM_DEFAULT & ~U.FORM_PMV), None
    pf.set_grid(pb.n, pb.h, pb.solid, pb.wall)
    pp, sf = pf.solve(r, 400, tol)                     # the same with the CG passes as launches of their own
    pf.close()
    c.close()
    assert st.status == sf.status == 0 and st.iters == sf.iters and np.array_equal(p, pp)
    if prec == U.FP64:
        assert abs(st.iters - res.iters) <= 1, (st.iters, res.iters)
    a, b = p[m], po[m]
    if wall is None:
        a, b = a - a.mean(), b - b.mean()
    bar = (1e-7 if prec == U.FP64 else 2e-5) * np.abs(b).max()
    assert np.abs(a - b).max() <= bar


GMG_SIZES = [(111, 47), (112, 48), (113, 49), (57, 97), (168, 72), (169, 73), (224, 25), (300, 200), (80, 40), (40, 24)]


@pytest.mark.parametrize("n", GMG_SIZES, ids=lambda n: f"{n[0]}x{n[1]}")
@pytest.mark.parametrize("kind", [(U.PRECOND_GMG, ob.PRECOND_GMG), (U.PRECOND_AMG, ob.PRECOND_AMG)], ids=["gmg", "amg"])
def test_gmg_tiles(gpu, kind, n):
    """The GMG / AMG tile kernels (56 x 24 cells) and their one-workgroup levels
    at the sizes where tiles end and where levels move into the one workgroup:
    the FP64 cycle equals the oracle's bit for bit, FP32 to 1e-4."""
    pb = _problem(n, None)
    print(f"[gmg tiles] n={n}", flush=True)
    m = pb.fluid_interior_mask()
    r = cases.random_rhs(pb, np.random.default_rng(7)) * m
    zo = ob.precond_apply(pb, r, kind[1])
    for prec in (U.FP64, U.FP32, U.MIXED_F64):
        c = U.Context(precision=prec, preconditioner=kind[0])
        c.set_grid(pb.n, pb.h, pb.solid, pb.wall)
        z = c.apply(r)
        c.close()
        if prec == U.FP64:
            assert np.array_equal(z[m], zo[m])
        assert np.abs(z[m] - zo[m]).max() <= 1e-4 * np.abs(zo[m]).max()
