"""GPU: FP64 vectors give the same bits whichever kernels run: the default
forms (3D: row kernels and fused flat passes) against the march kernels with
CG passes of their own, at whole rows and windows (128 / 129, 252 / 253), odd
sides, chunks of two planes and more, one level more than the small ones,
walls and solids, cold and warm.  Against the oracle, solved to relres 1e-11:
what is left of the residual is at most in the smoothest mode, where it is
1e-11 sqrt(N) of a white right-hand side's share, 3e-9 at 1e5 cells for each of
the two solves: 1e-8 of the largest pressure."""
import numpy as np
import pytest

import cases
import oracle_bind as ob
import uaamg_amd as U

pytestmark = pytest.mark.gpu

SIZES = [(40, 33, 31), (64, 30, 21), (128, 20, 24), (129, 19, 13), (131, 18, 9), (252, 19, 14), (253, 17, 12), (375, 18, 12), (7, 60, 90), (90, 70, 7), (34, 50, 44)]
PLAIN = U.FORM_DEFAULT & ~(U.FORM_ROWS | U.FORM_PMV)


def _problem(n, wall):
    pb = ob.Problem(n, tuple(v / 64.0 for v in n), None, wall)
    s = np.zeros(pb.shape[::-1], np.uint8)
    rng = np.random.default_rng(sum(n))
    for _ in range(8):
        at = [int(rng.integers(1, max(2, v - 1))) for v in n]
        s[tuple(slice(a, a + 2) for a in reversed(at))] = 1
    pb.solid = s.reshape(-1)
    return pb


def _solve(pb, prec, forms, rhs, tol, p0=None, **kw):
    import torch
    c = U.Context(precision=prec, tol_mode=U.TOL_REL, forms=forms, **kw)
    c.set_grid(pb.n, pb.h, pb.solid, pb.wall)
    r = torch.from_numpy(rhs).cuda()
    p = torch.zeros_like(r) if p0 is None else torch.from_numpy(p0).cuda()
    torch.cuda.synchronize()
    st = c.solve_device(r.data_ptr(), p.data_ptr(), int(p0 is not None), 400, tol)
    torch.cuda.synchronize()
    c.close()
    return p.cpu().numpy(), st


@pytest.mark.parametrize("wall", [None, [1, 1, 0, 1, 0, 0]], ids=["neumann", "dirichlet"])
@pytest.mark.parametrize("n", SIZES, ids=lambda n: "x".join(map(str, n)))
def test_same_bits_3d(gpu, n, wall):
    pb = _problem(n, wall)
    print(f"[fp64 order] n={n} wall={wall}", flush=True)
    m = pb.fluid_interior_mask()
    rng = np.random.default_rng(9)
    rhs, p0 = 1e3 * cases.random_rhs(pb, rng) * m, rng.standard_normal(pb.N) * m
    for prec in (U.FP64, U.MIXED_F64):
        for start in (None, p0):
            a, sa = _solve(pb, prec, U.FORM_DEFAULT, rhs, 1e-8, start)
            b, sb = _solve(pb, prec, PLAIN, rhs, 1e-8, start)
            assert sa.kernel_set == 2 and sa.forms_used & U.FORM_ROWS and sb.kernel_set == 0
            assert sa.status == sb.status == 0 and sa.iters == sb.iters
            assert np.array_equal(a, b), (prec, np.abs(a - b).max())
    po, res = ob.pcg(pb, rhs, 400, 1e-11, tol_mode=1)
    a, sa = _solve(pb, U.FP64, U.FORM_DEFAULT, rhs, 1e-11)
    # the reference's breakdown test (p.Ap < 1e-15, pcg.cpp:100) may end either there
    assert sa.status in (U.OK, U.BREAKDOWN) and abs(sa.iters - res.iters) <= 1
    x, y = a[m], po[m]
    if wall is None:
        x, y = x - x.mean(), y - y.mean()
    assert np.abs(x - y).max() <= 1e-8 * np.abs(y).max()


@pytest.mark.parametrize("kc", [6, 8, 10, 12, 14])
@pytest.mark.parametrize("n", [(130, 97), (251, 50), (253, 63), (300, 41)], ids=lambda n: f"{n[0]}x{n[1]}")
def test_chunk_lengths_2d(gpu, n, kc):
    """The 2D level-0 up kernel with three and four rows a thread and, above 12
    rows a chunk, the march kernel: V-cycle equal to the oracle's to 1e-12, the
    fused CG passes equal to the separate ones bit for bit, and so in FP32."""
    print(f"[chunks 2d] n={n} kc={kc}", flush=True)
    for wall in (None, [1, 0, 0, 1, 0, 0]):
        pb = _problem(n, wall)
        m = pb.fluid_interior_mask()
        rhs = 1e3 * cases.random_rhs(pb, np.random.default_rng(5)) * m
        for prec in (U.FP64, U.FP32):
            c = U.Context(precision=prec, march_kc_min=kc)
            c.set_grid(pb.n, pb.h, pb.solid, pb.wall)
            z, zo = c.apply(rhs), ob.uaamg_apply(pb, rhs)
            c.close()
            assert np.abs(z[m] - zo[m]).max() <= (1e-12 if prec == U.FP64 else 2e-5) * np.abs(zo[m]).max()
            tol = 1e-8 if prec == U.FP64 else 1e-6
            a, sa = _solve(pb, prec, U.FORM_DEFAULT, rhs, tol, march_kc_min=kc)
            b, sb = _solve(pb, prec, U.FORM_DEFAULT & ~U.FORM_PMV, rhs, tol, march_kc_min=kc)
            assert sa.kernel_set == 2 and sb.kernel_set == 0 and sa.status == sb.status == 0
            assert sa.iters == sb.iters and np.array_equal(a, b)
