"""GPU: FP32 vectors on 3D grids of more than 256 cells a row: the fused CG
passes form p, r, the scalars and the dot products in FP64, each rounded once,
so r.r after one iteration is what numpy forms in FP64 from the same FP32
vectors.  (With FP32 products, or alpha, beta and mean rounded to FP32, it is
off by 1e-9 and more.)

The bar, 1e-11 relative: both sides add some 1e5 terms of FP64 products, in
trees or in chains of at most 50 (1e5 x 2^-53 at the very worst, 1e-11); a
cell of Ap or r on whose FP32 rounding the two orders of the FP64 operator
disagree changes r.r by 2^-24 of one cell's share, 1e-12."""
import numpy as np
import pytest

import oracle_bind as ob
import uaamg_amd as U

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wall", [None, [0, 1, 0, 0, 0, 0]], ids=["neumann", "outlet"])
@pytest.mark.parametrize("n", [(257, 19, 20), (300, 24, 9), (512, 18, 12), (747, 12, 10)], ids=lambda n: "x".join(map(str, n)))
@pytest.mark.parametrize("prec", [U.FP32, U.MIXED_BF16], ids=["fp32", "bf16"])
def test_first_iteration(gpu, prec, n, wall):
    print(f"[rows fp64 sums] precision={prec} n={n} wall={wall}", flush=True)
    pb = ob.Problem(n, tuple(float(v) for v in n), None, wall)
    rng = np.random.default_rng(n[0])
    s = np.zeros(pb.shape[::-1], np.uint8)
    for i in rng.integers(2, n[0], 10):
        s[3:5, 4:8, i:i + 3] = 1
    pb.solid = s.reshape(-1)
    m = pb.fluid_interior_mask()
    rhs = np.zeros(pb.N)
    v = rng.integers(-500, 501, int(m.sum())).astype(np.float64)
    d = int(v.sum())
    v[:abs(d)] -= np.sign(d)
    rhs[m] = v
    f32 = lambda a: a.astype(np.float32).astype(np.float64)
    mean = lambda a: a.sum() / a.size if wall is None else 0.0
    c = U.Context(precision=prec, tol_mode=U.TOL_REL)
    c.set_grid(pb.n, pb.h, pb.solid, pb.wall)
    r, p = np.zeros(pb.N), np.zeros(pb.N)
    r[m] = f32(-(v - mean(v)))
    r[m] = f32(r[m] - mean(r[m]))
    z = c.apply(r)[m]
    p[m] = f32(z - mean(z))
    Ap, _ = c.matvec(p)
    rz = (r[m] * z).sum() - mean(z) * r[m].sum()
    r1 = f32(r[m] - rz / (p[m] * Ap[m]).sum() * Ap[m])
    _, st = c.solve(rhs, 1, 1e-12)
    c.close()
    assert st.kernel_set == 2 and st.forms_used & U.FORM_ROWS and st.iters == 1
    want = float((r1 * r1).sum())
    print(f"  r.r {st.rnorm ** 2:.16e} numpy {want:.16e} rel {abs(st.rnorm ** 2 - want) / want:.1e}")
    assert abs(st.rnorm ** 2 - want) <= 1e-11 * want
