"""GPU: a breakdown (p.Ap < 1e-15, pcg.cpp:100) on grids of many workgroups,
where the workgroup that finds it sets the stop flag while others of the same
launch still start: x takes no update, so the pressure stays bit for bit what
it was, in single solves and in batches."""
import numpy as np
import pytest

import cases
import oracle_bind as ob
import uaamg_amd as U

pytestmark = pytest.mark.gpu

# spacing 1 and a right-hand side of 1e-12: p.Ap is about r.r / 4, 1e-18 here
SIZES = [(1024, 512), (1500, 1100), (96, 64, 64), (130, 90, 70)]


def _case(n):
    pb = ob.Problem(n, tuple(float(v) for v in n))
    rng = np.random.default_rng(sum(n))
    m = pb.fluid_interior_mask()
    return pb, 1e-12 * cases.random_rhs(pb, rng) * m, rng.standard_normal(pb.N)


@pytest.mark.parametrize("n", SIZES, ids=lambda n: "x".join(map(str, n)))
@pytest.mark.parametrize("prec", [U.FP64, U.FP32, U.MIXED_F64], ids=["fp64", "fp32", "mixed64"])
def test_single(gpu, prec, n):
    pb, rhs, p0 = _case(n)
    print(f"[breakdown] precision={prec} n={n}", flush=True)
    c = U.Context(precision=prec, tol_mode=U.TOL_REL)
    c.set_grid(pb.n, pb.h, pb.solid, pb.wall)
    for _ in range(3):
        p, st = c.solve(rhs, 20, 1e-8, p0=p0)
        assert st.status == U.BREAKDOWN and st.iters == 1
        np.testing.assert_array_equal(p, p0)
    c.close()


def test_batch(gpu):
    import torch
    b = U.Batch(precision=U.FP32, tol_mode=U.TOL_REL)
    rhs, p0 = [], []
    for n in SIZES:
        pb, r, p = _case(n)
        b.add(pb.n, pb.h, pb.solid, pb.wall)
        rhs.append(torch.from_numpy(r).cuda())
        p0.append(torch.from_numpy(p).cuda())
    print("[breakdown] batch", flush=True)
    for _ in range(3):
        p = [v.clone() for v in p0]
        torch.cuda.synchronize()
        _, st = b.solve_device([v.data_ptr() for v in rhs], [v.data_ptr() for v in p], None, 20, 1e-8)
        torch.cuda.synchronize()
        assert all(s.status == U.BREAKDOWN and s.iters == 1 for s in st)
        assert all(torch.equal(a, c) for a, c in zip(p, p0))
    b.close()
