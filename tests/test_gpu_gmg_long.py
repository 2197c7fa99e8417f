"""GPU: GMG and AMG on grids long in one dimension, whose coarsest level (a side
of at most 4) fills most of the one-workgroup kernel's LDS or its four pairs a
thread: the FP64 cycle equals the oracle's bit for bit, FP32 to 1e-4."""
import numpy as np
import pytest

import cases
import oracle_bind as ob
import uaamg_amd as U

pytestmark = pytest.mark.gpu

# padded cells of the coarsest level: FP64 at most 6144, FP32 11815
SIZES = {U.FP64: [(1020, 4), (4, 1020), (598, 4), (2040, 8)], U.FP32: [(1960, 4), (4, 1960), (1130, 4), (2, 2900), (3900, 9)]}


@pytest.mark.parametrize("kind", [(U.PRECOND_GMG, ob.PRECOND_GMG), (U.PRECOND_AMG, ob.PRECOND_AMG)], ids=["gmg", "amg"])
@pytest.mark.parametrize("prec,n", [(p, n) for p, ns in SIZES.items() for n in ns])
def test_long_coarsest(gpu, prec, n, kind):
    pb = ob.Problem(n, (n[0] / 64.0, n[1] / 64.0))
    print(f"[gmg long] precision={prec} n={n}", flush=True)
    m = pb.fluid_interior_mask()
    r = cases.random_rhs(pb, np.random.default_rng(7)) * m
    zo = ob.precond_apply(pb, r, kind[1])
    c = U.Context(precision=prec, preconditioner=kind[0])
    c.set_grid(pb.n, pb.h, pb.solid, pb.wall)
    z = c.apply(r)
    c.close()
    if prec == U.FP64:
        assert np.array_equal(z[m], zo[m])
    assert np.abs(z[m] - zo[m]).max() <= 1e-4 * np.abs(zo[m]).max()


def test_longer_is_refused(gpu):
    for prec, n in ((U.FP64, (1030, 4)), (U.FP32, (1980, 4))):
        pb = ob.Problem(n, (n[0] / 64.0, n[1] / 64.0))
        c = U.Context(precision=prec, preconditioner=U.PRECOND_GMG)
        with pytest.raises(RuntimeError, match="one-workgroup"):
            c.set_grid(pb.n, pb.h, pb.solid, pb.wall)
        c.close()
