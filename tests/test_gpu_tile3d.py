"""GPU: the 3D tile kernels of the record levels (rows of at most 64 cells
whole, longer ones in windows of 60; 4 x 4 rows a tile) at the level-1 sizes
where tiles and windows begin and end, with every level but the coarsest on
them (no one-workgroup tail, no row kernels above level 0), Dirichlet walls,
solids at tile borders.  16-bit records, which stay on the march kernels,
run through the same sizes.  Bars are the repository's: V-cycle 2e-5 (FP32
levels), 5e-2 (BF16 levels) of the oracle's, pressures 2e-5."""
import numpy as np
import pytest

import cases
import oracle_bind as ob
import uaamg_amd as U

pytestmark = pytest.mark.gpu

FORMS = U.FORM_DEFAULT & ~U.FORM_TAIL & ~U.FORM_ROWS_COARSE
#: level-1 sides; the grid has twice the cells, one more where `odd`
LEVEL1 = [((59, 7, 5), 0), ((60, 8, 9), 1), ((61, 9, 12), 0), ((63, 12, 13), 1), ((64, 13, 16), 0), ((65, 5, 7), 0),
          ((66, 17, 8), 1), ((120, 6, 6), 0), ((121, 11, 5), 1), ((9, 31, 33), 0), ((33, 32, 10), 1)]


@pytest.mark.parametrize("wall", [None, [1, 0, 0, 1, 0, 1]], ids=["neumann", "dirichlet"])
@pytest.mark.parametrize("n1,odd", LEVEL1, ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
@pytest.mark.parametrize("prec,bar", [(U.FP32, 2e-5), (U.MIXED_F64, 2e-5), (U.MIXED_BF16, 5e-2), (U.MIXED_BF16R, 5e-2)],
                         ids=["fp32", "mixed64", "bf16", "bf16r"])
def test_tile_levels(gpu, prec, bar, n1, odd, wall):
    n = tuple(2 * v + odd for v in n1)
    pb = ob.Problem(n, tuple(v / 64.0 for v in n), None, wall)
    s = np.zeros(pb.shape[::-1], np.uint8)
    rng = np.random.default_rng(sum(n))
    for i, j, k in zip(rng.integers(2, n[0], 5), rng.integers(2, n[1], 5), rng.integers(2, n[2], 5)):
        s[k:k + 3, j:j + 2, i:i + 3] = 1
    for a in range(8, min(n[1], n[2]), 8):                 # where tiles meet
        s[a:a + 2, a:a + 2, 118:124] = 1
        s[a:a + 2, a:a + 2, 3:6] = 1
    pb.solid = s.reshape(-1)
    print(f"[tile3d] precision={prec} n={n} wall={wall}", flush=True)
    c = U.Context(precision=prec, tol_mode=U.TOL_REL, forms=FORMS)
    c.set_grid(pb.n, pb.h, pb.solid, pb.wall)
    m = pb.fluid_interior_mask()
    r = cases.random_rhs(pb, np.random.default_rng(5)) * m
    z, zo = c.apply(r), ob.uaamg_apply(pb, r)
    assert np.abs(z[m] - zo[m]).max() <= bar * np.abs(zo[m]).max()
    po, _ = ob.pcg(pb, r, 400, 1e-6, tol_mode=1)
    p, st = c.solve(r, 400, 1e-6)
    c.close()
    assert st.status == 0
    a, b = p[m], po[m]
    if wall is None:
        a, b = a - a.mean(), b - b.mean()
    assert np.abs(a - b).max() <= 2e-5 * np.abs(b).max()
