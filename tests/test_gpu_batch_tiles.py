"""GPU: batches whose members end where the tile kernels' tiles do (2D: 60 x
12 cells, level-0 up 252 columns; 3D record levels: 4 x 4 rows, rows of 64
cells or windows of 60) and the batched CG passes with their finishes, of a
fixed and of a flexible beta, replayed from a graph and eager.  Bar: the
repository's 2e-5 of the oracle's pressure."""
import numpy as np
import pytest

import cases
import oracle_bind as ob
import uaamg_amd as U

pytestmark = pytest.mark.gpu

SIZES = [(59, 23), (60, 24), (61, 25), (121, 37), (251, 21), (252, 36), (253, 22), (505, 40), (150, 300),
         (40, 33, 31), (66, 34, 50), (120, 26, 40), (122, 40, 24), (131, 48, 33)]


def _problem(n):
    pb = ob.Problem(n, tuple(v / 64.0 for v in n), None, [1, 0, 0, 0, 0, 0] if sum(n) % 2 else None)
    s = np.zeros(pb.shape[::-1], np.uint8)
    rng = np.random.default_rng(sum(n))
    for _ in range(5):
        at = [int(rng.integers(2, v - 1)) for v in n]
        s[tuple(slice(a, a + 2) for a in reversed(at))] = 1
    pb.solid = s.reshape(-1)
    return pb


@pytest.mark.parametrize("flexible", [0, 1])
@pytest.mark.parametrize("prec", [U.FP32, U.MIXED_BF16], ids=["fp32", "bf16"])
def test_batch_at_tile_edges(gpu, prec, flexible):
    import torch
    pbs = [_problem(n) for n in SIZES]
    rhs = [1e3 * cases.random_rhs(pb, np.random.default_rng(3)) * pb.fluid_interior_mask() for pb in pbs]
    out = []
    for graph in (1, 0):
        b = U.Batch(precision=prec, tol_mode=U.TOL_REL, use_graph=graph, flexible=flexible)
        for pb in pbs:
            b.add(pb.n, pb.h, pb.solid, pb.wall)
        r = [torch.from_numpy(v).cuda() for v in rhs]
        for _ in range(2):                                  # the second solve replays the first one's graph
            p = [torch.zeros_like(v) for v in r]
            torch.cuda.synchronize()
            rc, st = b.solve_device([v.data_ptr() for v in r], [v.data_ptr() for v in p], None, 500, 1e-6)
            torch.cuda.synchronize()
            out.append([v.cpu().numpy() for v in p])
            assert rc == 0 and all(s.status == 0 for s in st)
        b.close()
    for k, pb in enumerate(pbs):
        print(f"[batch tiles] precision={prec} n={pb.n}", flush=True)
        po, _ = ob.pcg(pb, rhs[k], 500, 1e-8, tol_mode=1)
        m = pb.fluid_interior_mask()
        c = po[m] - (0 if any(pb.wall) else po[m].mean())
        for o in out:
            a = o[k][m] - (0 if any(pb.wall) else o[k][m].mean())
            assert np.abs(a - c).max() <= 2e-5 * np.abs(c).max(), pb.n
        assert np.array_equal(out[0][k], out[1][k])
