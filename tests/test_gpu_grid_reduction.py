"""Grid reductions at the group sizes where their shape changes: one workgroup, a part-filled
and a full pass of 16 members, the most that reduce in one hop (64) and one more (65)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layout,variant", [("sell", 1), ("sell", 2), ("sell", 4), ("chunks", 4)])
@pytest.mark.parametrize("grid", [1, 2, 15, 16, 17, 33, 63, 64, 65, 128])
def test_fixed_iterations_follow_the_oracle(mf, orc, torch, grid, layout, variant):
    """Seven binary64 iterations on a ragged matrix (n = 2046, 128 tile rows).  A lost, repeated
    or stale record changes a scalar at order 1/grid; rounding in seven steps stays near 1e-14."""
    rp, ci, va = mf.workloads.poisson2d(33, 62)
    b, _ = mf.workloads.rhs_from_solution(rp, ci, va, seed=5)
    A = mf.TiledMatrix(rp, ci, va)
    x, info = A.cg(b, max_iter=7, fixed_iterations=True, layout=layout, variant=variant, grid=grid)
    ref = orc.cg(rp, ci, va, b, tol=0.0, maxit=7)
    assert info["status"] == 0 and info["iterations"] == 7 and info["grid"] == grid
    assert np.allclose(x.cpu().numpy(), ref["x"], rtol=1e-10, atol=1e-12)
    A.close()
