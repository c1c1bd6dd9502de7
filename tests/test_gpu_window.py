"""CG whose search direction is gathered from an LDS window: systems small enough for one
workgroup (the default up to 2,048 rows) and irregular rows over several."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("nx,ny,one", [(1, 1, True), (1, 16, True), (17, 1, True), (31, 33, True), (32, 32, True),
                                       (25, 41, True), (32, 64, True), (3, 683, False)])
def test_one_workgroup_systems(mf, orc, torch, nx, ny, one, precision):
    """Iterates of the textbook recurrence (binary64), and solves to 1e-10, at the edges of the
    rows a thread holds (1,024) and of the one-workgroup range (2,048)."""
    rp, ci, va = mf.workloads.poisson2d(nx, ny)
    b, _ = mf.workloads.rhs_from_solution(rp, ci, va, seed=2)
    A = mf.TiledMatrix(rp, ci, va)
    if precision == "fp64":
        its = min(7, nx * ny // 4)
        x, info = A.cg(b, max_iter=its, fixed_iterations=True)
        ref = orc.cg(rp, ci, va, b, tol=0.0, maxit=its)
        assert info["status"] == 0 and (info["grid"] == 1) == one
        assert np.allclose(x.cpu().numpy(), ref["x"], rtol=1e-10, atol=1e-12)
    x, info = A.cg(b, tol=1e-10, precision=precision)
    ref = orc.cg(rp, ci, va, b, tol=1e-10)
    assert info["status"] == 0
    assert abs(info["iterations"] - ref["iterations"]) <= max(1, int(0.02 * ref["iterations"]))
    assert orc.true_relres(rp, ci, va, x.cpu().numpy(), b) <= 1.2e-10
    # a second right-hand side and an initial guess on the same plan
    x2, info2 = A.cg(2.0 * b, x0=x, tol=1e-10, precision=precision)
    assert info2["status"] == 0 and orc.true_relres(rp, ci, va, x2.cpu().numpy(), 2.0 * b) <= 1.2e-10
    A.close()


@pytest.mark.parametrize("n,grid", [(1500, 1), (1500, 2), (5003, 3), (5003, 5), (20000, 16), (20000, 5), (20000, 3)])
def test_irregular_rows_window(mf, orc, torch, n, grid):
    """Lognormal rows in a band: sorted rows, halo below and above, 1, 2, 4 and 8 rows per
    thread.  Two iterations, as every product enters while rounding is not yet amplified."""
    rp, ci, va, b, _ = mf.workloads.irregular_spd(n=n, band=400, logd_max=2.0)
    A = mf.TiledMatrix(rp, ci, va)
    ref = orc.cg(rp, ci, va, b, tol=0.0, maxit=2)
    x, info = A.cg(b, max_iter=2, fixed_iterations=True, layout="sell", grid=grid)
    assert info["status"] == 0 and info["layout"] in (2, 4, 6) and info["variant"] == 4
    assert np.allclose(x.cpu().numpy(), ref["x"], rtol=1e-10, atol=1e-13 * np.abs(ref["x"]).max())
    # tile-mixed: the window holds the binary32 copy that the other variants gather from
    # memory; only the order of the reductions differs
    xm, im = A.cg(b, max_iter=2, fixed_iterations=True, precision="mixed", layout="sell", grid=grid)
    x2, i2 = A.cg(b, max_iter=2, fixed_iterations=True, precision="mixed", layout="sell", grid=grid, variant=2)
    assert im["variant"] == 4 and i2["variant"] == 2
    assert np.allclose(xm.cpu().numpy(), x2.cpu().numpy(), rtol=1e-9, atol=1e-12 * np.abs(ref["x"]).max())
    A.close()
