"""Multi-kernel solvers on the tile chunks: the layout option."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("dims", [(33, 95), (31, 37, 41)])
def test_chunks_on_request(mf, orc, torch, dims, precision):
    make = mf.workloads.poisson2d if len(dims) == 2 else mf.workloads.poisson3d
    rp, ci, va = make(*dims)
    b, _ = mf.workloads.rhs_from_solution(rp, ci, va, seed=4)
    A = mf.TiledMatrix(rp, ci, va)
    for fn, ref in ((A.cg_multikernel, orc.cg), (A.bicgstab_multikernel, orc.bicgstab)):
        _, auto = fn(b, max_iter=3, fixed_iterations=True, precision=precision)
        assert auto["layout"] in (2, 3)
        x, info = fn(b, max_iter=3, fixed_iterations=True, precision=precision, layout="chunks")
        assert info["status"] == 0 and info["layout"] == 1
        want = ref(rp, ci, va, b, tol=0.0, maxit=3)["x"]
        # tile-mixed CG multiplies the binary32 copy of p: a relative 2^-24 a product
        tol = 1e-10 if precision == "fp64" or ref is orc.bicgstab else 1e-5
        assert np.allclose(x.cpu().numpy(), want, rtol=tol, atol=tol * np.abs(want).max())
        x, info = fn(b, tol=1e-10, precision=precision, layout="chunks")
        assert info["status"] == 0 and info["layout"] == 1
        assert orc.true_relres(rp, ci, va, x.cpu().numpy(), b) <= 1.2e-10
    A.close()
