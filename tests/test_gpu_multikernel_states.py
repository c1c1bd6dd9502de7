"""Multi-kernel solvers on the tile chunks: the layout option, and what is launched once a solve is
decided."""
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


@pytest.fixture(scope="module")
def far_planes(mf):
    """A 3D Laplacian whose planes lie beyond the streams' 16-bit offsets: tile chunks, and
    products (14 million entries) that outweigh launches."""
    rp, ci, va = mf.workloads.poisson3d(200, 200, 50)
    return (rp, ci, va) + tuple(mf.workloads.rhs_from_solution(rp, ci, va, seed=1))


def _best(A, b, precision, **kw):
    times = []
    for _ in range(5):
        _, info = A.cg_multikernel(b, precision=precision, **kw)
        times.append(info["time_ms"])
    assert info["layout"] == 1
    return min(times), info


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_a_converged_guess_runs_no_products(mf, torch, far_planes, precision):
    """A solve that starts converged takes about as long as one whose iteration limit is 0 (the
    residuals before and after): no batch of iterations is launched."""
    rp, ci, va, b, xs = far_planes
    A = mf.TiledMatrix(rp, ci, va)
    bt, xt = torch.as_tensor(b, device="cuda"), torch.as_tensor(xs, device="cuda")
    limit, info = _best(A, bt, precision, x0=xt, tol=0.0, max_iter=0)
    assert info["status"] == 4 and info["iterations"] == 0
    done, info = _best(A, bt, precision, x0=xt, tol=1e-6)
    assert info["status"] == 0 and info["iterations"] == 0 and 0 <= info["relres_true"] <= 1e-6
    assert info["replacements"] == (1 if precision == "mixed" else 0)
    print(f"limit {limit:.3f} ms, converged {done:.3f} ms", flush=True)
    # tile-mixed: one replaced residual more (three products to two); a batch is sixteen
    assert done <= 2.5 * limit + 0.1
    A.close()


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_launches_after_convergence_do_nothing(mf, torch, far_planes, precision):
    """A solve that converges in its second iteration takes about as long as one that is limited
    to it, although the host enqueued a batch of sixteen."""
    rp, ci, va, b, _ = far_planes
    A = mf.TiledMatrix(rp, ci, va)
    bt = torch.as_tensor(b, device="cuda")
    limit, info = _best(A, bt, precision, tol=0.0, max_iter=2)
    assert info["status"] == 4 and info["iterations"] == 2 and info["relres"] < 1.0
    done, info = _best(A, bt, precision, tol=1.001 * info["relres"])
    assert info["status"] == 0 and info["iterations"] == 2
    print(f"limit {limit:.3f} ms, converged {done:.3f} ms", flush=True)
    # of four products one more (a replaced residual), and 42 launches that do nothing, instead
    # of seventeen products
    assert done <= 1.25 * limit + 0.2
    A.close()
