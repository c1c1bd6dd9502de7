"""All-FP64 BiCGSTAB on both sides of the size at which its binary64 stream stops fitting the
workgroups' LDS next to x and v (80 bytes a row of 160 KB less 4 on 256 workgroups: 511,000
rows): the layout it reports, and the same bits with the stream read from memory."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,layout", [(70, 6), (78, 6), (82, 2), (90, 2)])
def test_layout_and_bits(mf, orc, torch, nx, layout):
    rp, ci, va = mf.workloads.convdiff3d(nx)
    b, _ = mf.workloads.rhs_from_solution(rp, ci, va, seed=2)
    A = mf.TiledMatrix(rp, ci, va)
    x, info = A.bicgstab(b, tol=1e-10)
    y, mem = A.bicgstab(b, tol=1e-10, value_cache=False)
    assert info["status"] == mem["status"] == 0
    assert info["layout"] == layout and mem["layout"] == 2
    assert info["iterations"] == mem["iterations"] and np.array_equal(x.cpu().numpy(), y.cpu().numpy())
    assert orc.true_relres(rp, ci, va, x.cpu().numpy(), b) <= 1.2e-10
    A.close()
