"""mf_cg_solve_noalloc on a system small enough for one workgroup, when the solve that built the
plan ran on another grid: the plan that exists is used."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("first", [dict(variant=2), dict(grid=64), dict()])
def test_plan_of_an_earlier_solve(mf, orc, torch, first, precision):
    rp, ci, va = mf.workloads.poisson2d(40)
    b, _ = mf.workloads.rhs_from_solution(rp, ci, va, seed=2)
    A = mf.TiledMatrix(rp, ci, va)
    _, i0 = A.cg(b, precision=precision, layout="sell", **first)
    assert i0["status"] == 0 and i0["grid"] == (64 if first else 1)
    o = mf.api.solve_options(precision=precision, layout="sell")
    bt = torch.as_tensor(b, device="cuda")
    for _ in range(2):
        x, info = torch.zeros_like(bt), mf._lib.SolveInfo()
        st = mf._lib.lib().mf_cg_solve_noalloc(A.h, ctypes.c_void_p(bt.data_ptr()), ctypes.c_void_p(x.data_ptr()),
                                               ctypes.byref(o), ctypes.byref(info), None)
        assert st == 0 and info.grid == i0["grid"]
        assert orc.true_relres(rp, ci, va, x.cpu().numpy(), b) <= 1.2e-10
    A.close()
