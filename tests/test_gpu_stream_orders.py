"""Rows sorted by length for one solver leave the other solvers and variants as on a fresh matrix:
the layout they report and the bits they return do not depend on which call came first."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# fixed iterations: every product of the call enters the iterate
CALLS = {
    "cg": ("cg", {}),
    "cg1": ("cg", dict(variant=1)),
    "cg3": ("cg", dict(variant=3)),
    "cgm": ("cg", dict(precision="mixed")),
    "bicg": ("bicgstab", {}),
    "bicgm": ("bicgstab", dict(precision="mixed")),
}


@pytest.fixture(scope="module")
def system(mf):
    rp, ci, va, b, _ = mf.workloads.irregular_spd(n=20000, band=400, logd_max=2.0)
    return rp, ci, va, b


def _run(A, b, call, grid):
    fn, kw = CALLS[call]
    x, info = getattr(A, fn)(b, max_iter=2, fixed_iterations=True, layout="sell", grid=grid, **kw)
    assert info["status"] == 0 and info["grid"] == grid
    return x.cpu().numpy(), info["layout"]


# 1, 2 and 4 rows per thread
@pytest.mark.parametrize("grid", [40, 16, 5])
def test_layout_and_bits_do_not_depend_on_earlier_calls(mf, torch, system, grid):
    rp, ci, va, b = system
    # at 4 rows per thread the pipelined variant is refused, and the textbook variant keeps the
    # tile chunks beside sorted streams
    calls = [c for c in CALLS if grid > 5 or c not in ("cg1", "cg3")]
    fresh = {}
    for c in set(calls) | {"cg1"}:
        A = mf.TiledMatrix(rp, ci, va)
        fresh[c] = _run(A, b, c, grid)
        A.close()
    assert fresh["cg"][1] in (4, 5)  # sorted
    for first in ("cg", "cg1", "bicg", "cgm"):
        A = mf.TiledMatrix(rp, ci, va)
        for c in [first] + calls:
            x, layout = _run(A, b, c, grid)
            assert layout == fresh[c][1], (first, c)
            assert np.array_equal(x, fresh[c][0]), (first, c)
        # values given on the device reach both orders
        A.update_values(torch.as_tensor(va, device="cuda"))
        for c in calls:
            x, layout = _run(A, b, c, grid)
            assert layout == fresh[c][1] and np.array_equal(x, fresh[c][0]), (first, c)
        A.close()
