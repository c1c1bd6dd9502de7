"""A batch member's solve reads its own system only: a neighbour whose right-hand side is not
finite, or overflows, leaves every other system's bits as they are without it."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _batch_cg(mf, torch, B, b, **kw):
    """Batch.cg without its exception for a system that breaks down."""
    o = mf.api.solve_options(**kw)
    x = torch.zeros_like(b)
    infos = (mf._lib.SolveInfo * B.count)()
    mf._lib.lib().mf_cg_solve_batched(B.h, ctypes.c_void_p(b.data_ptr()), ctypes.c_void_p(x.data_ptr()),
                                      ctypes.byref(o), 0, infos, None, None)
    torch.cuda.synchronize()
    return B.unpack(x), mf._lib.info_dicts(infos)


# rows of 1, 2, 4 and 16 members of at most 1,024 rows; planes narrow (LDS window) and wide (p
# gathered from memory)
NARROW = [(17, 61), (31, 33), (40, 50), (60, 61), (11, 12, 13), (64, 65), (120, 130), (33, 32)]
WIDE = [(40, 50, 3), (50, 41, 2), (45, 45, 7), (60, 50, 5), (25, 41)]


@pytest.mark.parametrize("bad", [np.nan, np.inf, 1e200])
@pytest.mark.parametrize("prec,layout,shift", [("fp64", "auto", 0.05), ("mixed", "sell", 0.05), ("mixed", "auto", 0.0)])
@pytest.mark.parametrize("dims", [NARROW, WIDE], ids=["window", "memory"])
def test_neighbours_of_a_bad_right_hand_side(mf, torch, dims, prec, layout, shift, bad):
    systems, rhs = [], []
    for i, d in enumerate(dims):
        rp, ci, va = (mf.workloads.poisson2d if len(d) == 2 else mf.workloads.poisson3d)(*d)
        rows = np.repeat(np.arange(rp.size - 1), np.diff(rp))
        va = np.where(rows == ci, va + shift, va)
        systems.append((rp, ci, va))
        rhs.append(mf.workloads.rhs_from_solution(rp, ci, va, seed=i)[0])
    B = mf.Batch(systems)
    B.set_rows_per_workgroup(1024)
    kw = dict(tol=1e-10, max_iter=2000, precision=prec, layout=layout)
    want, info = _batch_cg(mf, torch, B, B.pack(rhs), **kw)
    assert all(i["status"] == 0 and i["layout"] != 1 for i in info)
    for first in (0, 1):  # every other system is spoilt, so each healthy one has such neighbours
        spoilt = [np.where(np.arange(r.size) % 97 == 5, bad, r) if i % 2 == first else r for i, r in enumerate(rhs)]
        got, info = _batch_cg(mf, torch, B, B.pack(spoilt), **kw)
        for i, (g, w) in enumerate(zip(got, want)):
            if i % 2 != first:
                assert info[i]["status"] == 0 and 0 <= info[i]["relres_true"] <= 1.2e-10, (i, info[i])
                assert np.array_equal(g, w), i
    B.close()
