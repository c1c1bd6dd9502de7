"""Which arithmetic and which SpMV a tile-mixed request runs by default, at the sizes where the
choice changes, and batched members that gather p from an LDS window or from memory."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _shifted(mf, dims, shift):
    make = mf.workloads.poisson2d if len(dims) == 2 else mf.workloads.poisson3d
    rp, ci, va = make(*dims)
    rows = np.repeat(np.arange(rp.size - 1), np.diff(rp))
    return rp, ci, np.where(rows == ci, va + shift, va)


@pytest.mark.parametrize("dims,shift,arith", [((5, 7), 0.03, 0), ((33, 62), 0.03, 0), ((316, 317), 0.03, 0),
                                              ((40, 41, 43), 0.0, 0), ((64, 64, 64), 0.03, 0), ((77, 81, 83), 0.01, None),
                                              ((100, 101, 103), 0.1, 1)])
def test_binary64_stream_on_chip_takes_mixed_requests(mf, orc, torch, dims, shift, arith):
    rp, ci, va = _shifted(mf, dims, shift)
    b, _ = mf.workloads.rhs_from_solution(rp, ci, va, seed=8)
    A = mf.TiledMatrix(rp, ci, va)
    x, info = A.cg(b, tol=1e-10, precision="mixed")
    assert info["status"] == 0 and (arith is None or info["precision"] == arith)
    assert orc.true_relres(rp, ci, va, x.cpu().numpy(), b) <= 1.2e-10
    y, i64 = A.cg(b, tol=1e-10, precision="fp64")
    assert i64["status"] == 0 and orc.true_relres(rp, ci, va, y.cpu().numpy(), b) <= 1.2e-10
    if info["precision"] == 0:  # the same launch
        assert info["layout"] == i64["layout"] == 6 and np.array_equal(x.cpu().numpy(), y.cpu().numpy())
    # a forced layout keeps the tile classes
    x, info = A.cg(b, tol=1e-10, precision="mixed", layout="sell")
    assert info["status"] == 0 and info["precision"] == 1
    assert orc.true_relres(rp, ci, va, x.cpu().numpy(), b) <= 1.2e-10
    A.close()


@pytest.mark.parametrize("rows_per_wg", [1024, 2048, 4096])
@pytest.mark.parametrize("prec,layout,shift,arith", [("fp64", "auto", 0.05, 0), ("mixed", "auto", 0.05, 0),
                                                     ("mixed", "sell", 0.05, 1), ("mixed", "auto", 0.0, 1)])
def test_batched_members(mf, orc, torch, rows_per_wg, prec, layout, shift, arith):
    """Groups of one to sixteen members, ragged last tiles, windows of 1 to 5 columns a row (the
    widest gather from memory)."""
    dims = [(17, 61), (1, 1), (31, 33), (64, 65), (90, 91), (9, 11, 13), (17, 18, 19), (23, 24, 25), (40, 20, 20)]
    systems = []
    for i, d in enumerate(dims):
        rp, ci, va = _shifted(mf, d, shift)
        systems.append((rp, ci, va, mf.workloads.rhs_from_solution(rp, ci, va, seed=i)[0]))
    B = mf.Batch([s[:3] for s in systems])
    B.set_rows_per_workgroup(rows_per_wg)
    b = B.pack([s[3] for s in systems])
    for graph in (False, True, True):
        x, infos, _ = B.cg(b, use_graph=graph, tol=1e-10, precision=prec, layout=layout)
        for (rp, ci, va, bs), xi, inf in zip(systems, B.unpack(x), infos):
            assert inf["status"] == 0 and inf["precision"] == arith
            assert orc.true_relres(rp, ci, va, xi, bs) <= 1.2e-10
            if arith == 0:
                ref = orc.cg(rp, ci, va, bs, tol=1e-10)
                assert abs(inf["iterations"] - ref["iterations"]) <= max(1, 0.02 * ref["iterations"])
    B.close()


@pytest.mark.parametrize("nx", [3, 10, 31, 40, 63, 70])
def test_bicgstab_stream_in_lds(mf, orc, torch, nx):
    """All-FP64 BiCGSTAB with its binary64 stream in LDS: the words and the order of the sums
    are those of the stream in memory, so the bits agree; also transposed."""
    rp, ci, va = mf.workloads.convdiff3d(nx)
    b, _ = mf.workloads.rhs_from_solution(rp, ci, va, seed=2)
    A = mf.TiledMatrix(rp, ci, va)
    for transpose in (False, True):
        x, info = A.bicgstab(b, tol=1e-10, transpose=transpose)
        y, mem = A.bicgstab(b, tol=1e-10, transpose=transpose, value_cache=False)
        assert info["status"] == mem["status"] == 0 and mem["layout"] == 2
        assert info["layout"] == (6 if nx <= 63 else info["layout"])
        assert info["iterations"] == mem["iterations"] and np.array_equal(x.cpu().numpy(), y.cpu().numpy())
    A.close()
