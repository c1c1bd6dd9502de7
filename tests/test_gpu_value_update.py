"""Values given on the device: the updated matrix gives the bits of one built from them, when the
storage classes stay and when they change, on every layout and partition already built."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _results(A, b, kinds):
    out = []
    for kind in kinds:
        if kind[0] == "spmv":
            out.append(A.spmv(b, **kind[1]))
        else:
            out.append(getattr(A, kind[0])(b, **kind[1])[0])
    return [o.cpu().numpy() for o in out]


# fixed iterations on grids of at least two workgroups; row streams, persistent streams of both
# kinds, the transposed matrix
KINDS = [("spmv", {}), ("spmv", {"precision": "mixed"}), ("spmv", {"transpose": True}),
         ("cg", dict(max_iter=5, fixed_iterations=True, grid=3, layout="sell")),
         ("cg", dict(max_iter=5, fixed_iterations=True, grid=3, layout="sell", precision="mixed")),
         ("bicgstab", dict(max_iter=4, fixed_iterations=True, precision="mixed", transpose=True))]


def _draw(rng, kind, n):
    """n values of one storage class (0 binary64, 1 binary32, 2 binary16, 3 int8), in class."""
    v = rng.uniform(1.0, 2.0, n)
    if kind == 0:
        return v
    if kind == 1:
        return (v + 2.0 ** -20).astype(np.float32).astype(np.float64)
    if kind == 2:
        return np.round(v * 64.0) / 64.0 + 1.0 / 256.0
    return np.round(v * 20.0)


@pytest.mark.parametrize("policy", ["lossless", "rowscaled", "fp64"])
@pytest.mark.parametrize("n,before,after", [(1, 0, 0), (17, 1, 1), (1037, 2, 2), (4100, 3, 3), (4100, 0, 0), (4100, 1, 1),
                                            (4100, 0, 2), (4100, 3, 1), (4100, 2, 0)])
def test_same_bits_as_a_new_matrix(mf, torch, n, before, after, policy):
    rp, ci, _ = mf.workloads.poisson2d(n, 1) if n < 20 else mf.workloads.poisson2d(17, n // 17)
    n, nnz = rp.size - 1, ci.size
    rng = np.random.default_rng(6)
    diag = np.repeat(np.arange(n), np.diff(rp)) == ci
    va, vb = (np.where(diag, 8.0, -1.0) * _draw(rng, k, nnz) for k in (before, after))
    vb[:: 97] = -vb[:: 97]
    b = rng.uniform(-1, 1, n)
    kinds = KINDS if n > 100 else [k for k in KINDS if "grid" not in k[1]]
    A = mf.TiledMatrix(rp, ci, va, class_policy=policy)
    _results(A, b, kinds)  # every partition and stream exists before the update
    for _ in range(2):     # and the second update starts from the first one's state
        A.update_values(torch.as_tensor(vb, device="cuda"))
        got = _results(A, b, kinds)
        B = mf.TiledMatrix(rp, ci, vb, class_policy=policy)
        assert A.stats()["nnz_by_class"] == B.stats()["nnz_by_class"]
        for g, w, k in zip(got, _results(B, b, kinds), kinds):
            assert np.array_equal(g, w), k
        B.close()
        vb = vb[::-1].copy() if after == before and policy != "rowscaled" else vb
    A.close()


@pytest.mark.parametrize("special", [0.0, -0.0, np.inf, np.nan, 65519.999, 65520.0, 2.0 ** -24, 2.0 ** -25, 1e-300, 127.0,
                                     128.0, -128.0, -129.0, 1.0 + 2.0 ** -11, 1.0 + 2.0 ** -24])
def test_classes_of_special_values(mf, torch, special):
    """A device update gives a tile the class that the host's rule gives it."""
    rp, ci = np.arange(0, 33, dtype=np.int32), np.arange(32, dtype=np.int32)
    for policy in ("lossless", "rowscaled"):
        A = mf.TiledMatrix(rp, ci, np.ones(32), class_policy=policy)
        v = np.ones(32)
        v[5] = special
        A.update_values(torch.as_tensor(v, device="cuda"))
        B = mf.TiledMatrix(rp, ci, v, class_policy=policy)
        assert A.stats()["tiles_by_class"] == B.stats()["tiles_by_class"]
        x = np.arange(32.0)
        for prec in ("fp64", "mixed"):
            assert np.array_equal(A.spmv(x, precision=prec).cpu().numpy(), B.spmv(x, precision=prec).cpu().numpy(),
                                  equal_nan=True)
        A.close()
        B.close()


def test_sorted_rows_after_an_update(mf, orc, torch):
    """Streams of sorted rows are built on the host: they follow values given on the device."""
    rp, ci, va, b, _ = mf.workloads.irregular_spd(n=5003, band=400, logd_max=2.0)
    A = mf.TiledMatrix(rp, ci, va)
    A.cg(b, max_iter=2, fixed_iterations=True, layout="sell", grid=3)
    A.update_values(torch.as_tensor(2.0 * va, device="cuda"))
    x, info = A.cg(b, max_iter=2, fixed_iterations=True, layout="sell", grid=3)
    ref = orc.cg(rp, ci, 2.0 * va, b, tol=0.0, maxit=2)
    assert info["status"] == 0 and info["layout"] in (4, 5)
    assert np.allclose(x.cpu().numpy(), ref["x"], rtol=1e-10, atol=1e-13 * np.abs(ref["x"]).max())
    A.close()
