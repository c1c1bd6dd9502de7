"""Products and multi-kernel CG on sliced-ELL row streams: sizes at the edges of waves, ranges
and rows per thread, both precisions, columns that only fit fewer rows per thread, non-finite
elements of x, rows too uneven for the streams, and the states a multi-kernel CG can end in."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _matrix(mf, n, far=0, seed=0):
    """Rows of 3 to 6 entries within 40 columns (one at distance `far`), some missing their
    diagonal, values of every storage class."""
    rng = np.random.default_rng(seed)
    k = rng.integers(3, 7, n)
    rows = np.repeat(np.arange(n), k)
    cols = np.clip(rows + rng.integers(-40, 41, rows.size), 0, n - 1)
    if far:
        cols = np.where(rng.random(rows.size) < 0.01, np.clip(rows + far, 0, n - 1), cols)
    key = np.unique(rows.astype(np.int64) * n + cols)
    rows, cols = key // n, key % n
    kind = rng.integers(0, 4, rows.size)
    val = np.select([kind == 0, kind == 1, kind == 2], [rng.integers(-9, 10, rows.size).astype(float),
                    rng.integers(-99, 100, rows.size) / 64.0, np.float32(rng.normal(size=rows.size)).astype(float)],
                    rng.normal(size=rows.size))
    rp = np.zeros(n + 1, np.int64)
    np.add.at(rp, rows + 1, 1)
    return np.cumsum(rp).astype(np.int32), cols.astype(np.int32), val, rows


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("n,far", [(1, 0), (63, 0), (64, 0), (1023, 0), (1025, 0), (4097, 0), (40000, 31000),
                                   (40000, 33000), (530007, 0)])
def test_product(mf, orc, torch, n, far, precision):
    rp, ci, va, rows = _matrix(mf, n, far)
    A = mf.TiledMatrix(rp, ci, va)
    x = np.random.default_rng(1).uniform(-1, 1, n)
    y = A.spmv(x, precision=precision).cpu().numpy()
    mag = np.bincount(rows, np.abs(va * x[ci]), n)
    if precision == "fp64":
        ref, tol = np.bincount(rows, va * x[ci], n), 8 * np.finfo(float).eps
    else:
        # binary32 copies of x and products: two roundings of 2^-24 a term in the lower classes
        ref, tol = np.bincount(rows, va * x[ci], n), 3 * 2.0 ** -24
    assert np.all(np.abs(y - ref) <= tol * mag)
    # twice the same bits (columns beyond the 16-bit offsets keep the tile chunks, whose LDS
    # sums vary in order), and the transposed product
    if far < 32767 - 1024:
        assert np.array_equal(y, A.spmv(x, precision=precision).cpu().numpy())
    yt = A.spmv(x, precision=precision, transpose=True).cpu().numpy()
    reft, magt = np.bincount(ci, va * x[rows], n), np.bincount(ci, np.abs(va * x[rows]), n)
    assert np.all(np.abs(yt - reft) <= tol * 2 * magt)
    A.close()


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
def test_non_finite_elements_reach_only_their_rows(mf, torch, bad, precision):
    rp, ci, va = mf.workloads.poisson2d(40, 37)
    n = rp.size - 1
    rows = np.repeat(np.arange(n), np.diff(rp))
    A = mf.TiledMatrix(rp, ci, va)
    x = np.random.default_rng(2).uniform(-1, 1, n)
    for at in (0, 39, 40, 700, n - 1):
        xb = x.copy()
        xb[at] = bad
        y = A.spmv(xb, precision=precision).cpu().numpy()
        with np.errstate(invalid="ignore"):
            ref = np.zeros(n)
            np.add.at(ref, rows, va * xb[ci])
        hit = np.zeros(n, bool)
        hit[rows[ci == at]] = True
        assert np.array_equal(np.isfinite(y), ~hit)
        assert np.array_equal(np.isnan(y), np.isnan(ref)) and np.array_equal(y[np.isinf(y)], ref[np.isinf(ref)])
    A.close()


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("dims", [(1, 1), (17, 61), (32, 32), (33, 95), (9, 11, 13), (31, 37, 41)])
def test_multikernel_cg(mf, orc, torch, dims, precision):
    make = mf.workloads.poisson2d if len(dims) == 2 else mf.workloads.poisson3d
    rp, ci, va = make(*dims)
    b, _ = mf.workloads.rhs_from_solution(rp, ci, va, seed=4)
    A = mf.TiledMatrix(rp, ci, va)
    ref = orc.cg(rp, ci, va, b, tol=1e-10)
    x, info = A.cg_multikernel(b, tol=1e-10, precision=precision)
    # (a row of one entry pads to two: one unknown keeps the tile chunks)
    assert info["status"] == 0 and info["variant"] == 0 and info["layout"] in ((1,) if dims == (1, 1) else (2, 3))
    assert abs(info["iterations"] - ref["iterations"]) <= max(1, int(0.02 * ref["iterations"]))
    assert orc.true_relres(rp, ci, va, x.cpu().numpy(), b) <= 1.2e-10
    # a guess, an iteration limit within and at the end of a batch of launches, b = 0
    x2, info2 = A.cg_multikernel(3.0 * b, x0=x, tol=1e-10, precision=precision)
    assert info2["status"] == 0 and orc.true_relres(rp, ci, va, x2.cpu().numpy(), 3.0 * b) <= 1.2e-10
    for its in (0, 7, 15, 16, 17):
        if its + 2 >= ref["iterations"]:
            continue
        xf, inf = A.cg_multikernel(b, max_iter=its, fixed_iterations=True)
        rf = orc.cg(rp, ci, va, b, tol=0.0, maxit=its)
        assert inf["status"] == 0 and inf["iterations"] == its
        assert np.allclose(xf.cpu().numpy(), rf["x"], rtol=1e-9, atol=1e-11)
        xl, inl = A.cg_multikernel(b, tol=1e-10, max_iter=its)
        assert inl["status"] == 4 and inl["iterations"] == its
        assert np.array_equal(xl.cpu().numpy(), xf.cpu().numpy())
    x0, info0 = A.cg_multikernel(0.0 * b, precision=precision)
    assert info0["status"] == 0 and info0["iterations"] == 0 and not x0.any()
    A.close()


def test_uneven_rows_keep_the_tile_chunks(mf, orc, torch):
    rp, ci, va, b, _ = mf.workloads.irregular_spd(n=4000, band=400, logd_max=1.0)
    A = mf.TiledMatrix(rp, ci, va)
    ref = orc.cg(rp, ci, va, b, tol=0.0, maxit=3)
    x, info = A.cg_multikernel(b, max_iter=3, fixed_iterations=True)
    assert info["status"] == 0 and info["layout"] == 1
    assert np.allclose(x.cpu().numpy(), ref["x"], rtol=1e-9, atol=1e-12 * np.abs(ref["x"]).max())
    A.close()


def test_multikernel_breakdown_leaves_the_iterate(mf, torch):
    """A skew-symmetric matrix: p'A p = 0 at the first step."""
    A = mf.TiledMatrix(np.array([0, 1, 2], np.int32), np.array([1, 0], np.int32), np.array([1.0, -1.0]))
    b = torch.ones(2, dtype=torch.float64, device="cuda")
    with pytest.raises(mf.MfError) as e:
        A.cg_multikernel(b)
    assert e.value.status == 5
    A.close()
