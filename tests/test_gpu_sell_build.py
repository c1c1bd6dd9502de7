"""Sliced-ELL streams built on the GPU: ragged sizes around the slice, wave and workgroup edges,
rows whose columns are unsorted, repeated or missing, bands at the limit of the 16-bit column
offsets, classes mixed within a row, and regular wide rows (shared column words)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _random(n, band, seed, unsorted=False, holes=False):
    """Symmetric pattern not needed: one CG step only takes products with A."""
    rng = np.random.default_rng(seed)
    rows, cols = [], []
    for i in range(n):
        k = int(rng.integers(0 if holes else 1, 12))
        c = np.clip(i + rng.integers(-band, band + 1, k), 0, n - 1)
        c = np.append(c, i)
        c = c if unsorted else np.unique(c)
        if holes and i % 7 == 3:
            c = c[:0]
        rows.append(np.full(c.size, i))
        cols.append(c)
    rows, cols = np.concatenate(rows), np.concatenate(cols)
    kind = rng.integers(0, 4, rows.size)
    val = np.select([kind == 0, kind == 1, kind == 2], [rng.integers(-9, 10, rows.size).astype(float),
                    rng.integers(-99, 100, rows.size) / 64.0, np.float32(rng.normal(size=rows.size)).astype(float)],
                    rng.normal(size=rows.size))
    rp = np.zeros(n + 1, np.int64)
    np.add.at(rp, rows + 1, 1)
    return np.cumsum(rp).astype(np.int32), cols.astype(np.int32), val


def _band(n, half):
    i = np.repeat(np.arange(n), 2 * half + 1)
    c = i + np.tile(np.arange(-half, half + 1), n)
    ok = (c >= 0) & (c < n)
    i, c = i[ok], c[ok]
    rp = np.zeros(n + 1, np.int64)
    np.add.at(rp, i + 1, 1)
    return np.cumsum(rp).astype(np.int32), c.astype(np.int32), np.sin(0.1 * i + 0.7 * c) + np.cos(0.1 * c + 0.7 * i)


CASES = [("n1", lambda: _random(1, 1, 0), 1), ("n15", lambda: _random(15, 9, 1), 1), ("n64", lambda: _random(64, 64, 2), 2),
         ("n65 unsorted, repeated", lambda: _random(65, 20, 3, unsorted=True), 3),
         ("n1023 holes", lambda: _random(1023, 90, 4, holes=True), 1), ("n1025", lambda: _random(1025, 90, 5), 1),
         ("n2500 unsorted", lambda: _random(2500, 700, 6, unsorted=True), 2), ("n5000", lambda: _random(5000, 4000, 7), 3),
         ("far columns", lambda: _random(33000, 31000, 8, holes=True), 40), ("wide rows", lambda: _band(3000, 100), 5)]


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("name,make,grid", CASES, ids=[c[0] for c in CASES])
def test_one_step_from_a_guess(mf, torch, name, make, grid, precision):
    """x1 = x0 + alpha r with r = b - A x0 shows every row of the product A x0 (binary64
    stream); alpha = r'r / r'A r takes the product with r (the class streams under "mixed",
    whose binary32 copy of r leaves it within 2^-23 of the sum of |r_i a_ij r_j|)."""
    rp, ci, va = make()
    n = rp.size - 1
    rng = np.random.default_rng(11)
    x0, b = rng.uniform(-1, 1, n), rng.uniform(-1, 1, n)
    rows = np.repeat(np.arange(n), np.diff(rp))

    def times(v, a=va):
        return np.bincount(rows, a * v[ci], n)

    A = mf.TiledMatrix(rp, ci, va)
    x, info = A.cg(b, x0=x0, max_iter=1, fixed_iterations=True, precision=precision, layout="sell", grid=grid)
    assert info["status"] == 0 and info["iterations"] == 1 and info["layout"] != 1
    r = b - times(x0)
    # rounding of a row's sum: its terms' magnitudes times the unit roundoff, times its length
    slack = 32 * np.finfo(float).eps * (np.abs(b) + times(np.abs(x0), np.abs(va))) * (1 + np.diff(rp).max())
    step = x.cpu().numpy() - x0
    pq = r @ times(r)
    got = (step @ r) / (r @ r)
    assert np.all(np.abs(step - got * r) <= np.abs(got) * slack + 1e-15 * (np.abs(x0) + np.abs(step)))
    eps = 2.0 ** -22 if precision == "mixed" else 1e-13
    assert abs((r @ r) / got - pq) <= eps * (np.abs(r) @ times(np.abs(r), np.abs(va)))
    A.close()
