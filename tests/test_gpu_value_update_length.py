"""Device value updates of a matrix whose CSR arrays hold more than its rows use: entries before
``rowptr[0]`` and after ``rowptr[n]``.  Values are indexed by CSR position, as in the host array,
so a tensor has to reach ``rowptr[n]``; other lengths are refused before anything is launched."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _padded(mf, lead, trail, seed):
    rp, ci, va = mf.workloads.poisson2d(23, 19)
    rng = np.random.default_rng(seed)
    va = va * np.where(rng.random(va.size) < 0.5, 1.0, rng.uniform(1.0, 2.0, va.size))
    pad = np.full(lead, np.nan), np.full(trail, np.nan)
    col = np.concatenate([np.zeros(lead, np.int32), ci, np.zeros(trail, np.int32)]).astype(np.int32)
    return (rp + lead).astype(np.int32), col, np.concatenate([pad[0], va, pad[1]])


@pytest.mark.parametrize("policy", ["lossless", "rowscaled"])
@pytest.mark.parametrize("lead,trail", [(0, 0), (5, 0), (0, 3), (37, 11)])
def test_positions_of_a_padded_csr(mf, torch, lead, trail, policy):
    rp, ci, v0 = _padded(mf, lead, trail, 1)
    v1 = _padded(mf, lead, trail, 2)[2]
    x = np.random.default_rng(3).uniform(-1, 1, rp.size - 1)
    A, B = (mf.TiledMatrix(rp, ci, v0, class_policy=policy) for _ in range(2))
    try:
        t = torch.as_tensor(v1, device="cuda")
        for other in (t[:0], t[: int(rp[-1]) - 1], torch.cat([t, t[:1]])):
            with pytest.raises(ValueError):
                A.update_values(other)
        A.update_values(torch.zeros_like(t))
        A.update_values(t if trail else t[: int(rp[-1])])
        B.update_values(v1)
        assert A.stats()["nnz_by_class"] == B.stats()["nnz_by_class"]
        for precision in ("fp64", "mixed"):
            for transpose in (False, True):
                y, w = (M.spmv(x, precision=precision, transpose=transpose).cpu().numpy() for M in (A, B))
                assert np.isfinite(w).all() and np.array_equal(y, w)
    finally:
        A.close()
        B.close()


@pytest.mark.parametrize("lead,trail", [(5, 0), (0, 3)])
def test_operator_on_a_padded_csr(mf, orc, torch, lead, trail):
    rp, ci, v0 = _padded(mf, lead, trail, 1)
    op = mf.autograd.SparseOperator(rp, ci, v0, spd=False, precision="fp64")
    try:
        v1 = np.where(np.isnan(v0), 0.0, 1.5 * v0)
        op.set_values(torch.as_tensor(v1, device="cuda"))
        b = np.random.default_rng(4).uniform(-1, 1, rp.size - 1)
        x = op.solve(torch.as_tensor(b, device="cuda")).cpu().numpy()
        used = slice(int(rp[0]), int(rp[-1]))
        assert orc.true_relres((rp - rp[0]).astype(np.int32), ci[used], v1[used], x, b) <= 1.2e-10
    finally:
        op.close()
