"""A fixed number of iterations on a system that binary64 arithmetic solves exactly after one: a
tile-mixed request keeps its answer where the launchers run binary64 for it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [40, 5000, 100_000])
def test_tile_mixed_request_on_a_multiple_of_the_identity(mf, torch, n):
    eye = (np.arange(n + 1, dtype=np.int32), np.arange(n, dtype=np.int32), np.full(n, 2.0))
    b = np.random.default_rng(0).uniform(-1, 1, n)
    kw = dict(max_iter=9, fixed_iterations=True, precision="mixed")
    A = mf.TiledMatrix(*eye)
    for call in (dict(), dict(layout="sell"), dict(layout="chunks")):
        x, info = A.cg(b, **kw, **call)
        assert info["status"] == 0 and info["iterations"] == 9
        if info["precision"] == 0:  # (class streams: the recurrence's r, not x, goes to zero)
            assert np.allclose(x.cpu().numpy(), 0.5 * b, rtol=1e-14, atol=0)
    # a binary64 request reports the breakdown
    with pytest.raises(mf.MfError) as e:
        A.cg(b, max_iter=9, fixed_iterations=True)
    assert e.value.status == 5
    A.close()
    B = mf.Batch([eye] * 3)
    x, infos, _ = B.cg(B.pack([b, 3.0 * b, 0.0 * b]), **kw)
    for s, (xi, info) in enumerate(zip(B.unpack(x), infos)):
        assert info["status"] == 0 and info["iterations"] == (0 if s == 2 else 9)
        assert info["precision"] == 0 and np.allclose(xi, (0.5, 1.5, 0.0)[s] * b, rtol=1e-14, atol=0)
    B.close()
