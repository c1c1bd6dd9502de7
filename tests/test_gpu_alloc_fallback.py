"""Products and multi-kernel solves when the row streams do not fit the device memory: the tile
chunks, which need no more of it, give the result.  A child process loads the library behind a
hipMalloc that refuses what is larger than a limit."""
import pathlib
import subprocess
import sys
import textwrap

import pytest

pytestmark = pytest.mark.gpu

SHIM = r"""
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stddef.h>
static size_t limit = (size_t)-1;
static int refused = 0;
void shim_limit(size_t bytes) { limit = bytes; refused = 0; }
int shim_refused(void) { return refused; }
int hipMalloc(void **p, size_t n)
{
    static int (*real)(void **, size_t);
    if (!real) {
        void *h = dlopen("libamdhip64.so.7", RTLD_LAZY | RTLD_NOLOAD);
        if (!h) h = dlopen("libamdhip64.so", RTLD_LAZY | RTLD_NOLOAD);
        real = h ? (int (*)(void **, size_t))dlsym(h, "hipMalloc") : 0;
        if (!real) return 2;
    }
    if (n > limit) {
        refused++;
        return 2; /* hipErrorOutOfMemory */
    }
    return real(p, n);
}
"""

CHILD = textwrap.dedent("""
    import ctypes, sys
    import numpy as np
    import torch
    shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
    sys.path[:0] = sys.argv[2:4]
    from __graft_entry__ import load_package
    import oracle
    mf = load_package()
    rp, ci, va = mf.workloads.poisson3d(64)
    va = va * np.where(np.arange(va.size) % 5 == 0, 1.0 + 2.0 ** -30, 1.0)  # classes 0 and 3
    n = rp.size - 1
    rows = np.repeat(np.arange(n), np.diff(rp))
    x = np.random.default_rng(0).uniform(-1, 1, n)
    b = np.random.default_rng(1).uniform(-1, 1, n)
    bt = torch.as_tensor(b, device="cuda")
    mag = np.bincount(rows, np.abs(va * x[ci]), n)
    want = np.bincount(rows, va * x[ci], n)
    for precision, tol in (("fp64", 8 * 2.0 ** -52), ("mixed", 3 * 2.0 ** -24)):
        A = mf.TiledMatrix(rp, ci, va)
        # the workspace vectors (2 MB each) fit, the binary64 stream's values (16 MB) do not
        shim.shim_limit(ctypes.c_size_t(6 << 20))
        for _ in range(2):
            y = A.spmv(x, precision=precision).cpu().numpy()
            assert np.all(np.abs(y - want) <= tol * mag), precision
        assert shim.shim_refused() > 0 or precision == "mixed"
        xs, info = A.cg_multikernel(bt, max_iter=3, fixed_iterations=True, precision=precision)
        assert info["status"] == 0 and info["layout"] == 1, info
        ref = oracle.cg(rp, ci, va, b, tol=0.0, maxit=3)["x"]
        assert np.allclose(xs.cpu().numpy(), ref, rtol=1e-4, atol=1e-4 * np.abs(ref).max())
        xs, info = A.bicgstab_multikernel(bt, max_iter=3, fixed_iterations=True, precision=precision)
        assert info["status"] == 0 and info["layout"] == 1, info
        refused = shim.shim_refused()
        assert refused > 0
        A.spmv(x, precision="fp64")
        assert shim.shim_refused() == refused  # the streams are not tried again on every call
        shim.shim_limit(ctypes.c_size_t(-1))
        A.update_values(va)  # nor given up for good: the next values' layout tries them
        _, info = A.cg_multikernel(bt, max_iter=3, fixed_iterations=True, precision=precision)
        assert info["layout"] in (2, 3), info
        A.close()
        print(precision, "ok", flush=True)
""")


def test_tile_chunks_when_streams_do_not_fit(mf, torch, tmp_path):
    root = pathlib.Path(__file__).resolve().parents[1]
    (tmp_path / "shim.c").write_text(SHIM)
    (tmp_path / "child.py").write_text(CHILD)
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(tmp_path / "shim.so"), str(tmp_path / "shim.c"), "-ldl"], check=True)
    r = subprocess.run([sys.executable, str(tmp_path / "child.py"), str(tmp_path / "shim.so"), str(root), str(root / "oracle")],
                       capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "mixed ok" in r.stdout, r.stdout + r.stderr


def test_tile_mixed_product_builds_no_binary64_stream(mf, torch):
    """Device memory of the first tile-mixed product: the class streams and the workspace, not
    the binary64 stream that it does not read (80 bytes a row here)."""
    rp, ci, va = mf.workloads.poisson3d(100)
    n = rp.size - 1
    A = mf.TiledMatrix(rp, ci, va)
    x = torch.rand(n, dtype=torch.float64, device="cuda")
    y = torch.empty_like(x)
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    A.spmv(x, precision="mixed", out=y)
    torch.cuda.synchronize()
    used = before - torch.cuda.mem_get_info()[0]
    print(f"{used / n:.1f} bytes a row", flush=True)
    assert used < 110 * n
    # the other streams follow when they are asked for
    z = A.spmv(x)
    assert torch.allclose(y, z, rtol=0, atol=12 * 2.0 ** -23)
    xs, info = A.cg_multikernel(z, tol=1e-10, precision="mixed")
    assert info["status"] == 0 and info["precision"] == 1 and info["layout"] in (2, 3)
    A.close()
