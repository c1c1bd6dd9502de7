"""Performance cases of the solver library: the calls that a program using it makes.

A case is one pass through the public Python entry points (``TiledMatrix.cg`` /
``.bicgstab`` / ``.spmv``, ``Batch.cg``, ``autograd.sparse_solve``) on a system that was
converted and uploaded beforehand, as a program that solves with one matrix many times
keeps it.  Right-hand sides are b = A x* with x* ~ U[-1, 1], so x* is the exact solution.
Solves run to a relative residual of 1e-12: two solves that differ only in the order of
their sums then agree to about the same number of digits, whatever the iteration count.

Kinds and ranges (``draw`` spreads sizes over the logarithm of the range, odd boxes):

* ``cg``         5-point (2D) and 7-point (3D) Laplacians on a box with a small reaction term,
                 576 .. 3.2 million rows, binary64 or tile-mixed.
* ``irregular``  CG on a regularised graph Laplacian with lognormal row lengths and random
                 banded columns, 20,000 .. 300,000 rows.
* ``bicg``       BiCGSTAB on 3D upwind convection-diffusion, 4,096 .. 2.1 million rows.
* ``spmv``       one product y = A x, 4,096 .. 4 million rows.
* ``batch``      24 .. 192 independent systems of 1,024 .. 65,536 rows in one launch.
* ``autograd``   forward and backward of two coefficient fields through one operator (its
                 values change within the pass), 16^3 .. 64^3 cells.
"""
import importlib
import math

import numpy as np
import torch

mf = importlib.import_module("mille-feuille_amd")

DEV = "cuda"
TOL = 1e-12


def listed():
    return [
        # the smallest solves: latency of one launch and of its iterations
        dict(name="cg_2d_31x33_fp64", kind="cg", nx=31, ny=33, nz=0, shift=0.0, precision="fp64"),
        # the 2D benchmark size: 64 x 64 Laplacian in binary64
        dict(name="cg_2d_64x64_fp64", kind="cg", nx=64, ny=64, nz=0, shift=0.0, precision="fp64"),
        # an ordinary 3D solve on an odd box
        dict(name="cg_3d_77x81x83_mixed", kind="cg", nx=77, ny=81, nz=83, shift=0.01, precision="mixed"),
        # the headline system, tile-mixed and in binary64
        dict(name="cg_3d_128_mixed", kind="cg", nx=128, ny=128, nz=128, shift=0.0, precision="mixed"),
        dict(name="cg_3d_128_fp64", kind="cg", nx=128, ny=128, nz=128, shift=0.0, precision="fp64"),
        # more rows than one persistent launch holds
        dict(name="cg_3d_144x145x147_mixed", kind="cg", nx=144, ny=145, nz=147, shift=0.01, precision="mixed"),
        # irregular rows and columns (meshes, graphs)
        dict(name="cg_irregular_300k_fp64", kind="irregular", n=300_007, precision="fp64"),
        # nonsymmetric systems: the convection-diffusion benchmark, and an ordinary odd one
        dict(name="bicg_3d_128_mixed", kind="bicg", nx=128, ny=128, nz=128, precision="mixed"),
        dict(name="bicg_3d_63x65x61_fp64", kind="bicg", nx=63, ny=65, nz=61, precision="fp64"),
        # a single product, as a program with its own iteration calls it
        dict(name="spmv_3d_127x129x125_fp64", kind="spmv", nx=127, ny=129, nz=125, precision="fp64"),
        # many small and ordinary systems at once
        dict(name="batch_192_mixed", kind="batch", count=192, precision="mixed"),
        # a training step over two samples of a 64^3 diffusion problem
        dict(name="autograd_64_mixed", kind="autograd", nx=64, precision="mixed"),
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _box(rng, n, d):
    """Sides of a d-dimensional box of about n cells, unequal by up to a fifth."""
    s = n ** (1.0 / d)
    a = max(3, round(s * rng.uniform(0.8, 1.2)))
    b = max(3, round(s * rng.uniform(0.8, 1.2)))
    if d == 2:
        return a, max(3, round(n / a)), 0
    return a, b, max(3, round(n / (a * b)))


def draw(rng):
    kind = rng.choice(["cg", "cg", "cg", "irregular", "bicg", "bicg", "spmv", "batch", "autograd"])
    case = dict(kind=kind, precision=rng.choice(["fp64", "mixed"]))
    if kind == "cg":
        d = rng.choice([2, 3, 3])
        nx, ny, nz = _box(rng, _log_uniform(rng, 576, 100_000 if d == 2 else 3_200_000), d)
        case.update(nx=nx, ny=ny, nz=nz, shift=round(rng.uniform(0.005, 0.1), 6))
    elif kind == "irregular":
        case.update(n=round(_log_uniform(rng, 20_000, 300_000)))
    elif kind in ("bicg", "spmv"):
        nx, ny, nz = _box(rng, _log_uniform(rng, 4096, 2_000_000 if kind == "bicg" else 4_000_000), 3)
        case.update(nx=nx, ny=ny, nz=nz)
    elif kind == "batch":
        case.update(count=round(_log_uniform(rng, 24, 192)))
    else:
        case.update(nx=round(_log_uniform(rng, 16, 64)), precision="mixed")
    return case


# ------------------------------------------------------------------------------------
# systems (built on the GPU; CSR arrays on the host, as the conversion takes them)
# ------------------------------------------------------------------------------------
class Csr:
    """A CSR matrix as padded rows on the GPU (for right-hand sides and exact products)."""

    def __init__(self, cols, vals, ok):
        self.cols, self.vals, self.ok = cols, torch.where(ok, vals, torch.zeros_like(vals)), ok
        self.n = cols.shape[0]

    def host(self):
        rowptr = torch.zeros(self.n + 1, dtype=torch.int64, device=self.cols.device)
        rowptr[1:] = torch.cumsum(self.ok.sum(1), 0)
        return (rowptr.int().cpu().numpy(), self.cols[self.ok].int().cpu().numpy(), self.vals[self.ok].cpu().numpy())

    def times(self, x):
        y = torch.zeros(self.n, dtype=torch.float64, device=x.device)
        for j in range(self.cols.shape[1]):
            y += self.vals[:, j] * x[self.cols[:, j]]
        return y


def _stencil(nx, ny, nz, center, lower, upper):
    """Box stencil: center, and per axis the coefficient of the lower and upper neighbour
    (numbers, or arrays over the cells)."""
    dims = [nx, ny] + ([nz] if nz else [])
    n = math.prod(dims)
    i = torch.arange(n, device=DEV)
    strides = [1, nx, nx * ny][: len(dims)]
    at = [(i // s) % d for s, d in zip(strides, dims)]
    order = [(-1, a) for a in reversed(range(len(dims)))] + [(0, 0)] + [(1, a) for a in range(len(dims))]
    cols = torch.empty(n, len(order), dtype=torch.int64, device=DEV)
    vals = torch.empty(n, len(order), dtype=torch.float64, device=DEV)
    ok = torch.empty(n, len(order), dtype=torch.bool, device=DEV)
    for j, (side, a) in enumerate(order):
        ok[:, j] = True if side == 0 else (at[a] > 0 if side < 0 else at[a] < dims[a] - 1)
        cols[:, j] = torch.where(ok[:, j], i + side * strides[a], i)
        vals[:, j] = center if side == 0 else (lower[a] if side < 0 else upper[a])
    return Csr(cols, vals, ok)


def _laplacian(nx, ny, nz, shift):
    d = 3 if nz else 2
    return _stencil(nx, ny, nz, 2.0 * d + shift, [-1.0] * d, [-1.0] * d)


def _convection_diffusion(nx, ny, nz):
    """Unit diffusion and first-order upwind convection with velocity (1, 1/2, 1/4)."""
    v = (1.0, 0.5, 0.25)
    return _stencil(nx, ny, nz, 6.0 + sum(v), [-1.0 - c for c in v], [-1.0] * 3)


def _diffusion(nx, seed):
    """-div(k grad u) with k = exp(g), g a smooth Gaussian field of unit variance; faces take
    the harmonic mean, boundary faces the cell's own k."""
    g = mf.workloads.gaussian_random_field((nx, nx, nx), 8.0, 1.0, seed)
    k = torch.as_tensor(np.exp(g).reshape(-1), device=DEV)
    i = torch.arange(nx ** 3, device=DEV)
    center, lower, upper = torch.zeros_like(k), [], []
    for s in (1, nx, nx * nx):
        for side, into in ((-1, lower), (1, upper)):
            ok = ((i // s) % nx > 0) if side < 0 else ((i // s) % nx < nx - 1)
            other = k[torch.where(ok, i + side * s, i)]
            face = torch.where(ok, 2.0 * k * other / (k + other), k)
            center += face
            into.append(-face)
    return _stencil(nx, nx, nx, center, lower, upper)


def _graph(n, seed):
    """Weighted graph Laplacian plus a twentieth of its diagonal: lognormal degrees (mean
    about 20, at most 200), neighbours uniform within 8,000 rows, a third of the weights 1."""
    gen = torch.Generator(device=DEV).manual_seed(seed)
    half = torch.exp(torch.randn(n, generator=gen, device=DEV, dtype=torch.float64) * 0.8 + 2.0)
    half = half.round().clamp(1, 100).long()
    rows = torch.repeat_interleave(torch.arange(n, device=DEV), half)
    cols = rows - torch.randint(1, 8001, (rows.numel(),), generator=gen, device=DEV)
    key = torch.unique(torch.where(cols >= 0, rows * n + cols, -torch.ones_like(rows)))
    key = key[key >= 0]
    rows, cols = key // n, key % n
    w = torch.rand(key.numel(), generator=gen, device=DEV, dtype=torch.float64) + 0.1
    w = torch.where(torch.rand(key.numel(), generator=gen, device=DEV) < 1.0 / 3.0, torch.ones_like(w), w)
    r, c, v = torch.cat([rows, cols]), torch.cat([cols, rows]), torch.cat([w, w])
    diag = torch.zeros(n, dtype=torch.float64, device=DEV).index_add_(0, r, v) * 1.05 + 1e-3
    i = torch.arange(n, device=DEV)
    r, c, v = torch.cat([r, i]), torch.cat([c, i]), torch.cat([-v, diag])
    key, order = torch.sort(r * n + c)
    r, c, v = key // n, key % n, v[order]
    rowptr = torch.zeros(n + 1, dtype=torch.int64, device=DEV)
    rowptr[1:] = torch.cumsum(torch.bincount(r, minlength=n), 0)
    return rowptr, r, c, v


def _solution(n, seed, k=0):
    gen = torch.Generator(device=DEV).manual_seed(1_000_003 * (k + 1) + seed)
    return torch.rand(n, generator=gen, device=DEV, dtype=torch.float64) * 2.0 - 1.0


def _system(case):
    """The padded matrix of a cg, bicg or spmv case (it does not depend on the seed)."""
    if case["kind"] == "cg":
        return _laplacian(case["nx"], case["ny"], case["nz"], case["shift"])
    return _convection_diffusion(case["nx"], case["ny"], case["nz"])


def _batch_systems(case, seed):
    """Shifted Laplacians of log-uniform size, 2D and 3D in turn; the shifts are the seed's."""
    sizes, rng = np.random.default_rng(case["count"]), np.random.default_rng(seed)
    for s in range(case["count"]):
        n = math.exp(sizes.uniform(math.log(1024), math.log(65536)))
        shift = float(rng.uniform(0.01, 0.1))
        if s % 2 == 0:
            nx = max(2, round(n ** 0.5))
            yield _laplacian(nx, max(2, round(n / nx)), 0, shift)
        else:
            nx = max(2, round(n ** (1.0 / 3.0)))
            yield _laplacian(nx, nx, max(2, round(n / nx ** 2)), shift)


# ------------------------------------------------------------------------------------
# prepare, run
# ------------------------------------------------------------------------------------
def prepare(case, seed):
    kind = case["kind"]
    s = dict(kind=kind, precision=case["precision"])
    if kind == "batch":
        systems = list(_batch_systems(case, seed))
        s["batch"] = mf.Batch([a.host() for a in systems])
        s["b"] = s["batch"].pack([a.times(_solution(a.n, seed, k)).cpu().numpy() for k, a in enumerate(systems)])
    elif kind == "autograd":
        fields = [_diffusion(case["nx"], seed + 500_000 * k) for k in range(2)]
        rowptr, colidx, vals = fields[0].host()
        s["op"] = mf.autograd.SparseOperator(rowptr, colidx, vals, spd=True, precision=case["precision"], tol=TOL)
        s["vals"] = [torch.as_tensor(a.host()[2], device=DEV).requires_grad_() for a in fields]
        s["b"] = [a.times(_solution(a.n, seed, k)).requires_grad_() for k, a in enumerate(fields)]
        s["g"] = [a.times(_solution(a.n, seed, 2 + k)) for k, a in enumerate(fields)]
    elif kind == "irregular":
        rowptr, r, c, v = _graph(case["n"], seed)
        s["A"] = mf.TiledMatrix(rowptr.int().cpu().numpy(), c.int().cpu().numpy(), v.cpu().numpy())
        x = _solution(case["n"], seed)
        s["b"] = torch.zeros_like(x).index_add_(0, r, v * x[c])
    else:
        a = _system(case)
        s["A"] = mf.TiledMatrix(*a.host())
        x = _solution(a.n, seed)
        s["b"] = x if kind == "spmv" else a.times(x)
    return s


def run(s):
    kind = s["kind"]
    if kind in ("cg", "irregular"):
        return s["A"].cg(s["b"], tol=TOL, precision=s["precision"])[0]
    if kind == "bicg":
        return s["A"].bicgstab(s["b"], tol=TOL, precision=s["precision"])[0]
    if kind == "spmv":
        return s["A"].spmv(s["b"], precision=s["precision"])
    if kind == "batch":
        return s["batch"].cg(s["b"], tol=TOL, precision=s["precision"])[0]
    xs = [mf.autograd.sparse_solve(v, b, s["op"]) for v, b in zip(s["vals"], s["b"])]
    grads = torch.autograd.grad(xs, s["vals"] + s["b"], s["g"])
    return [x.detach() for x in xs], list(grads)


# ------------------------------------------------------------------------------------
# exact results and necessary work
# ------------------------------------------------------------------------------------
def exact(case, seed):
    kind = case["kind"]
    if kind == "batch":
        parts = []
        for k, a in enumerate(_batch_systems(case, seed)):
            parts.append(torch.nn.functional.pad(_solution(a.n, seed, k), (0, -a.n % 16)))
        return torch.cat(parts)
    if kind == "autograd":
        xs, grad_vals, grad_b = [], [], []
        for k in range(2):
            a = _diffusion(case["nx"], seed + 500_000 * k)
            x, lam = _solution(a.n, seed, k), _solution(a.n, seed, 2 + k)
            xs.append(x)
            grad_vals.append((-lam[:, None] * x[a.cols])[a.ok])
            grad_b.append(lam)
        return xs, grad_vals + grad_b
    if kind == "spmv":
        a = _system(case)
        x = _solution(a.n, seed)
        if case["precision"] == "mixed":
            # values as stored, the binary32 copy of x, binary32 products, binary64 sums
            a.vals, x = a.vals.float(), x.float()
            y = torch.zeros(a.n, dtype=torch.float64, device=DEV)
            for j in range(a.cols.shape[1]):
                y += (a.vals[:, j] * x[a.cols[:, j]]).double()
            return y
        return a.times(x)
    n = case["n"] if kind == "irregular" else case["nx"] * case["ny"] * max(1, case["nz"])
    return _solution(n, seed)


def _box_work(nx, ny, nz, value_bytes):
    """Rows and matrix bytes (a value and a byte of index an entry) of a box stencil."""
    n = nx * ny * max(1, nz)
    entries = n * (7 if nz else 5) - 2 * (n // nx + n // ny + (n // nz if nz else 0))
    return n, entries, entries * (value_bytes + 1.0)


def _iterations(sides, shift, damp=0.5):
    """About how many CG iterations a box Laplacian takes to TOL from a random solution."""
    low = sum(4.0 * math.sin(math.pi / (2 * (d + 1))) ** 2 for d in sides) + shift
    return damp * 0.5 * math.sqrt((4.0 * len(sides) + shift) / low) * math.log(2.0 / TOL)


def work(case):
    """The matrix and 16 bytes a row (read p, write the next one) once an iteration; an
    iteration count that the size gives stands for the one that the data gives."""
    kind, mixed = case["kind"], case["precision"] == "mixed"
    if kind == "irregular":
        n, entries, its = case["n"], case["n"] * 20.0, 75.0
        return {"bytes": its * (entries * 9.0 + 16.0 * n), "flops": its * (2.0 * entries + 12.0 * n)}
    if kind == "batch":
        total = {"bytes": 0.0, "flops": 0.0}
        for s in range(case["count"]):  # the median of each octave's sizes, in turn
            n = 1024 * 64 ** ((s // 2 + 0.5) / max(1.0, case["count"] / 2.0))
            side = round(n ** (0.5 if s % 2 == 0 else 1.0 / 3.0))
            one = work(dict(kind="cg", nx=side, ny=side, nz=0 if s % 2 == 0 else side, shift=0.05,
                            precision=case["precision"]))
            total = {k: total[k] + one[k] for k in total}
        return total
    if kind == "autograd":
        nx = case["nx"]
        n, entries, matrix = _box_work(nx, nx, nx, 4.0 if mixed else 8.0)
        its = 4 * 8.0 * _iterations((nx, nx, nx), 0.0)
        return {"bytes": its * (matrix + 16.0 * n) + 2 * 24.0 * entries, "flops": its * (2.0 * entries + 12.0 * n)}
    sides = [d for d in (case["nx"], case["ny"], case["nz"]) if d]
    # unshifted diagonals and unit neighbours are held in a byte, shifted ones in eight
    small = 1.0 if not case.get("shift") else 2.0
    n, entries, matrix = _box_work(case["nx"], case["ny"], case["nz"], small if mixed else 8.0)
    if kind == "spmv":
        return {"bytes": matrix + 16.0 * n, "flops": 2.0 * entries}
    its = _iterations(sides, case.get("shift", 0.0), 0.5 if kind == "cg" else 0.3)
    per = 2.0 if kind == "bicg" else 1.0
    return {"bytes": its * per * (matrix + 16.0 * n), "flops": its * per * (2.0 * entries + 12.0 * n)}
