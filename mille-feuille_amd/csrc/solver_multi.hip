// Multi-kernel fallback: CG / BiCGSTAB driven by a host loop (the reference's
// cg_solve_reduce, main-cg.cu:258-292, and multi-kernel bicgstab, main-bicg.cu:1619-1656).
// No co-residency requirement, so it runs any size.  Scalars live on the device; dot
// products are deterministic two-pass sums.
//
// CG is two launches an iteration, the recurrence of the persistent kernels' variant 4:
//   mk_cg_spmv    q = A p and each workgroup's part of {p'q, r'q, q'q, r'r}
//   mk_cg_update  every workgroup sums the parts, decides alike (convergence, replacement,
//                 breakdown), and updates x, r and p in one pass
// The host enqueues kBatch iterations at a time and reads the state once per batch; after a
// decision the remaining launches of a batch do nothing.  An iteration reads the matrix, 24
// bytes a row in the product and 32 in the update, and writes 8 and 24 (28 tile-mixed); it
// took 11 launches, 155 bytes a row and two host synchronisations before (3D 144 x 145 x 147
// tile-mixed: 204 us, of which the SpMV on tile chunks 80).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <vector>

#include "device_common.h"
#include "launch_common.h"
#include "mf_internal.h"
#include "solver_internal.h"

namespace mfk {

constexpr int kDotBlocks = 512;

// State of a multi-kernel CG, in the solve's 32 scalars.
enum { MKS_RR = 0, MKS_IT = 1, MKS_STATE = 2 };
enum { MK_RUN = 0, MK_CHECK = 1, MK_BREAK = 2, MK_MAXIT = 3 };

// PM: product mode of the tile-mixed SpMV (sell.h): kPmLow32 for CG, kPmWide64 for
// BiCGSTAB, as in the persistent kernels.  sc: the state of the CG whose batch of iterations
// the product belongs to (nothing is done once it is decided), or null.
template <bool MIXED, int PM>
__global__ __launch_bounds__(1024) void mk_spmv(DevMatrix A, const double *__restrict__ x64,
                                                const float *__restrict__ x32, double *__restrict__ y,
                                                const double *sc)
{
    if (sc && sc[MKS_STATE] != (double)MK_RUN) return;
    extern __shared__ double q[];
    __shared__ double qdummy[64];
    const int w = blockIdx.x;
    const int tr0 = A.wg_tr[w], tr1 = A.wg_tr[w + 1];
    const int row0 = tr0 * kTile, row1 = min(tr1 * kTile, A.n);
    for (int i = threadIdx.x; i < row1 - row0; i += blockDim.x) q[i] = 0.0;
    __syncthreads();
    spmv_chunks<MIXED, 2, false, PM>(A, A.wg_chunk + 4 * (size_t)w, row0, x64, x32, q, qdummy);
    __syncthreads();
    for (int i = threadIdx.x; i < row1 - row0; i += blockDim.x) y[row0 + i] = q[i];
}

// partial[blockIdx] = sum over the block's grid-stride slice of a[i]*b[i]
__global__ __launch_bounds__(256) void mk_dot(const double *__restrict__ a, const double *__restrict__ b, int n,
                                              double *__restrict__ partial)
{
    __shared__ double s[4];
    double v = 0.0;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) v += a[i] * b[i];
    v = wave_sum(v);
    if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) partial[blockIdx.x] = s[0] + s[1] + s[2] + s[3];
}

__global__ __launch_bounds__(256) void mk_finish(const double *__restrict__ partial, int nb, double *out)
{
    __shared__ double s[4];
    double v = 0.0;
    for (int i = threadIdx.x; i < nb; i += blockDim.x) v += partial[i];
    v = wave_sum(v);
    if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) *out = s[0] + s[1] + s[2] + s[3];
}

constexpr int kUpdBlocks = 512, kUpdThreads = 512;

// q = A p over row streams, range blockIdx.x, + gridDim.x, ...; part[4 b ..] = this
// workgroup's {p'q, r'q, q'q, r'r}.
template <int RPT, bool MIXED, bool NAR>
__global__ __launch_bounds__(1024) void mk_cg_spmv(DevSell S, const int *wg_tr, int ranges, int n,
                                                   const double *__restrict__ p, const float *__restrict__ p32,
                                                   const double *__restrict__ r, double *__restrict__ q,
                                                   double *__restrict__ part, const double *sc)
{
    __shared__ double scratch[64];
    if (sc[MKS_STATE] != (double)MK_RUN) return;
    double d[4] = {0.0, 0.0, 0.0, 0.0};
    const int b = logical_wg(blockIdx.x, gridDim.x);
    // a workgroup's ranges are neighbours
    const int r_lo = (int)((long long)ranges * b / gridDim.x), r_hi = (int)((long long)ranges * (b + 1) / gridDim.x);
    for (int g = r_lo; g < r_hi; g++) {
        const int slot = __builtin_amdgcn_readfirstlane(g * 16 + (int)(threadIdx.x >> 6));
        const int row0 = wg_tr[g] * kTile, nrows = min(wg_tr[g + 1] * kTile, n) - row0;
        const int t = threadIdx.x;
        double qv[RPT];
        spmv_sell<MIXED, RPT, 1024, NAR, MIXED ? kPmLow32 : kPmTiles, false, false, 0>(
            S, slot, row0 + min(t, nrows - 1), p, p32, qv);
#pragma unroll
        for (int k = 0; k < RPT; k++) {
            const int row = row0 + t + 1024 * k;
            if (t + 1024 * k >= nrows) continue;
            const double pk = p[row], rk = r[row], qk = qv[k];
            q[row] = qk;
            d[0] += pk * qk;
            d[1] += rk * qk;
            d[2] += qk * qk;
            d[3] += rk * rk;
        }
    }
    block_sum<4>(d, scratch);
    if (threadIdx.x < 4) part[4 * (size_t)b + threadIdx.x] = threadIdx.x == 0 ? d[0] : threadIdx.x == 1 ? d[1]
                                                                             : threadIdx.x == 2 ? d[2] : d[3];
}

// The same sums for a product made by the tile-chunk SpMV.
__global__ __launch_bounds__(1024) void mk_cg_dots(int n, const double *__restrict__ p, const double *__restrict__ r,
                                                   const double *__restrict__ q, double *__restrict__ part,
                                                   const double *sc)
{
    __shared__ double scratch[64];
    if (sc[MKS_STATE] != (double)MK_RUN) return;
    double d[4] = {0.0, 0.0, 0.0, 0.0};
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const double pk = p[i], rk = r[i], qk = q[i];
        d[0] += pk * qk;
        d[1] += rk * qk;
        d[2] += qk * qk;
        d[3] += rk * rk;
    }
    block_sum<4>(d, scratch);
    if (threadIdx.x < 4) part[4 * (size_t)blockIdx.x + threadIdx.x] = threadIdx.x == 0 ? d[0] : threadIdx.x == 1 ? d[1]
                                                                                      : threadIdx.x == 2 ? d[2] : d[3];
}

// Iteration `it`: the tests of the recurrence on the exact r'r, then x += alpha p,
// r -= alpha q, p = r + beta p.  check2: r'r at or below which the host has to look (it
// converged, or a tile-mixed residual is due for replacement); negative: never.  Block 0
// records the state, which the launches after this one read.
__global__ __launch_bounds__(kUpdThreads) void mk_cg_update(int n, int nparts, const double *__restrict__ part, double check2,
                                                            int it, int maxit, double *__restrict__ x,
                                                            double *__restrict__ r, double *__restrict__ p,
                                                            float *__restrict__ p32, const double *__restrict__ q,
                                                            double *sc)
{
    __shared__ double scratch[64];
    if (sc[MKS_STATE] != (double)MK_RUN) return;
    double d[4] = {0.0, 0.0, 0.0, 0.0};
    for (int i = threadIdx.x; i < nparts; i += kUpdThreads) {
        const double2 a = reinterpret_cast<const double2 *>(part)[2 * i], b = reinterpret_cast<const double2 *>(part)[2 * i + 1];
        d[0] += a.x;
        d[1] += a.y;
        d[2] += b.x;
        d[3] += b.y;
    }
    block_sum<4>(d, scratch);
    const double rr = d[3];
    const int state = rr <= check2 ? MK_CHECK : it >= maxit ? MK_MAXIT : (!(d[0] != 0.0) || !isfinite(d[0])) ? MK_BREAK : MK_RUN;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        sc[MKS_RR] = rr;
        sc[MKS_IT] = (double)it;
        if (state != MK_RUN) sc[MKS_STATE] = (double)state;
    }
    if (state != MK_RUN) return;
    const double alpha = rr / d[0];
    double rr_new = rr - 2.0 * alpha * d[1] + alpha * alpha * d[2];
    if (!(rr_new > 0.0)) rr_new = 0.0;
    const double beta = rr_new / rr;
    const int step = 2 * gridDim.x * kUpdThreads;
    for (int i = 2 * (blockIdx.x * kUpdThreads + threadIdx.x); i + 1 < n; i += step) {
        double2 xv = *reinterpret_cast<double2 *>(x + i), rv = *reinterpret_cast<double2 *>(r + i);
        double2 pv = *reinterpret_cast<double2 *>(p + i);
        const double2 qv = *reinterpret_cast<const double2 *>(q + i);
        xv.x += alpha * pv.x;
        xv.y += alpha * pv.y;
        rv.x -= alpha * qv.x;
        rv.y -= alpha * qv.y;
        pv.x = rv.x + beta * pv.x;
        pv.y = rv.y + beta * pv.y;
        *reinterpret_cast<double2 *>(x + i) = xv;
        *reinterpret_cast<double2 *>(r + i) = rv;
        *reinterpret_cast<double2 *>(p + i) = pv;
        if (p32) *reinterpret_cast<float2 *>(p32 + i) = make_float2((float)pv.x, (float)pv.y);
    }
    if ((n & 1) && blockIdx.x == 0 && threadIdx.x == 0) {
        const int i = n - 1;
        x[i] += alpha * p[i];
        r[i] -= alpha * q[i];
        p[i] = r[i] + beta * p[i];
        if (p32) p32[i] = (float)p[i];
    }
}

// Whether every scalar slot named in `mask` (bit k: sc[k]) is finite and nonzero.  The
// vector updates of an iteration do nothing when a denominator broke down, so the
// iterate the host finds on MF_BREAKDOWN is the last finite one.
__device__ __forceinline__ bool mk_ok(const double *sc, unsigned mask)
{
    for (int k = 0; k < 8; k++)
        if ((mask >> k) & 1u) {
            const double d = sc[k];
            if (!(d != 0.0) || !isfinite(d)) return false;
        }
    return true;
}

__global__ void mk_copy(const double *__restrict__ a, double *__restrict__ b, float *__restrict__ b32, int n)
{
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        b[i] = a[i];
        if (b32) b32[i] = (float)a[i];
    }
}

// r = b - q; optional p += (r_new - r_old)
// (q and r may alias: each element is read before it is written)
__global__ void mk_residual(const double *b, const double *q, double *r, double *p, float *p32, int n)
{
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const double rn = b[i] - q[i];
        if (p) {
            const double pn = p[i] + (rn - r[i]);
            p[i] = pn;
            if (p32) p32[i] = (float)pn;
        }
        r[i] = rn;
    }
}

// BiCGSTAB steps.  sc: [0] rho [1] rhat'v [2] t's [3] t't [4] rho' [5] r'r [6] b'b
__global__ void mk_bicg_s(const double *__restrict__ sc, const double *__restrict__ r, const double *__restrict__ v,
                          double *__restrict__ s, float *__restrict__ s32, int n)
{
    if (!mk_ok(sc, 1u << 1)) return;
    const double alpha = sc[0] / sc[1];
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const double sv = r[i] - alpha * v[i];
        s[i] = sv;
        if (s32) s32[i] = (float)sv;
    }
}

__global__ void mk_bicg_xr(const double *__restrict__ sc, double *__restrict__ x, double *__restrict__ r,
                           const double *__restrict__ p, const double *__restrict__ s, const double *__restrict__ t,
                           int n)
{
    if (!mk_ok(sc, (1u << 1) | (1u << 3))) return;
    const double alpha = sc[0] / sc[1], omega = sc[2] / sc[3];
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        x[i] += alpha * p[i] + omega * s[i];
        r[i] = s[i] - omega * t[i];
    }
}

__global__ void mk_bicg_p(double *__restrict__ sc, double *__restrict__ p, float *__restrict__ p32,
                          const double *__restrict__ r, const double *__restrict__ v, int n)
{
    if (!mk_ok(sc, (1u << 0) | (1u << 1) | (1u << 2) | (1u << 3))) return;
    const double alpha = sc[0] / sc[1], omega = sc[2] / sc[3];
    const double beta = (sc[4] / sc[0]) * (alpha / omega);
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const double pv = r[i] + beta * (p[i] - omega * v[i]);
        p[i] = pv;
        if (p32) p32[i] = (float)pv;
    }
}

__global__ void mk_set(double *sc, int dst, int src) { sc[dst] = sc[src]; }

}  // namespace mfk

namespace mf {

namespace {

struct MkCtx {
    mf_matrix *A;
    hipStream_t s;
    const Partition *P;
    mfk::DevMatrix dm;
    int G;
    size_t lds;
    bool mixed;
    int n;
    double *partial = nullptr;
    double *sc = nullptr;
    RowStreams rows;   // the products' streams, when the matrix suits them (else tile chunks)
    std::vector<void *> bufs;

    ~MkCtx()
    {
        for (void *p : bufs) free_dev(p);
    }
    template <class T>
    T *alloc(size_t count)
    {
        void *p = nullptr;
        if (hipMalloc(&p, std::max<size_t>(count, 1) * sizeof(T)) != hipSuccess) return nullptr;
        bufs.push_back(p);
        return (T *)p;
    }
    // use_mixed: tile classes with product mode pm (kPmLow32 CG, kPmWide64 BiCGSTAB); state:
    // mk_spmv's sc
    void spmv(const double *x64, const float *x32, double *y, bool use_mixed, int pm = mfk::kPmLow32,
              const double *state = nullptr)
    {
        if (rows.ok)
            row_spmv(rows, n, x64, x32, y, use_mixed, pm, s);
        else if (use_mixed && pm == mfk::kPmWide64)
            hipLaunchKernelGGL((mfk::mk_spmv<true, mfk::kPmWide64>), dim3(G), dim3(1024), lds, s, dm, x64, x32, y, state);
        else if (use_mixed)
            hipLaunchKernelGGL((mfk::mk_spmv<true, mfk::kPmLow32>), dim3(G), dim3(1024), lds, s, dm, x64, x32, y, state);
        else
            hipLaunchKernelGGL((mfk::mk_spmv<false, mfk::kPmTiles>), dim3(G), dim3(1024), lds, s, dm, x64, x32, y, state);
    }
    void dot(const double *a, const double *b, int slot)
    {
        hipLaunchKernelGGL(mfk::mk_dot, dim3(mfk::kDotBlocks), dim3(256), 0, s, a, b, n, partial);
        hipLaunchKernelGGL(mfk::mk_finish, dim3(1), dim3(256), 0, s, partial, mfk::kDotBlocks, sc + slot);
    }
    double read(int slot)
    {
        double v = 0;
        (void)hipMemcpyAsync(&v, sc + slot, sizeof(double), hipMemcpyDeviceToHost, s);
        (void)hipStreamSynchronize(s);
        return v;
    }
    dim3 vgrid() const { return dim3(std::min(2048, std::max(1, (n + 255) / 256))); }
};

mf_status mk_setup(mf_matrix *A, const mf_solve_options *o, hipStream_t s, MkCtx &c)
{
    c.A = A;
    c.s = s;
    c.n = A->L.n_rows;
    c.mixed = o->precision == MF_PREC_MIXED && A->L.has_lowp;
    if (A->L.tilem == 0 || A->L.n_rows != A->L.n_cols) return MF_ERR_INVALID;
    if (o->layout != 1) {  // 1: the caller asked for the tile chunks
        const mf_status rst = row_streams(A, sell_need(c.mixed), s, &c.rows);
        if (rst != MF_SUCCESS) return rst;
    }
    c.partial = c.alloc<double>(mfk::kDotBlocks);
    c.sc = c.alloc<double>(32);
    if (!c.partial || !c.sc) return MF_ERR_ALLOC;
    if (c.rows.ok) {
        c.G = c.rows.P->G;
        return MF_SUCCESS;
    }
    // at most 4096 rows (32 KB of LDS) per workgroup; any number of workgroups
    int G = std::max(1, std::min(A->L.tilem, std::max(A->num_cus, (A->L.n_rows + 4095) / 4096)));
    mf_status st;
    for (;;) {
        if ((st = A->L.partition(G, s, &c.P)) != MF_SUCCESS) return st;
        if (c.P->rows_cap <= 4096 || G >= A->L.tilem) break;
        G = std::min(A->L.tilem, G * 2);
    }
    c.G = G;
    c.dm = A->L.dev(*c.P);
    c.lds = (size_t)std::max(c.P->rows_cap, 1) * 8;
    if (c.lds > (size_t)A->max_lds) return MF_ERR_TOO_LARGE;
    for (auto k : {(const void *)mfk::mk_spmv<true, mfk::kPmLow32>, (const void *)mfk::mk_spmv<true, mfk::kPmWide64>,
                   (const void *)mfk::mk_spmv<false, mfk::kPmTiles>})
        (void)hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)c.lds);
    return MF_SUCCESS;
}

void fill_info(mf_solve_info *info, const MkCtx &c, int status, int it, int repl, double rr, double bb,
               double rt, double ms, double bytes)
{
    if (!info) return;
    memset(info, 0, sizeof(*info));
    info->status = status;
    info->iterations = it;
    info->replacements = repl;
    info->grid = c.G;
    info->block = 1024;
    info->layout = c.rows.ok ? (c.mixed && c.rows.narrow ? 3 : 2) : 1;
    info->precision = c.mixed ? MF_PREC_MIXED : MF_PREC_FP64;
    info->relres = bb > 0 ? std::sqrt(std::max(rr, 0.0) / bb) : 0.0;
    info->relres_true = bb > 0 ? std::sqrt(std::max(rt, 0.0) / bb) : std::sqrt(std::max(rt, 0.0));
    info->time_ms = ms;
    info->bytes_per_iter = bytes;
    info->gbs = ms > 0 ? bytes * it / (ms * 1e-3) / 1e9 : 0.0;
}

}  // namespace

// One product of the iteration with its partial sums; returns the number of parts.
static int mk_cg_product(MkCtx &c, const double *p, const float *p32, const double *r, double *q, double *part)
{
    if (!c.rows.ok) {
        c.spmv(p, p32, q, c.mixed, mfk::kPmLow32, c.sc);
        hipLaunchKernelGGL(mfk::mk_cg_dots, dim3(mfk::kDotBlocks), dim3(1024), 0, c.s, c.n, p, r, q, part, c.sc);
        return mfk::kDotBlocks;
    }
    const RowStreams &R = c.rows;
    // one range a workgroup while their parts stay few: a workgroup that loops over two holds its
    // place while others have left (750 ranges, 512 workgroups 28.5 ms a solve, 750 26.9)
    const int ranges = R.P->G, G = std::min(ranges, 4 * c.A->num_cus);
    auto go = [&](auto k) {
        hipLaunchKernelGGL(k, dim3(G), dim3(1024), 0, c.s, R.S, R.P->wg_tr, ranges, c.n, p, p32, r, q, part, c.sc);
    };
    if (!c.mixed) go(R.rpt == 4 ? mfk::mk_cg_spmv<4, false, false> : R.rpt == 2 ? mfk::mk_cg_spmv<2, false, false>
                                                                                : mfk::mk_cg_spmv<1, false, false>);
    else if (R.narrow) go(R.rpt == 4 ? mfk::mk_cg_spmv<4, true, true> : R.rpt == 2 ? mfk::mk_cg_spmv<2, true, true>
                                                                                   : mfk::mk_cg_spmv<1, true, true>);
    else go(R.rpt == 4 ? mfk::mk_cg_spmv<4, true, false> : R.rpt == 2 ? mfk::mk_cg_spmv<2, true, false>
                                                                      : mfk::mk_cg_spmv<1, true, false>);
    return G;
}

mf_status cg_multikernel(mf_matrix *A, const double *b, double *x, const mf_solve_options *o, mf_solve_info *info,
                         hipStream_t s)
{
    MkCtx c;
    mf_status st = mk_setup(A, o, s, c);
    if (st != MF_SUCCESS) return st;
    const int n = c.n;
    // vectors from the matrix's workspace, kept from one solve to the next
    if ((st = A->ws.ensure(n, 1, s)) != MF_SUCCESS) return st;
    double *r = A->ws.v64, *p = A->ws.p64, *q = A->ws.s64;
    float *p32 = c.mixed ? A->ws.p32 : nullptr;
    double *part = c.alloc<double>(4 * (size_t)std::max(mfk::kDotBlocks, 4 * A->num_cus));
    if (!part) return MF_ERR_ALLOC;
    const dim3 vg = c.vgrid();
    auto t0 = std::chrono::steady_clock::now();
    // sc: [0] r'r [1] iteration [2] state [3] b'b [4] sums of the host's steps
    if (hipMemsetAsync(c.sc, 0, sizeof(double) * 32, s) != hipSuccess) return MF_ERR_HIP;
    if (o->use_x0) {
        c.spmv(x, nullptr, q, false);
        hipLaunchKernelGGL(mfk::mk_residual, vg, dim3(256), 0, s, b, q, r, (double *)nullptr, (float *)nullptr, n);
    } else {
        (void)hipMemsetAsync(x, 0, sizeof(double) * n, s);
        hipLaunchKernelGGL(mfk::mk_copy, vg, dim3(256), 0, s, b, r, (float *)nullptr, n);
    }
    hipLaunchKernelGGL(mfk::mk_copy, vg, dim3(256), 0, s, r, p, p32, n);
    c.dot(r, r, mfk::MKS_RR);
    c.dot(b, b, 3);
    const double bb = c.read(3);
    double rr = c.read(mfk::MKS_RR), rbase = rr;
    int it = 0, repl = 0, status = MF_NOT_CONVERGED;
    const double tol2 = o->tol * o->tol, dl = o->replace_delta > 0 ? o->replace_delta : 1e-3;
    const int max_repl = o->max_replacements > 0 ? o->max_replacements : 64;
    if (bb == 0.0) status = MF_SUCCESS;
    constexpr int kBatch = 16;
    bool rr_of_r = true;  // rr is r'r of the present r (at the start, after a replacement)
    while (status == MF_NOT_CONVERGED) {
        // r'r at or below which the host decides; a tile-mixed solve also looks before the
        // strict bound dl^2 rbase of a replacement, and at exactly that value goes on
        const bool may_replace = c.mixed && repl < max_repl;
        const double below = std::nextafter(dl * dl * rbase, 0.0);
        const double check2 = o->fixed_iterations ? -1.0 : may_replace ? std::max(tol2 * bb, below) : tol2 * bb;
        int state = mfk::MK_RUN;
        if (rr_of_r) state = rr <= check2 ? mfk::MK_CHECK : it >= o->max_iter ? mfk::MK_MAXIT : mfk::MK_RUN;
        if (state == mfk::MK_RUN) {
            int last = it;
            for (int i = 0; i < kBatch && last <= o->max_iter; i++, last++) {
                const int parts = mk_cg_product(c, p, p32, r, q, part);
                hipLaunchKernelGGL(mfk::mk_cg_update, dim3(mfk::kUpdBlocks), dim3(mfk::kUpdThreads), 0, s, n, parts,
                                   part, check2, last, o->max_iter, x, r, p, p32, q, c.sc);
            }
            double h[3];
            if (hipMemcpyAsync(h, c.sc, sizeof(h), hipMemcpyDeviceToHost, s) != hipSuccess ||
                hipStreamSynchronize(s) != hipSuccess)
                return MF_ERR_HIP;
            rr = h[mfk::MKS_RR];
            rr_of_r = false;
            state = (int)h[mfk::MKS_STATE];
            if (state == mfk::MK_RUN) {
                it = last;
                continue;
            }
            it = (int)h[mfk::MKS_IT];
        }
        if (state == mfk::MK_BREAK) {
            status = MF_BREAKDOWN;
        } else if (state == mfk::MK_MAXIT) {
            status = o->fixed_iterations ? MF_SUCCESS : MF_NOT_CONVERGED;
            break;
        } else if (!may_replace) {
            status = MF_SUCCESS;
        } else {
            // r = b - A x in binary64, p corrected alike; the iteration is then redone
            c.spmv(x, nullptr, q, false);
            hipLaunchKernelGGL(mfk::mk_residual, vg, dim3(256), 0, s, b, q, r, p, p32, n);
            c.dot(r, r, 4);
            rr = rbase = c.read(4);
            rr_of_r = true;
            repl++;
            if (rr <= tol2 * bb) status = MF_SUCCESS;
            else if (hipMemsetAsync(c.sc + mfk::MKS_STATE, 0, sizeof(double), s) != hipSuccess) return MF_ERR_HIP;
        }
    }
    // true residual
    c.spmv(x, nullptr, q, false);
    hipLaunchKernelGGL(mfk::mk_residual, vg, dim3(256), 0, s, b, q, q, (double *)nullptr, (float *)nullptr, n);
    c.dot(q, q, 4);
    const double rt = c.read(4);
    if (hipStreamSynchronize(s) != hipSuccess) return MF_ERR_HIP;
    const double ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    const double M = c.mixed ? A->L.alg_bytes_mixed : A->L.alg_bytes_f64;
    fill_info(info, c, status, it, repl, rr, bb, rt, ms, M + 16.0 * n);
    return (mf_status)status;
}

mf_status bicg_multikernel(mf_matrix *A, const double *b, double *x, const mf_solve_options *o,
                           mf_solve_info *info, hipStream_t s)
{
    MkCtx c;
    mf_status st = mk_setup(A, o, s, c);
    if (st != MF_SUCCESS) return st;
    const int n = c.n;
    double *r = c.alloc<double>(n), *rh = c.alloc<double>(n), *p = c.alloc<double>(n), *v = c.alloc<double>(n);
    double *sv = c.alloc<double>(n), *t = c.alloc<double>(n);
    float *p32 = c.mixed ? c.alloc<float>(n) : nullptr, *s32 = c.mixed ? c.alloc<float>(n) : nullptr;
    if (!r || !rh || !p || !v || !sv || !t || (c.mixed && (!p32 || !s32))) return MF_ERR_ALLOC;
    const dim3 vg = c.vgrid();
    auto t0 = std::chrono::steady_clock::now();
    if (o->use_x0) {
        c.spmv(x, nullptr, t, false);
        hipLaunchKernelGGL(mfk::mk_residual, vg, dim3(256), 0, s, b, t, r, (double *)nullptr, (float *)nullptr, n);
    } else {
        (void)hipMemsetAsync(x, 0, sizeof(double) * n, s);
        hipLaunchKernelGGL(mfk::mk_copy, vg, dim3(256), 0, s, b, r, (float *)nullptr, n);
    }
    hipLaunchKernelGGL(mfk::mk_copy, vg, dim3(256), 0, s, r, rh, (float *)nullptr, n);
    hipLaunchKernelGGL(mfk::mk_copy, vg, dim3(256), 0, s, r, p, p32, n);
    c.dot(rh, r, 0);
    c.dot(r, r, 5);
    c.dot(b, b, 6);
    const double bb = c.read(6);
    double rr = c.read(5), rbase = rr;
    int it = 0, repl = 0, status = MF_NOT_CONVERGED;
    const double tol2 = o->tol * o->tol, dl = o->replace_delta > 0 ? o->replace_delta : 1e-3;
    const int max_repl = o->max_replacements > 0 ? o->max_replacements : 64;
    if (bb == 0.0) status = MF_SUCCESS;
    while (status == MF_NOT_CONVERGED) {
        if (!o->fixed_iterations) {
            bool conv = rr <= tol2 * bb;
            if (c.mixed && repl < max_repl && (conv || rr < dl * dl * rbase)) {
                c.spmv(x, nullptr, t, false);
                hipLaunchKernelGGL(mfk::mk_residual, vg, dim3(256), 0, s, b, t, r, (double *)nullptr,
                                   (float *)nullptr, n);
                c.dot(r, r, 5);
                c.dot(rh, r, 0);
                rr = rbase = c.read(5);
                repl++;
                conv = rr <= tol2 * bb;
            }
            if (conv) {
                status = MF_SUCCESS;
                break;
            }
        }
        if (it >= o->max_iter) {
            status = o->fixed_iterations ? MF_SUCCESS : MF_NOT_CONVERGED;
            break;
        }
        c.spmv(p, p32, v, c.mixed, mfk::kPmWide64);
        c.dot(rh, v, 1);
        hipLaunchKernelGGL(mfk::mk_bicg_s, vg, dim3(256), 0, s, c.sc, r, v, sv, s32, n);
        c.spmv(sv, s32, t, c.mixed, mfk::kPmWide64);
        c.dot(t, sv, 2);
        c.dot(t, t, 3);
        hipLaunchKernelGGL(mfk::mk_bicg_xr, vg, dim3(256), 0, s, c.sc, x, r, p, sv, t, n);
        c.dot(rh, r, 4);
        c.dot(r, r, 5);
        hipLaunchKernelGGL(mfk::mk_bicg_p, vg, dim3(256), 0, s, c.sc, p, p32, r, v, n);
        hipLaunchKernelGGL(mfk::mk_set, dim3(1), dim3(1), 0, s, c.sc, 0, 4);
        double h[6];
        (void)hipMemcpyAsync(h, c.sc, sizeof(h), hipMemcpyDeviceToHost, s);
        (void)hipStreamSynchronize(s);
        it++;
        if (!(h[1] != 0.0) || !(h[3] != 0.0) || !(h[2] != 0.0) || !std::isfinite(h[4])) {
            status = MF_BREAKDOWN;
            break;
        }
        rr = h[5];
    }
    c.spmv(x, nullptr, t, false);
    hipLaunchKernelGGL(mfk::mk_residual, vg, dim3(256), 0, s, b, t, t, (double *)nullptr, (float *)nullptr, n);
    c.dot(t, t, 7);
    const double rt = c.read(7);
    const double ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    const double M = c.mixed ? A->L.alg_bytes_mixed : A->L.alg_bytes_f64;
    fill_info(info, c, status, it, repl, rr, bb, rt, ms, 2.0 * M + 32.0 * n);
    return (mf_status)status;
}

}  // namespace mf

using namespace mf;

extern "C" mf_status mf_cg_solve_multikernel(mf_matrix *A, const double *d_b, double *d_x,
                                             const mf_solve_options *opt, mf_solve_info *info, void *stream)
{
    if (!A || !d_b || !d_x || !aligned16(d_b) || !aligned16(d_x)) return MF_ERR_INVALID;
    if (hipSetDevice(A->device) != hipSuccess) return MF_ERR_HIP;
    mf_solve_options o;
    mf_solve_options_default(&o);
    if (opt) o = *opt;
    if (o.dynamic_precision) return MF_ERR_UNSUPPORTED;  // single-kernel CG only
    if (o.transpose) {
        mf_status st = transposed(A, (hipStream_t)stream, &A);
        if (st != MF_SUCCESS) return st;
        o.transpose = 0;
    }
    return cg_multikernel(A, d_b, d_x, &o, info, (hipStream_t)stream);
}

extern "C" mf_status mf_bicgstab_solve_multikernel(mf_matrix *A, const double *d_b, double *d_x,
                                                   const mf_solve_options *opt, mf_solve_info *info, void *stream)
{
    if (!A || !d_b || !d_x || !aligned16(d_b) || !aligned16(d_x)) return MF_ERR_INVALID;
    if (hipSetDevice(A->device) != hipSuccess) return MF_ERR_HIP;
    mf_solve_options o;
    mf_solve_options_default(&o);
    if (opt) o = *opt;
    if (o.dynamic_precision) return MF_ERR_UNSUPPORTED;  // single-kernel CG only
    if (o.transpose) {
        mf_status st = transposed(A, (hipStream_t)stream, &A);
        if (st != MF_SUCCESS) return st;
        o.transpose = 0;
    }
    return bicg_multikernel(A, d_b, d_x, &o, info, (hipStream_t)stream);
}
