// One product y = A x on sliced-ELL streams (sell.h) over ranges of whole rows, as a launch of
// its own: the standalone SpMV and the products of the multi-kernel solvers.
//
// The tile-chunk SpMV adds every entry into LDS (ds_add_f64) and stays near 3 TB/s whatever
// its block size, depth and grid (3D 127 x 129 x 125 binary64: 52 to 57 us); here a lane sums
// its own row in a register and a wave's slot is independent of every other, so the kernel
// only waits for its stream (35.8 us, 4.3 TB/s of the values, a byte of index and the vectors;
// tile-mixed 63 -> 28 us).  Used where rows pad little (rows_padding); matrices with rows of
// very different lengths keep the tile chunks.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include "device_common.h"
#include "mf_internal.h"
#include "solver_internal.h"

namespace mfk {

// The tile chunks in tile order (DeviceLayout::ensure_tile_order) and their entries.
struct TileOrder {
    DevMatrix A;                // chunks: tile order
    const long long *tr_chunk;
};

// One row of A x from the tile chunks, entry by entry, in the arithmetic of kPmTiles.
template <bool MIXED>
__device__ __forceinline__ double tile_row_sum(const TileOrder &T, int row, const double *x64, const float *x32)
{
    const int bi = row / kTile;
    double s = 0.0;
    for (long long c = T.tr_chunk[bi]; c < T.tr_chunk[bi + 1]; c++) {
        const int3 h = T.A.chunks[c];
        const int cls = MIXED ? chunk_class(h) : 0;
        for (int j = 0; j <= chunk_last(h); j++) {
            const int e = h.x + j, id = T.A.eidx[e];
            if ((id >> 4) != (row & 15)) continue;
            const int col = chunk_colbase(h) + (id & 15);
            s += cls == 0 ? T.A.v64[e] * x64[col] : (double)(val_lowp(T.A, cls, e) * x32[col]);
        }
    }
    return s;
}

// Block b of 4 waves: wave slots 4 b .. 4 b + 3 (16 a range).  Consecutive blocks of one XCD
// take consecutive rows, so the x that neighbouring rows share stays in one L2.  x was
// written by earlier launches: plain loads.  The streams' zero padding multiplies x at columns
// the row may not have, so a row whose sum is not finite is summed again from its own entries
// (an infinite or NaN element of x reaches the rows that have its column, and no others).
template <int RPT, bool MIXED, bool NAR, int PM>
__global__ __launch_bounds__(256) void sell_spmv_kernel(DevSell S, const int *wg_tr, int ranges, int n,
                                                        const double *__restrict__ x64, const float *__restrict__ x32,
                                                        double *__restrict__ y, TileOrder T)
{
    const int b = logical_wg(blockIdx.x, gridDim.x);
    if (b >= 4 * ranges) return;
    const int slot = __builtin_amdgcn_readfirstlane(4 * b + (int)(threadIdx.x >> 6)), r = slot >> 4;
    const int row0 = wg_tr[r] * kTile, nrows = min(wg_tr[r + 1] * kTile, n) - row0;
    const int t = 64 * (slot & 15) + (int)(threadIdx.x & 63);
    double q[RPT];
    spmv_sell<MIXED, RPT, 1024, NAR, PM, false, false, 0>(S, slot, row0 + min(t, nrows - 1), x64, x32, q);
#pragma unroll
    for (int k = 0; k < RPT; k++) {
        if (t + 1024 * k >= nrows) continue;
        if constexpr (PM == kPmTiles)
            if (!isfinite(q[k])) q[k] = tile_row_sum<MIXED>(T, row0 + t + 1024 * k, x64, x32);
        y[row0 + t + 1024 * k] = q[k];
    }
}

}  // namespace mfk

namespace mf {

// Entries of slices of 64 consecutive rows, each row padded to its slice's longest, over the
// entries themselves.
static double rows_padding(const mf_matrix *A)
{
    const int n = A->L.n_rows;
    const int *rp = A->rowptr.data();
    int64_t pad = 0;
#pragma omp parallel for schedule(static) reduction(+ : pad)
    for (int s = 0; s < (n + 63) / 64; s++) {
        int mx = 0;
        for (int i = 64 * s; i < std::min(n, 64 * s + 64); i++) mx = std::max(mx, rp[i + 1] - rp[i]);
        pad += (int64_t)(std::min(n, 64 * s + 64) - 64 * s) * ((mx + 1) / 2 * 2);
    }
    return A->L.nnz > 0 ? (double)pad / (double)A->L.nnz : 1e30;
}

// Most padding with which the row streams still beat the tile chunks.
constexpr double kRowsPadding = 1.6;

// Streams that do not fit the device memory: the tile chunks, which are there already, from
// now on (a matrix created or given new values on the host tries the streams again).
static mf_status no_streams(DeviceLayout &L)
{
    (void)hipGetLastError();  // the refused allocation is not the next launch's error
    L.rows_regular = 0;
    return MF_SUCCESS;
}

mf_status row_streams(mf_matrix *A, unsigned need, hipStream_t s, RowStreams *out)
{
    out->ok = false;
    DeviceLayout &L = A->L;
    if (L.n_rows != L.n_cols || L.n_rows == 0 || A->rowptr.size() != (size_t)L.n_rows + 1) return MF_SUCCESS;
    // Rows per thread.  Binary64 rows fill the pipeline with one slice a wave, and more waves
    // hide more (3D 127 x 129 x 125: 35.8 / 37.8 / 43.9 us at 1 / 2 / 4 rows); of the class
    // streams a slice is a unit or two, so large matrices take four (35.5 / 27.9 / 27.8 us).
    int rpt = (need & kNeedClasses) && L.n_rows >= (1 << 19) ? 4 : 1;
    while (rpt > 1 && !sell_supported(A, rpt)) rpt /= 2;
    if (!sell_supported(A, rpt)) return MF_SUCCESS;
    if (L.rows_regular < 0) L.rows_regular = rows_padding(A) <= kRowsPadding;
    if (!L.rows_regular) return MF_SUCCESS;
    // ranges of 1024 rpt rows, kept under the key -rpt
    auto it = L.parts.find(-rpt);
    if (it == L.parts.end()) {
        Partition P;
        for (int t = 0; t < L.tilem; t += 64 * rpt) P.h_tr.push_back(t);
        P.G = (int)P.h_tr.size();
        P.h_tr.push_back(L.tilem);
        P.rows_cap = 1024 * rpt;
        const mf_status st = upload((void **)&P.wg_tr, P.h_tr.data(), sizeof(int) * P.h_tr.size(), s);
        if (st != MF_SUCCESS || hipStreamSynchronize(s) != hipSuccess) {
            free_partition(P);
            return st == MF_ERR_ALLOC ? no_streams(L) : st != MF_SUCCESS ? st : MF_ERR_HIP;
        }
        it = L.parts.emplace(-rpt, P).first;
    }
    const SellLayout *SL = nullptr;
    mf_status st = ensure_sell(A, &it->second, rpt, need, s, &out->S, &SL, false);
    if (st == MF_SUCCESS) st = L.ensure_tile_order(s);
    if (st == MF_ERR_ALLOC || st == MF_ERR_TOO_LARGE) return no_streams(L);
    if (st != MF_SUCCESS) return st;
    out->narrow = SL->narrow;
    out->L = &L;
    out->P = &it->second;
    out->rpt = rpt;
    out->ok = true;
    return MF_SUCCESS;
}

template <int RPT, bool MIXED, bool NAR, int PM>
static void launch_rows(const RowStreams &R, int n, const double *x64, const float *x32, double *y, hipStream_t s)
{
    const int blocks = (4 * R.P->G + 7) / 8 * 8;
    mfk::TileOrder T;
    T.A = R.L->dev(*R.P);
    T.A.chunks = R.L->chunks;
    T.tr_chunk = R.L->d_tr_chunk;
    hipLaunchKernelGGL((mfk::sell_spmv_kernel<RPT, MIXED, NAR, PM>), dim3(blocks), dim3(256), 0, s, R.S, R.P->wg_tr,
                       R.P->G, n, x64, x32, y, T);
}

template <int RPT>
static void launch_rows(const RowStreams &R, int n, const double *x64, const float *x32, double *y, bool mixed, int pm,
                        hipStream_t s)
{
    using namespace mfk;
    if (!mixed) return launch_rows<RPT, false, false, kPmTiles>(R, n, x64, x32, y, s);
    if (pm == kPmWide64)
        return R.narrow ? launch_rows<RPT, true, true, kPmWide64>(R, n, x64, x32, y, s)
                        : launch_rows<RPT, true, false, kPmWide64>(R, n, x64, x32, y, s);
    if (pm == kPmLow32)
        return R.narrow ? launch_rows<RPT, true, true, kPmLow32>(R, n, x64, x32, y, s)
                        : launch_rows<RPT, true, false, kPmLow32>(R, n, x64, x32, y, s);
    return R.narrow ? launch_rows<RPT, true, true, kPmTiles>(R, n, x64, x32, y, s)
                    : launch_rows<RPT, true, false, kPmTiles>(R, n, x64, x32, y, s);
}

void row_spmv(const RowStreams &R, int n, const double *x64, const float *x32, double *y, bool mixed, int pm, hipStream_t s)
{
    if (R.rpt == 1) launch_rows<1>(R, n, x64, x32, y, mixed, pm, s);
    else if (R.rpt == 2) launch_rows<2>(R, n, x64, x32, y, mixed, pm, s);
    else launch_rows<4>(R, n, x64, x32, y, mixed, pm, s);
}

}  // namespace mf
