// New values for a resident matrix from a device vector.
//
// The pattern and the tiles stay; what a change of values can move is a tile's storage class.
// One pass over the entries decides the class of every tile as the host does (tile_classes); a
// second writes the value arrays.  When no class moved the streams are filled again in place;
// when some did, the chunk headers take the new classes and the partitions and streams are
// dropped, to be built by the next solve (sell_build.hip).  The values never cross to the host.
// A 64^3 diffusion operator (1.8 million entries, row-scaled classes, a few tiles of which move
// with any new field) updates in 1.0 ms and its next solve builds its streams in 1.3, where the
// host's classes, layout and uploads took 11.5 and its streams 7.5.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include "device_common.h"
#include "mf_internal.h"
#include "solver_internal.h"

namespace mfk {

// v rounded to binary16 (nearest even, subnormals, overflow to infinity), as a double.
__device__ __forceinline__ double half_round(double v)
{
    const double a = fabs(v);
    if (!(a > 0.0)) return v;  // zeros and NaN
    if (a >= 65520.0) return copysign(INFINITY, v);
    const int q = max(ilogb(a), -14) - 10;
    return copysign(ldexp(rint(ldexp(a, -q)), q), v);
}

// Lowest class that holds v under the policy (entry_class of tile_format.cpp).
__device__ __forceinline__ int value_class(double v, int policy, double rowscale)
{
    if (policy == 2) return 0;
    if (v == floor(v) && v >= -128.0 && v <= 127.0) return 3;
    const double h = half_round(v), f = (double)(float)v;
    if (policy == 0) return h == v ? 2 : f == v ? 1 : 0;
    const double tau = 0x1p-24 * rowscale;
    if (isfinite(h) && fabs(h - v) <= tau) return 2;
    if (isfinite(f) && fabs(f - v) <= tau) return 1;
    return 0;
}

__global__ void row_scale_kernel(const int *__restrict__ rowptr, const double *__restrict__ val, int n,
                                 double *__restrict__ scale)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double s = 0.0;
    for (int j = rowptr[i]; j < rowptr[i + 1]; j++) {
        const double a = fabs(val[j]);
        s = s < a ? a : s;
    }
    scale[i] = s;
}

// 16 lanes a chunk; the group of a tile's first chunk walks the tile's chunks, writes the tile's
// class for each of them, and sets *moved when it is not the one their headers carry.
__global__ void class_check_kernel(const int3 *__restrict__ chunks, long long nchunks, const uint8_t *__restrict__ eidx,
                                   const int *__restrict__ src, const double *__restrict__ val,
                                   const double *__restrict__ scale, int policy, uint8_t *__restrict__ out, int *moved)
{
    const long long c0 = (blockIdx.x * (long long)blockDim.x + threadIdx.x) >> 4;
    if (c0 >= nchunks) return;  // whole groups
    const int k = threadIdx.x & 15;
    const int3 h0 = chunks[c0];
    if (c0 > 0) {
        const int3 hp = chunks[c0 - 1];
        if (chunk_coltile(hp) == chunk_coltile(h0) && chunk_rowbase(hp) == chunk_rowbase(h0)) return;
    }
    int cls = 3;
    int3 h = h0;
    for (long long c = c0;;) {
        if (k <= chunk_last(h)) {
            const int e = h.x + k;
            const double rs = scale ? scale[chunk_rowbase(h) + (eidx[e] >> 4)] : 0.0;
            cls = min(cls, value_class(val[src[e]], policy, rs));
        }
        if (++c >= nchunks) break;
        h = chunks[c];
        if (chunk_coltile(h) != chunk_coltile(h0) || chunk_rowbase(h) != chunk_rowbase(h0)) break;
    }
#pragma unroll
    for (int o = 8; o; o >>= 1) cls = min(cls, __shfl_xor(cls, o, 16));
    if (k != 0) return;
    if (cls != chunk_class(h0)) *moved = 1;
    for (long long c = c0; c < nchunks; c++) {
        const int3 t = chunks[c];
        if (chunk_coltile(t) != chunk_coltile(h0) || chunk_rowbase(t) != chunk_rowbase(h0)) break;
        out[c] = (uint8_t)cls;
    }
}

__global__ void set_class_kernel(int3 *__restrict__ chunks, long long nchunks, const uint8_t *__restrict__ cls)
{
    const long long c = blockIdx.x * (long long)blockDim.x + threadIdx.x;
    if (c < nchunks) chunks[c].y = (int)(((unsigned)chunks[c].y & kTileIdxMask) | ((unsigned)cls[c] << 28));
}

// The value arrays of every chunk from the CSR values (build_layout's copies).
__global__ void value_scatter_kernel(const int3 *__restrict__ chunks, long long nchunks, const int *__restrict__ src,
                                     const double *__restrict__ val, double *__restrict__ v64, float *__restrict__ v32,
                                     _Float16 *__restrict__ v16, int8_t *__restrict__ v8)
{
    const long long c = (blockIdx.x * (long long)blockDim.x + threadIdx.x) >> 4;
    if (c >= nchunks) return;
    const int3 h = chunks[c];
    const int k = threadIdx.x & 15;
    if (k > chunk_last(h)) return;
    const int e = h.x + k, cls = chunk_class(h);
    const double v = val[src[e]];
    v64[e] = v;
    if (!v32) return;
    const float f = (float)v;
    v32[e] = f;
    v16[e] = (_Float16)(float)half_round(cls == 2 ? v : (double)f);
    const double t = trunc(v);
    v8[e] = cls == 3 ? (int8_t)v : isnan(v) ? (int8_t)0 : (int8_t)(t > 127.0 ? 127 : t < -128.0 ? -128 : (int)t);
}

}  // namespace mfk

namespace mf {

mf_status host_values(mf_matrix *A, hipStream_t s)
{
    if (!A->host_stale) return MF_SUCCESS;
    if (hipMemcpyAsync(A->hval.data(), A->d_csr, sizeof(double) * A->hval.size(), hipMemcpyDeviceToHost, s) != hipSuccess ||
        hipStreamSynchronize(s) != hipSuccess)
        return MF_ERR_HIP;
    const TileStruct &ts = A->ts;
#pragma omp parallel for schedule(static)
    for (int64_t e = 0; e < ts.nnz; e++) A->L.h_ev[e] = A->hval[ts.src[e]];
    A->host_stale = false;
    return MF_SUCCESS;
}

}  // namespace mf

using namespace mf;

extern "C" mf_status mf_matrix_update_values_device(mf_matrix *A, const double *d_val, void *stream)
{
    if (!A || (!d_val && A->ts.nnz > 0)) return MF_ERR_INVALID;
    if (hipSetDevice(A->device) != hipSuccess) return MF_ERR_HIP;
    hipStream_t s = (hipStream_t)stream;
    DeviceLayout &L = A->L;
    if (A->ts.nnz == 0) return MF_SUCCESS;
    const size_t count = (size_t)A->rowptr[A->ts.rows];  // CSR positions, from 0
    mf_status st = L.ensure_tile_order(s);
    if (st != MF_SUCCESS) return st;
    // row pointer, row scales, flag and the values' device copy: kept for the next update
    const bool scaled = A->class_policy == MF_CLASS_ROWSCALED;
    if (scaled && !A->d_rowptr &&
        ((st = upload((void **)&A->d_rowptr, A->rowptr.data(), sizeof(int) * A->rowptr.size(), s)) != MF_SUCCESS ||
         (st = upload((void **)&A->d_scale, nullptr, sizeof(double) * (size_t)A->ts.rows, s)) != MF_SUCCESS))
        return st;
    if (!A->d_moved && (st = upload((void **)&A->d_moved, nullptr, sizeof(int), s)) != MF_SUCCESS) return st;
    if (!A->d_csr && (st = upload((void **)&A->d_csr, nullptr, sizeof(double) * count, s)) != MF_SUCCESS) return st;
    if (!A->d_cls && (st = upload((void **)&A->d_cls, nullptr, (size_t)L.nchunks, s)) != MF_SUCCESS) return st;
    int moved = 0;
    if (hipMemcpyAsync(A->d_moved, &moved, sizeof(int), hipMemcpyHostToDevice, s) != hipSuccess) return MF_ERR_HIP;
    if (scaled)
        hipLaunchKernelGGL(mfk::row_scale_kernel, dim3((A->ts.rows + 255) / 256), dim3(256), 0, s, A->d_rowptr, d_val,
                           A->ts.rows, A->d_scale);
    const dim3 grid((unsigned)((L.nchunks * 16 + 255) / 256)), blk(256);
    hipLaunchKernelGGL(mfk::class_check_kernel, grid, blk, 0, s, L.chunks, (long long)L.nchunks, L.eidx, L.src, d_val,
                       scaled ? A->d_scale : nullptr, A->class_policy, A->d_cls, A->d_moved);
    if (hipGetLastError() != hipSuccess ||
        hipMemcpyAsync(&moved, A->d_moved, sizeof(int), hipMemcpyDeviceToHost, s) != hipSuccess ||
        hipStreamSynchronize(s) != hipSuccess)
        return MF_ERR_HIP;
    if (moved) {
        std::vector<uint8_t> c((size_t)L.nchunks);
        if (hipMemcpyAsync(c.data(), A->d_cls, c.size(), hipMemcpyDeviceToHost, s) != hipSuccess) return MF_ERR_HIP;
        hipLaunchKernelGGL(mfk::set_class_kernel, dim3((unsigned)((L.nchunks + 255) / 256)), dim3(256), 0, s, L.chunks,
                           (long long)L.nchunks, A->d_cls);
        if (hipGetLastError() != hipSuccess || hipStreamSynchronize(s) != hipSuccess) return MF_ERR_HIP;
        for (auto &kv : L.parts) free_partition(kv.second);
        L.parts.clear();
        const TileStruct &ts = A->ts;
        int64_t at = 0;
        for (int64_t t = 0; t < ts.tiles(); t++) {
            const int64_t n = (ts.tile_off[t + 1] - ts.tile_off[t] + 15) / 16;
            A->cls[t] = c[at];
            for (int64_t k = 0; k < n; k++, at++)
                L.h_chunks[at].y = (int)(((unsigned)L.h_chunks[at].y & mfk::kTileIdxMask) | ((unsigned)c[at] << 28));
        }
        class_totals(ts, A->cls, L);
    }
    if (hipMemcpyAsync(A->d_csr, d_val, sizeof(double) * count, hipMemcpyDeviceToDevice, s) != hipSuccess) return MF_ERR_HIP;
    A->hval.resize(count);
    A->host_stale = true;
    delete A->AT;  // rebuilt from the new values on the next transposed call
    A->AT = nullptr;
    hipLaunchKernelGGL(mfk::value_scatter_kernel, grid, blk, 0, s, L.chunks, (long long)L.nchunks, L.src, d_val, L.v64,
                       L.v32, (_Float16 *)L.v16, L.v8);
    if (hipGetLastError() != hipSuccess) return MF_ERR_HIP;
    for (auto &kv : L.parts)
        if ((st = refill_sell(A, kv.second, s)) != MF_SUCCESS) return st;
    return hipStreamSynchronize(s) == hipSuccess ? MF_SUCCESS : MF_ERR_HIP;
}
