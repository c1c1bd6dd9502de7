// Sliced-ELL streams (sell.h) built on the GPU from the tile chunks, for ranges whose rows
// keep their order.
//
// A slot (range, wave, slice) holds 64 consecutive rows starting at a multiple of 16: four
// whole tile rows.  One wave builds one slot.  Its four groups of 16 lanes walk the chunks of
// the four tile rows side by side, one entry a lane, in tile order (column tiles ascending,
// row-major inside a tile), so the entries of a row come in the order the streams store them
// and no row index of the matrix is needed.  Two passes per stream:
//   count  the slot's longest row, its relative columns (col - row) as a bitmap in LDS, their
//          number, and whether every row lists them ascending; the host turns these into
//          units, offsets and the choice between the plain and the shared layout;
//   fill   the padding, then every entry at its place: its position in the row (plain), or
//          its column's rank among the slot's relative columns (shared: the bitmap again,
//          with prefix counts).
// The streams are those of the host builder (build_sell), which keeps the ranges whose rows
// are sorted by length.  The passes read the chunks from the L2 or HBM once or twice and
// write the streams; for 3D Poisson 128^3 (a 134 MB binary64 and a 17 MB int8 stream) the
// first tile-mixed solve on a new matrix takes 16 ms where the host builder, its zero fills
// and its uploads made it 83.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <vector>

#include "device_common.h"
#include "mf_internal.h"
#include "solver_internal.h"

namespace mfk {

struct SellBuildArgs {
    const int3 *chunks;          // headers in tile order
    const long long *tr_chunk;   // tilem + 1
    const int *wg_tr;            // R + 1 tile-row cut points
    const uint8_t *eidx;
    const double *v64;
    const float *v32;
    const uint16_t *v16;
    const int8_t *v8;
    int n, rpt, max_off, words;  // words: of the bitmap, covers [-max_off, max_off]
    long long slots;
};

// Per (stream, slot): longest row, relative columns (INT_MAX: some row is not ascending),
// smallest and largest relative column and column.
struct SellSlot {
    int len, cols, rmin, rmax, cmin, cmax;
};

constexpr int kBuildWords = 2048;    // bitmap of 65,536 relative columns
constexpr int kBuildUnion = 1024;    // most relative columns of a shared slice

struct SlotRows {
    int r0, nr, l0, v, k;  // range's first row and rows; slot's first local row, wave, slice
};
__device__ __forceinline__ SlotRows slot_rows(const SellBuildArgs &a, long long slot)
{
    SlotRows s;
    s.k = (int)(slot % a.rpt);
    s.v = (int)(slot / a.rpt % 16);
    const int r = (int)(slot / a.rpt / 16);
    s.r0 = a.wg_tr[r] * kTile;
    s.nr = max(0, min(a.wg_tr[r + 1] * kTile, a.n) - s.r0);
    s.l0 = 1024 * s.k + 64 * s.v;
    return s;
}

// Walks the slot's entries of stream S (classes 0..3, or 4: every entry).  For each entry, in
// row order: f(lane's row 0..63, position in the row, relative column, column, position in
// the entry arrays, whether it is the row's first of the step, its predecessor's column).
// cnt and last: 64 ints of LDS each.
template <class F>
__device__ __forceinline__ void walk_slot(const SellBuildArgs &a, const SlotRows &s, int S, int *cnt, int *last, F f)
{
    const int lane = threadIdx.x, g = lane >> 4, i16 = lane & 15;
    cnt[lane] = 0;
    last[lane] = INT_MIN;
    __syncthreads();
    const int bi = (s.r0 + s.l0) / kTile + g;
    const bool in = s.l0 + 16 * g < s.nr;  // the range holds whole tile rows
    const long long c0 = in ? a.tr_chunk[bi] : 0, c1 = in ? a.tr_chunk[bi + 1] : 0;
    for (long long j = 0; __ballot(c0 + j < c1) != 0ull; j++) {
        const bool have = c0 + j < c1;
        const int3 h = have ? a.chunks[c0 + j] : make_int3(0, 0, -1);
        const bool act = have && i16 <= chunk_last(h) && (S == kSellAll64 || chunk_class(h) == S);
        const int e = h.x + i16;
        const int id = act ? (int)a.eidx[e] : 0;
        const int lr = act ? 16 * g + (id >> 4) : -1;
        const int row = chunk_rowbase(h) + (id >> 4), col = chunk_colbase(h) + (id & 15);
        // first lane of this row's run of entries in the chunk
        const int plr = __shfl_up(lr, 1, 16), pcol = __shfl_up(col, 1, 16), nlr = __shfl_down(lr, 1, 16);
        const bool first = act && (i16 == 0 || plr != lr);
        int start = first ? i16 : 0;
#pragma unroll
        for (int o = 1; o < 16; o <<= 1) {
            const int t = __shfl_up(start, o, 16);
            if (i16 >= o) start = max(start, t);
        }
        int pos = 0, prev = 0;
        if (act) {
            pos = cnt[lr] + i16 - start;
            prev = first ? last[lr] : pcol;
        }
        __syncthreads();
        if (act) {
            f(lr, pos, col - row, col, e, prev);
            if (i16 == 15 || nlr != lr) {
                cnt[lr] = pos + 1;
                last[lr] = col;
            }
        }
        __syncthreads();
    }
}

__device__ __forceinline__ int wave_red(int v, int op)
{
#pragma unroll
    for (int o = 32; o; o >>= 1) {
        const int t = __shfl_xor(v, o);
        v = op == 0 ? v + t : op == 1 ? min(v, t) : max(v, t);
    }
    return v;
}

__global__ __launch_bounds__(64) void sell_count_kernel(SellBuildArgs a, unsigned mask, SellSlot *out)
{
    __shared__ unsigned bm[kBuildWords];
    __shared__ int cnt[64], last[64];
    const long long slot = blockIdx.x;
    const SlotRows s = slot_rows(a, slot);
    const int lane = threadIdx.x;
    if (s.l0 >= s.nr) {
        if (lane < kSellStreams && (mask >> lane & 1)) out[lane * a.slots + slot] = SellSlot{0, 0, 0, 0, INT_MAX, INT_MIN};
        return;
    }
    for (int S = 0; S < kSellStreams; S++) {
        if (!(mask >> S & 1)) continue;
        for (int w = lane; w < a.words; w += 64) bm[w] = 0u;
        int asc = 1, rmin = INT_MAX, rmax = INT_MIN, cmin = INT_MAX, cmax = INT_MIN;
        walk_slot(a, s, S, cnt, last, [&](int, int, int rel, int col, int, int prev) {
            asc &= col > prev;
            rmin = min(rmin, rel);
            rmax = max(rmax, rel);
            cmin = min(cmin, col);
            cmax = max(cmax, col);
            const int b = rel + a.max_off;
            atomicOr(&bm[b >> 5], 1u << (b & 31));
        });
        int cols = 0;
        for (int w = lane; w < a.words; w += 64) cols += __popc(bm[w]);
        const SellSlot r{wave_red(cnt[lane], 2), wave_red(asc, 1) ? wave_red(cols, 0) : INT_MAX, wave_red(rmin, 1),
                         wave_red(rmax, 2), wave_red(cmin, 1), wave_red(cmax, 2)};
        if (lane == 0) out[S * a.slots + slot] = r;
        __syncthreads();
    }
}

// One slot of stream S: VT the value type, src its values in the entry order.
template <class VT>
__global__ __launch_bounds__(64) void sell_fill_kernel(SellBuildArgs a, int S, int lgE, const int *soff,
                                                       const uint8_t *shared, const VT *src, int16_t *idx, VT *val)
{
    __shared__ unsigned bm[kBuildWords];
    __shared__ int pre[kBuildWords], cnt[64], last[64], U[kBuildUnion];
    const long long slot = blockIdx.x;
    const SlotRows s = slot_rows(a, slot);
    const int u0 = soff[slot], u1 = soff[slot + 1], lane = threadIdx.x;
    if (u0 >= u1) return;
    const bool sh = shared[slot] != 0;
    int nU = 0;
    if (sh) {
        for (int w = lane; w < a.words; w += 64) bm[w] = 0u;
        walk_slot(a, s, S, cnt, last, [&](int, int, int rel, int, int, int) {
            const int b = rel + a.max_off;
            atomicOr(&bm[b >> 5], 1u << (b & 31));
        });
        // prefix counts: each lane a run of words, then across the lanes
        const int run = (a.words + 63) / 64, w0 = min(lane * run, a.words), w1 = min(w0 + run, a.words);
        int own = 0;
        for (int w = w0; w < w1; w++) own += __popc(bm[w]);
        int inc = own;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int t = __shfl_up(inc, o);
            if (lane >= o) inc += t;
        }
        nU = __shfl(inc, 63);
        int at = inc - own;
        for (int w = w0; w < w1; w++) {
            pre[w] = at;
            for (unsigned m = bm[w]; m; m &= m - 1)
                if (at < kBuildUnion) U[at++] = w * 32 + __ffs(m) - 1 - a.max_off;
        }
        __syncthreads();
    }
    // padding: the lane's own row, or (shared) the slice's relative columns in every lane
    const int base = s.r0 + min(64 * s.v + lane, s.nr - 1);
    const int own = s.l0 + lane < s.nr ? s.r0 + s.l0 + lane : base;
    const int E = 1 << lgE, ne = (u1 - u0) << lgE;
    for (int p = 0; p < ne; p++) {
        const size_t q = ((size_t)(u0 + (p >> lgE)) * 64 + lane) * E + (p & (E - 1));
        idx[q] = sh ? (int16_t)((p < nU ? U[p] : 0) + 1024 * s.k) : (int16_t)(own - base);
        val[q] = VT(0);
    }
    // the entries of a row are written by other lanes: after the padding has arrived
    wait_own_stores();
    __syncthreads();
    walk_slot(a, s, S, cnt, last, [&](int lr, int pos, int rel, int col, int e, int) {
        int p = pos;
        if (sh) {
            const int b = rel + a.max_off;
            p = pre[b >> 5] + __popc(bm[b >> 5] & ((1u << (b & 31)) - 1u));
        }
        const size_t q = ((size_t)(u0 + (p >> lgE)) * 64 + lr) * E + (p & (E - 1));
        if (!sh) idx[q] = (int16_t)(col - (s.r0 + min(64 * s.v + lr, s.nr - 1)));
        val[q] = src[e];
    });
}

}  // namespace mfk

namespace mf {

namespace {
struct DevBuf {  // freed on every return
    void *p = nullptr;
    ~DevBuf() { free_dev(p); }
};
}  // namespace

static mfk::SellBuildArgs build_args(const DeviceLayout &L, const Partition &P, const SellLayout &SL)
{
    mfk::SellBuildArgs a;
    a.chunks = L.chunks;
    a.tr_chunk = L.d_tr_chunk;
    a.wg_tr = P.wg_tr;
    a.eidx = L.eidx;
    a.v64 = L.v64;
    a.v32 = L.v32;
    a.v16 = L.v16;
    a.v8 = L.v8;
    a.n = L.n_rows;
    a.rpt = SL.rpt;
    a.max_off = L.max_offset;
    a.words = (2 * L.max_offset + 1 + 31) / 32;
    a.slots = (long long)P.G * 16 * SL.rpt;
    return a;
}

// Column words and values of stream k, whose offsets and flags are in place.
static void fill_stream(const mfk::SellBuildArgs &a, const SellLayout &SL, int k, hipStream_t s)
{
    if (SL.units[k] == 0) return;
    const int E = mfk::sell_e_host(k, SL.narrow), lgE = E == 2 ? 1 : E == 4 ? 2 : 3;
    const dim3 grid((unsigned)a.slots), blk(64);
    int16_t *ix = (int16_t *)SL.idx[k];
    if (k == 0 || k == mfk::kSellAll64)
        hipLaunchKernelGGL(mfk::sell_fill_kernel<double>, grid, blk, 0, s, a, k, lgE, SL.soff[k], SL.shared[k], a.v64, ix,
                           (double *)SL.val[k]);
    else if (k == 1)
        hipLaunchKernelGGL(mfk::sell_fill_kernel<float>, grid, blk, 0, s, a, k, lgE, SL.soff[k], SL.shared[k], a.v32, ix,
                           (float *)SL.val[k]);
    else if (k == 2)
        hipLaunchKernelGGL(mfk::sell_fill_kernel<uint16_t>, grid, blk, 0, s, a, k, lgE, SL.soff[k], SL.shared[k], a.v16,
                           ix, (uint16_t *)SL.val[k]);
    else
        hipLaunchKernelGGL(mfk::sell_fill_kernel<int8_t>, grid, blk, 0, s, a, k, lgE, SL.soff[k], SL.shared[k], a.v8, ix,
                           (int8_t *)SL.val[k]);
}

mf_status refill_sell(mf_matrix *A, Partition &P, hipStream_t s)
{
    free_sell(P.sell[1]);
    P.sell[1] = nullptr;
    P.sort_pays = -1;
    if (!P.sell[0]) return MF_SUCCESS;
    const SellLayout &SL = *P.sell[0];
    const mfk::SellBuildArgs a = build_args(A->L, P, SL);
    for (int k = 0; k < mfk::kSellStreams; k++)
        if (SL.soff[k]) fill_stream(a, SL, k, s);
    return hipGetLastError() == hipSuccess ? MF_SUCCESS : MF_ERR_HIP;
}

mf_status build_sell_gpu(mf_matrix *A, const Partition &P, SellLayout &SL, unsigned mask, hipStream_t s)
{
    DeviceLayout &L = A->L;
    const int R = P.G, NW = 16, rpt = SL.rpt, n = L.n_rows;
    const int64_t slots = (int64_t)R * NW * rpt;
    mf_status st = L.ensure_tile_order(s);
    if (st != MF_SUCCESS) return st;
    const mfk::SellBuildArgs a = build_args(L, P, SL);
    if (a.words > mfk::kBuildWords) return MF_ERR_TOO_LARGE;
    std::vector<mfk::SellSlot> info((size_t)mfk::kSellStreams * slots);
    DevBuf dinfo;
    if (hipMalloc(&dinfo.p, sizeof(mfk::SellSlot) * info.size()) != hipSuccess) return MF_ERR_ALLOC;
    // streams of classes that no tile has stay empty
    const mfk::SellSlot none{0, 0, 0, 0, INT_MAX, INT_MIN};
    unsigned counted = mask;
    for (int k = 0; k < mfk::kSellAll64; k++)
        if ((mask >> k & 1) && L.nnz_by_class[k] == 0) {
            counted &= ~(1u << k);
            std::fill_n(info.begin() + k * slots, slots, none);
        }
    hipLaunchKernelGGL(mfk::sell_count_kernel, dim3((unsigned)slots), dim3(64), 0, s, a, counted,
                       (mfk::SellSlot *)dinfo.p);
    if (hipGetLastError() != hipSuccess) return MF_ERR_HIP;
    for (int k = 0; k < mfk::kSellStreams; k++)
        if ((counted >> k & 1) &&
            hipMemcpyAsync(info.data() + k * slots, (mfk::SellSlot *)dinfo.p + k * slots, sizeof(mfk::SellSlot) * slots,
                           hipMemcpyDeviceToHost, s) != hipSuccess)
            return MF_ERR_HIP;
    if (hipStreamSynchronize(s) != hipSuccess) return MF_ERR_HIP;
    // unit profile of the class streams: narrow when it saves at least 15 % of their bytes
    if (mask & 0xEu) {
        double bw = 0, bn = 0;
        for (int k = 1; k <= 3; k++) {
            if (!(mask >> k & 1)) continue;
            const int ew = mfk::sell_e_host(k, false), en = mfk::sell_e_host(k, true);
            const double per = 64.0 * (2 + mfk::sell_vbytes_host(k));
            for (int64_t i = 0; i < slots; i++) {
                const int len = info[k * slots + i].len;
                bw += per * ew * ((len + ew - 1) / ew);
                bn += per * en * ((len + en - 1) / en);
            }
        }
        SL.narrow = bn < 0.85 * bw;
    }
    std::vector<int> win[2];
    for (int w = 0; w < 2; w++) {
        if (!(mask & (w ? 0xFu : 1u << mfk::kSellAll64))) continue;
        win[w].resize(2 * (size_t)R);
        for (int r = 0; r < R; r++) {
            win[w][2 * r] = P.h_tr[r] * kTile;
            win[w][2 * r + 1] = std::max(P.h_tr[r] * kTile, std::min(P.h_tr[r + 1] * kTile, n));
        }
    }
    for (int k = 0; k < mfk::kSellStreams; k++) {
        if (!(mask >> k & 1)) continue;
        const mfk::SellSlot *in = info.data() + k * slots;
        const int E = mfk::sell_e_host(k, SL.narrow);
        std::vector<int> soff(slots + 1, 0), lm((size_t)R * NW, 63);
        std::vector<uint8_t> shared(slots, 0);
        int64_t u = 0;
        SL.max_wg_units[k] = 0;
        SL.shared_units[k] = 0;
        std::vector<int> &wn = win[k == mfk::kSellAll64 ? 0 : 1];
        for (int r = 0; r < R; r++) {
            const int r0 = P.h_tr[r] * kTile, nr = std::max(0, std::min(P.h_tr[r + 1] * kTile, n) - r0);
            const int64_t u_range = u;
            for (int v = 0; v < NW; v++) {
                const int64_t s0 = ((int64_t)r * NW + v) * rpt, u_wave = u;
                int k0 = -1, k1 = -1;  // first and last slice with entries
                for (int j = 0; j < rpt; j++)
                    if (in[s0 + j].len > 0) {
                        if (k0 < 0) k0 = j;
                        k1 = j;
                    }
                bool same = true;
                for (int j = 0; j < rpt; j++) {
                    const mfk::SellSlot &sl = in[s0 + j];
                    int nu = (sl.len + E - 1) / E;
                    // an empty slice between two others gets one zero unit (the SpMV ends at
                    // most one slice per unit)
                    if (k0 >= 0 && j > k0 && j < k1) nu = std::max(nu, 1);
                    soff[s0 + j] = (int)u;
                    u += nu;
                    if (!nu) continue;
                    // shared column words: the slice's relative columns fit its units, and in
                    // every lane name a column of the matrix
                    const int b0 = r0 + std::min(64 * v, nr - 1) + 1024 * j, b1 = r0 + std::min(64 * v + 63, nr - 1) + 1024 * j;
                    const int lo = b0 + (sl.len ? std::min(sl.rmin, 0) : 0), hi = b1 + (sl.len ? std::max(sl.rmax, 0) : 0);
                    shared[s0 + j] = (int64_t)sl.cols <= (int64_t)nu * E && sl.cols <= mfk::kBuildUnion && lo >= 0 && hi < n;
                    same = same && shared[s0 + j];
                    wn[2 * r] = std::min(wn[2 * r], shared[s0 + j] ? lo : sl.cmin);
                    wn[2 * r + 1] = std::max(wn[2 * r + 1], 1 + (shared[s0 + j] ? hi : sl.cmax));
                }
                if (u > u_wave && same) {
                    lm[(size_t)r * NW + v] = 0;
                    SL.shared_units[k] += u - u_wave;
                }
            }
            SL.max_wg_units[k] = std::max<int64_t>(SL.max_wg_units[k], u - u_range);
        }
        soff[slots] = (int)u;
        if (u >= INT32_MAX / 64) return MF_ERR_TOO_LARGE;
        SL.units[k] = u;
        const size_t ne = (size_t)u * 64 * E;
        if ((st = upload((void **)&SL.lmask[k], lm.data(), sizeof(int) * lm.size(), s)) != MF_SUCCESS ||
            (st = upload((void **)&SL.soff[k], soff.data(), sizeof(int) * soff.size(), s)) != MF_SUCCESS ||
            (st = upload((void **)&SL.shared[k], shared.data(), shared.size(), s)) != MF_SUCCESS ||
            (st = upload(&SL.idx[k], nullptr, sizeof(int16_t) * ne, s)) != MF_SUCCESS ||
            (st = upload(&SL.val[k], nullptr, ne * mfk::sell_vbytes_host(k), s)) != MF_SUCCESS)
            return st;
        SL.bytes += (double)sizeof(int) * soff.size() + 2.0 * ne + (double)ne * mfk::sell_vbytes_host(k);
        fill_stream(a, SL, k, s);
        // (the uploads above read these host vectors)
        if (hipGetLastError() != hipSuccess || hipStreamSynchronize(s) != hipSuccess) return MF_ERR_HIP;
    }
    for (int w = 0; w < 2; w++) {
        if (win[w].empty()) continue;
        SL.max_win[w] = 0;
        SL.sum_win[w] = 0;
        for (int r = 0; r < R; r++) {
            SL.max_win[w] = std::max(SL.max_win[w], win[w][2 * r + 1] - win[w][2 * r]);
            SL.sum_win[w] += win[w][2 * r + 1] - win[w][2 * r];
        }
        if ((st = upload((void **)&SL.win[w], win[w].data(), sizeof(int) * win[w].size(), s)) != MF_SUCCESS) return st;
    }
    return hipStreamSynchronize(s) == hipSuccess ? MF_SUCCESS : MF_ERR_HIP;
}

}  // namespace mf
