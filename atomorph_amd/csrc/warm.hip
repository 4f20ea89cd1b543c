// Learned warm start of the transport refinement.
//
// The reference starts every chain row in the row-major pixel order its
// blobs were built in (thread.cpp:740-891) and leaves the whole assignment
// to the pair-swap descent.  Here, before the descent, row y+1 of each chain
// is reordered so that slot i receives the point of key frame y+1 whose
// rank in raster order (y, then x, at 1/16 px) equals the rank of the
// MLP's prediction for slot i's row-y atom:
//   features  per atom of row y: x/W, y/H, RGBA/255 of its key-frame pixel,
//             (x - cx)/s, (y - cy)/s with (cx, cy) the chain row's centroid
//             and s its RMS radius + 1 px;
//   predict   MLP -> (u, v), target position (cx' + s' u, cy' + s' v) in the
//             statistics of row y+1;
//   match     sort (chain, raster key of the prediction) and (chain, raster
//             key of the row y+1 point) with an LSD radix sort and pair them
//             rank by rank, so every row stays a permutation of its points.
// The reference's start pairs the blobs' pixels rank by rank in the same
// raster order; a prediction that keeps each atom's position relative to
// its blob (scaled) reproduces that start, so what the network learns is
// what changes it.  Rows are processed y = 0 .. h-2 in order; row 0 keeps
// its order.  The same feature kernel writes training targets (the row y+1
// position of each slot, normalised the same way) from converged chains.
#include "common.h"
#include "../../include/atomorph_hip.h"
#include "shade.h"

#include <algorithm>

using namespace amh;
using namespace amh::shade;

namespace {

constexpr int kT = 256;

struct RowStat {
    double cx, cy, s;
};

__device__ __forceinline__ double pt_xd(uint64_t w) { return double(pt_fx(w)) * (1.0 / 256.0); }
__device__ __forceinline__ double pt_yd(uint64_t w) { return double(pt_fy(w)) * (1.0 / 256.0); }

// Centroid and RMS radius (+1 px) of every (row, chain): one block per pair.
__global__ __launch_bounds__(kT) void k_row_stats(amh_render R, RowStat *__restrict__ st) {
    __shared__ double part[4][4];
    const int c = blockIdx.x, y = blockIdx.y;
    const int64_t off = R.chain_off_dev[c];
    const int w = R.chain_w_dev[c];
    const uint64_t *row = R.pts_dev + int64_t(y) * R.wtot + off;
    double sx = 0, sy = 0, sxx = 0, syy = 0;
    for (int i = threadIdx.x; i < w; i += kT) {
        const double x = pt_xd(row[i]), v = pt_yd(row[i]);
        sx += x;
        sy += v;
        sxx += x * x;
        syy += v * v;
    }
    double q[4] = {sx, sy, sxx, syy};
    for (int k = 0; k < 4; ++k)
        for (int o = 32; o > 0; o >>= 1) q[k] += __shfl_down(q[k], o, 64);
    if ((threadIdx.x & 63) == 0)
        for (int k = 0; k < 4; ++k) part[threadIdx.x >> 6][k] = q[k];
    __syncthreads();
    if (threadIdx.x == 0) {
        double t[4] = {0, 0, 0, 0};
        for (int wv = 0; wv < kT / 64; ++wv)
            for (int k = 0; k < 4; ++k) t[k] += part[wv][k];
        const double n = w > 0 ? double(w) : 1.0;
        const double cx = t[0] / n, cy = t[1] / n;
        const double var = fmax(t[2] / n - cx * cx + t[3] / n - cy * cy, 0.0);
        st[int64_t(y) * R.nchains + c] = RowStat{cx, cy, sqrt(var) + 1.0};
    }
}

// Features of row y (x[wtot][8]) and, when t != NULL, the targets: the
// normalised positions the same slots hold in row y+1 (t[wtot][2]).
__global__ __launch_bounds__(kT) void k_features(amh_render R, int y, const RowStat *__restrict__ st,
                                                float *__restrict__ x, float *__restrict__ t) {
    const int64_t a = int64_t(blockIdx.x) * kT + threadIdx.x;
    const int c = block_chain(R.chain_off_dev, R.nchains, a);
    if (a >= R.wtot) return;
    const int yn = (y + 1) % R.nkeys;
    const uint64_t p = R.pts_dev[int64_t(y) * R.wtot + a];
    const RowStat s = st[int64_t(y) * R.nchains + c];
    const double px = pt_xd(p), py = pt_yd(p);
    uint32_t col = 0;
    if (pt_flags(p) & HAS_PIXEL) col = key_px(R.keys_dev, y, R.width, R.height, pt_x(p), pt_y(p));
    float *f = x + a * 8;
    f[0] = float(px / R.width);
    f[1] = float(py / R.height);
    for (int k = 0; k < 4; ++k) f[2 + k] = float(ch(col, k)) * (1.0f / 255.0f);
    f[6] = float((px - s.cx) / s.s);
    f[7] = float((py - s.cy) / s.s);
    if (t) {
        const uint64_t q = R.pts_dev[int64_t(yn) * R.wtot + a];
        const RowStat sn = st[int64_t(yn) * R.nchains + c];
        t[a * 2 + 0] = float((pt_xd(q) - sn.cx) / sn.s);
        t[a * 2 + 1] = float((pt_yd(q) - sn.cy) / sn.s);
    }
}

// Raster key of a position at 1/16 px: chain, y, x, with cx bits per
// coordinate (positions clamped to the frame's range).
__device__ __forceinline__ uint64_t raster_key(uint64_t chain, double x, double y, int cx) {
    const double lim = double((1ull << cx) - 1);
    const uint64_t fx = uint64_t(fmin(fmax(rint(x * 16.0), 0.0), lim));
    const uint64_t fy = uint64_t(fmin(fmax(rint(y * 16.0), 0.0), lim));
    return (chain << (2 * cx)) | (fy << cx) | fx;
}

// Two lists of n keys, sorted side by side: the predictions for row y+1, then
// the points row y+1 holds now; values are the slots.  Sorted, each lists
// chain by chain (each chain has its width in both), so rank r of chain c sits
// at the same place in both.  The row's points are kept in row[] for
// k_match_apply, which overwrites them.
__global__ __launch_bounds__(kT) void k_match_keys(amh_render R, int yn, const RowStat *__restrict__ st,
                                                  const float *__restrict__ pred, int cx,
                                                  uint64_t *__restrict__ key, uint32_t *__restrict__ val,
                                                  uint64_t *__restrict__ row) {
    const int64_t a = int64_t(blockIdx.x) * kT + threadIdx.x;
    const int c = block_chain(R.chain_off_dev, R.nchains, a);
    if (a >= R.wtot) return;
    const RowStat s = st[int64_t(yn) * R.nchains + c];
    const double ux = s.cx + s.s * double(pred[a * 2 + 0]), uy = s.cy + s.s * double(pred[a * 2 + 1]);
    const uint64_t q = R.pts_dev[int64_t(yn) * R.wtot + a];
    key[a] = raster_key(uint64_t(c), ux, uy, cx);
    const uint64_t lim = (1ull << cx) - 1;
    key[R.wtot + a] =
        (uint64_t(c) << (2 * cx)) | (min(uint64_t(pt_fy(q) >> 4), lim) << cx) | min(uint64_t(pt_fx(q) >> 4), lim);
    row[a] = q;
    val[a] = uint32_t(a);
    val[R.wtot + a] = uint32_t(a);
}

// Rank r of both sorted lists pairs up inside one chain: the slot with the
// r-th prediction takes the r-th point.
__global__ void k_match_apply(int64_t n, const uint32_t *__restrict__ sorted, const uint64_t *__restrict__ row,
                              uint64_t *__restrict__ out) {
    const int64_t r = int64_t(blockIdx.x) * kT + threadIdx.x;
    if (r < n) out[sorted[r]] = row[sorted[n + r]];
}

// ------------------------------------------------------- radix sort
// LSD radix sort of two lists of n (u64 key, u32 value) pairs (blockIdx.y is
// the list, the second n after the first) in as few passes of at most
// kRsBits bits as the keys need, their bits dealt evenly; a block covers
// kRsTile elements.  Launches and latency bound it: a pass is three launches
// (digit counts per block, their prefix per digit, scatter), so it takes nine
// bits rather than eight, and the scatter scans the digits' totals itself and
// meets two barriers, not four for each 256 elements.  2 x 229k pairs of 36
// bits on one MI355X: 72 us, 123 us as one list with a bit to tell them apart
// in five passes of four launches.
constexpr int kRsBits = 9, kRsDigits = 1 << kRsBits;
constexpr int kRsPer = 4;  // elements of a thread
constexpr int kRsTile = kT * kRsPer;

__global__ __launch_bounds__(kT) void k_rs_hist(const uint64_t *__restrict__ key, int64_t n, int shift, uint32_t mask,
                                               int nblk, int *__restrict__ hist) {
    __shared__ int h[kRsDigits];
    for (int d = threadIdx.x; d < kRsDigits; d += kT) h[d] = 0;
    __syncthreads();
    const int64_t base = int64_t(blockIdx.x) * kRsTile;
    key += blockIdx.y * n;
    hist += (int64_t(blockIdx.y) * nblk + blockIdx.x) * kRsDigits;
    for (int j = 0; j < kRsPer; ++j) {
        const int64_t e = base + j * kT + threadIdx.x;
        if (e < n) atomicAdd(&h[uint32_t(key[e] >> shift) & mask], 1);
    }
    __syncthreads();
    for (int d = threadIdx.x; d < kRsDigits; d += kT) hist[d] = h[d];
}

// kRsCols digits per block: their counts over the blocks, hist[block][digit],
// become exclusive prefixes, and total[digit] their sums.  A thread adds up a
// digit's counts over a share of the blocks, rows of kRsCols words at a time.
constexpr int kRsCols = 16, kPrefixT = 1024, kRsShares = kPrefixT / kRsCols;

__global__ __launch_bounds__(kPrefixT) void k_rs_prefix(int *__restrict__ hist, int nblk, int *__restrict__ total) {
    __shared__ int part[kRsShares][kRsCols];
    const int col = threadIdx.x % kRsCols, share = threadIdx.x / kRsCols, d = blockIdx.x * kRsCols + col;
    hist += int64_t(blockIdx.y) * nblk * kRsDigits + d;
    const int per = (nblk + kRsShares - 1) / kRsShares, lo = min(share * per, nblk), hi = min(lo + per, nblk);
    int sum = 0;
#pragma unroll 4
    for (int b = lo; b < hi; ++b) sum += hist[int64_t(b) * kRsDigits];
    part[share][col] = sum;
    __syncthreads();
    // (every share in the same steps, in place)
    int at = 0;
    for (int q = 0; q < kRsShares; ++q) at += q < share ? part[q][col] : 0;
    if (share == kRsShares - 1) total[blockIdx.y * kRsDigits + d] = at + sum;
#pragma unroll 8
    for (int b = lo; b < hi; ++b) {
        const int v = hist[int64_t(b) * kRsDigits];
        hist[int64_t(b) * kRsDigits] = at;
        at += v;
    }
}

// Inclusive sum over the block, in thread order.
__device__ __forceinline__ int block_inclusive(int v, int *wsum) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int off = 1; off < 64; off <<= 1) {
        const int u = __shfl_up(v, off, 64);
        if (lane >= off) v += u;
    }
    if (lane == 63) wsum[wave] = v;
    __syncthreads();
    for (int w = 0; w < wave; ++w) v += wsum[w];
    return v;
}

// Stable: a wave's elements are consecutive, its digits are counted in its
// own counters in order (ranks within 64 from per-digit lane masks built of
// ballots), and the waves' counts are summed once at the end.
__global__ __launch_bounds__(kT) void k_rs_scatter(const uint64_t *__restrict__ key, const uint32_t *__restrict__ val,
                                                  int64_t n, int shift, uint32_t mask, int nblk,
                                                  const int *__restrict__ hist, const int *__restrict__ total,
                                                  uint64_t *__restrict__ okey, uint32_t *__restrict__ oval) {
    static_assert(kRsDigits == 2 * kT, "two digits per thread");
    __shared__ int cnt[kT / 64][kRsDigits];
    __shared__ int wsum[kT / 64];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const uint64_t below = (1ull << lane) - 1ull;
    const int64_t e0 = int64_t(blockIdx.x) * kRsTile + wave * (64 * kRsPer) + lane;
    key += blockIdx.y * n;
    val += blockIdx.y * n;
    okey += blockIdx.y * n;
    oval += blockIdx.y * n;
    hist += (int64_t(blockIdx.y) * nblk + blockIdx.x) * kRsDigits;
    total += blockIdx.y * kRsDigits;
    uint64_t k[kRsPer];
    uint32_t v[kRsPer];
#pragma unroll
    for (int j = 0; j < kRsPer; ++j) {
        const int64_t e = e0 + j * 64;
        k[j] = e < n ? key[e] : 0;
        v[j] = e < n ? val[e] : 0;
    }
    // the two digits of this thread: where this block's elements of them go
    const int d0 = 2 * t, d1 = 2 * t + 1;
    const int2 tot = *reinterpret_cast<const int2 *>(total + d0), h = *reinterpret_cast<const int2 *>(hist + d0);
    for (int d = lane; d < kRsDigits; d += 64) cnt[wave][d] = 0;
    int pos[kRsPer];
#pragma unroll
    for (int j = 0; j < kRsPer; ++j) {
        const bool ok = e0 + j * 64 < n;
        const uint32_t d = uint32_t(k[j] >> shift) & mask;
        uint64_t same = __ballot(ok);
#pragma unroll
        for (int bit = 0; bit < kRsBits; ++bit) {
            const uint64_t bb = __ballot((d >> bit) & 1);
            same &= ((d >> bit) & 1) ? bb : ~bb;
        }
        const int rank = int(__popcll(same & below));
        wave_order();
        const int before = cnt[wave][d];
        wave_order();
        if (ok && rank == 0) cnt[wave][d] = before + int(__popcll(same));
        pos[j] = before + rank;
    }
    const int incl = block_inclusive(tot.x + tot.y, wsum);  // (its barrier publishes cnt)
    int b0 = incl - tot.x - tot.y + h.x, b1 = incl - tot.y + h.y;
    for (int w = 0; w < kT / 64; ++w) {
        const int c0 = cnt[w][d0], c1 = cnt[w][d1];
        cnt[w][d0] = b0;
        cnt[w][d1] = b1;
        b0 += c0;
        b1 += c1;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kRsPer; ++j) {
        if (e0 + j * 64 >= n) continue;
        const int to = cnt[wave][uint32_t(k[j] >> shift) & mask] + pos[j];
        okey[to] = k[j];
        oval[to] = v[j];
    }
}

struct WarmLayout {
    size_t stats, x, pred, kk, kv, k2, i2, hist, sums, row, total;
    int nblk;
};

WarmLayout warm_layout(int64_t wtot, int32_t nchains, int32_t nkeys) {
    WarmLayout L{};
    size_t o = 0;
    auto al = [](size_t v) { return (v + 255) & ~size_t(255); };
    const size_t n = size_t(wtot);
    L.nblk = int((wtot + kRsTile - 1) / kRsTile);
    const size_t hn = 2 * size_t(kRsDigits) * size_t(std::max(L.nblk, 1));
    L.stats = o; o = al(o + sizeof(RowStat) * size_t(nkeys) * size_t(std::max(nchains, 1)));
    L.x = o; o = al(o + n * 8 * 4);
    L.pred = o; o = al(o + n * 2 * 4);
    L.kk = o; o = al(o + 2 * n * 8);
    L.kv = o; o = al(o + 2 * n * 4);
    L.k2 = o; o = al(o + 2 * n * 8);
    L.i2 = o; o = al(o + 2 * n * 4);
    L.hist = o; o = al(o + hn * 4);
    L.sums = o; o = al(o + 2 * kRsDigits * 4);
    L.row = o; o = al(o + n * 8);
    L.total = o;
    return L;
}

// Sorts both lists of n in (k, v) by the low `bits` bits of the keys,
// ping-ponging through (k2, v2); returns the values array that holds the result.
uint32_t *radix_sort(uint64_t *k, uint32_t *v, uint64_t *k2, uint32_t *v2, int64_t n, int bits, char *base,
                     const WarmLayout &L, hipStream_t s) {
    int *hist = reinterpret_cast<int *>(base + L.hist);
    int *total = reinterpret_cast<int *>(base + L.sums);
    const int passes = (bits + kRsBits - 1) / kRsBits;
    for (int p = 0, shift = 0; p < passes; ++p) {
        const int digit = (bits - shift + passes - p - 1) / (passes - p);
        const uint32_t mask = (1u << digit) - 1u;
        hipLaunchKernelGGL(k_rs_hist, dim3(uint32_t(L.nblk), 2), dim3(kT), 0, s, k, n, shift, mask, L.nblk, hist);
        hipLaunchKernelGGL(k_rs_prefix, dim3(kRsDigits / kRsCols, 2), dim3(kPrefixT), 0, s, hist, L.nblk, total);
        hipLaunchKernelGGL(k_rs_scatter, dim3(uint32_t(L.nblk), 2), dim3(kT), 0, s, k, v, n, shift, mask, L.nblk, hist,
                           total, k2, v2);
        std::swap(k, k2);
        std::swap(v, v2);
        shift += digit;
    }
    return v;
}

}  // namespace

extern "C" size_t amh_warm_workspace_bytes(int64_t wtot, int32_t nchains, int32_t nkeys) {
    return warm_layout(wtot, nchains, nkeys).total;
}

// Features (x_dev[wtot][8]) of key frame y and, if t_dev != NULL, the
// targets (t_dev[wtot][2]) from row y+1; uses the workspace's statistics.
extern "C" int amh_learn_features(const amh_render *R, int32_t y, float *x_dev, float *t_dev, void *ws,
                                  size_t ws_bytes, void *stream) {
    if (!R || !x_dev || !ws || y < 0 || y >= R->nkeys || R->wtot <= 0 || R->nchains <= 0 || !R->pts_dev ||
        !R->keys_dev || !R->chain_off_dev || !R->chain_w_dev) {
        set_error("amh_learn_features: invalid argument");
        return AMH_E_ARG;
    }
    const WarmLayout L = warm_layout(R->wtot, R->nchains, R->nkeys);
    if (ws_bytes < L.total) {
        set_error("amh_learn_features: workspace %zu < %zu bytes", ws_bytes, L.total);
        return AMH_E_ARG;
    }
    hipStream_t s = static_cast<hipStream_t>(stream);
    RowStat *st = reinterpret_cast<RowStat *>(static_cast<char *>(ws) + L.stats);
    hipLaunchKernelGGL(k_row_stats, dim3(uint32_t(R->nchains), uint32_t(R->nkeys)), dim3(kT), 0, s, *R, st);
    hipLaunchKernelGGL(k_features, dim3(uint32_t((R->wtot + kT - 1) / kT)), dim3(kT), 0, s, *R, y, st, x_dev, t_dev);
    AMH_LAUNCH_CHECK("amh_learn_features");
    return AMH_OK;
}

// Reorders rows 1 .. nkeys-1 of pts_dev (the chains R describes; R->pts_dev
// must be pts_dev) by the MLP's predictions, in place.
extern "C" int amh_warm_start(void *mlp, const amh_render *R, uint64_t *pts_dev, void *ws, size_t ws_bytes,
                              void *stream) {
    if (!mlp || !R || !pts_dev || R->pts_dev != pts_dev || !ws || R->wtot <= 0 || R->nchains <= 0 ||
        R->nchains > 65535 || R->wtot > int64_t(0x3FFFFFFF) || !R->keys_dev || !R->chain_off_dev ||
        !R->chain_w_dev) {
        set_error("amh_warm_start: invalid argument");
        return AMH_E_ARG;
    }
    const WarmLayout L = warm_layout(R->wtot, R->nchains, R->nkeys);
    if (ws_bytes < L.total) {
        set_error("amh_warm_start: workspace %zu < %zu bytes", ws_bytes, L.total);
        return AMH_E_ARG;
    }
    hipStream_t s = static_cast<hipStream_t>(stream);
    amh::ProfScope ps_("warm_start", s);
    char *b = static_cast<char *>(ws);
    RowStat *st = reinterpret_cast<RowStat *>(b + L.stats);
    float *x = reinterpret_cast<float *>(b + L.x), *pred = reinterpret_cast<float *>(b + L.pred);
    uint64_t *kk = reinterpret_cast<uint64_t *>(b + L.kk), *k2 = reinterpret_cast<uint64_t *>(b + L.k2);
    uint32_t *kv = reinterpret_cast<uint32_t *>(b + L.kv), *i2 = reinterpret_cast<uint32_t *>(b + L.i2);
    uint64_t *row = reinterpret_cast<uint64_t *>(b + L.row);
    const uint32_t ga = uint32_t((R->wtot + kT - 1) / kT);
    hipLaunchKernelGGL(k_row_stats, dim3(uint32_t(R->nchains), uint32_t(R->nkeys)), dim3(kT), 0, s, *R, st);
    // key bits: chain, and y, x at 1/16 px over the frame
    int cb = 0, cx = 0;
    while ((1 << cb) < R->nchains) ++cb;
    while ((int64_t(1) << cx) < int64_t(std::max(std::max(R->width, R->height), 1)) * 16) ++cx;
    const int bits = cb + 2 * cx;
    for (int y = 0; y + 1 < R->nkeys; ++y) {
        hipLaunchKernelGGL(k_features, dim3(ga), dim3(kT), 0, s, *R, y, st, x, static_cast<float *>(nullptr));
        if (int r = amh_mlp_forward(mlp, x, R->wtot, pred, stream)) return r;
        hipLaunchKernelGGL(k_match_keys, dim3(ga), dim3(kT), 0, s, *R, y + 1, st, pred, cx, kk, kv,
                           row);
        const uint32_t *sorted = radix_sort(kk, kv, k2, i2, R->wtot, bits, b, L, s);
        uint64_t *dst = pts_dev + int64_t(y + 1) * R->wtot;
        hipLaunchKernelGGL(k_match_apply, dim3(ga), dim3(kT), 0, s, R->wtot, sorted, row, dst);
    }
    AMH_LAUNCH_CHECK("amh_warm_start");
    return AMH_OK;
}
