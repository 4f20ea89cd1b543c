// Key-frame ingest, blob segmentation, blob statistics and chain build.
//
// Segmentation replaces thread::blobify_frame (thread.cpp:225-412).  At the
// library default blob_threshold 1.0 every 4-neighbour pair of present pixels
// passes the colour test (color_distance <= 1, color.h:17-24), so the greedy
// merge ends with exactly one blob per 4-connected component.  Here it is a
// union-find over runs of present pixels: LDS-local within tiles of 64
// columns, then a global merge across tile borders (atomicMin links, root =
// smallest row-major index), then flatten.  An image of one tile is done
// after the first.
#include "colour.h"
#include "common.h"
#include "../../include/atomorph_hip.h"
#include "scan.h"

#include <mutex>

using namespace amh;

namespace {

constexpr int TW = 64, TH = 32;      // CCL tile: a row is one wave
constexpr int kScanBlock = 1024;     // pixels per compaction block

// ----------------------------------------------------------------- ingest
// 1024 pixels per workgroup.  The few that float leaves unclear are listed and
// redone in double precision side by side: redone where they turn up, one of
// them held back most waves, 29 us for 2048x2048 pixels where this takes 26.
constexpr int kIngestPer = 4;

__global__ __launch_bounds__(256) void k_ingest(const uint32_t *__restrict__ rgba, int64_t n, int hsp,
                                                uint32_t *__restrict__ stored, uint32_t *__restrict__ shown) {
    __shared__ uint16_t at[256 * kIngestPer];
    __shared__ uint32_t unclear[256 * kIngestPer];  // (kept: a frame may be ingested in place)
    __shared__ int nunclear;
    const int64_t i0 = int64_t(blockIdx.x) * (256 * kIngestPer);
    const int tid = threadIdx.x;
    if (tid == 0) nunclear = 0;
    __syncthreads();
    uint32_t c[kIngestPer];
#pragma unroll
    for (int k = 0; k < kIngestPer; ++k) {
        const int64_t i = i0 + k * 256 + tid;
        c[k] = i < n ? rgba[i] : 0u;
    }
#pragma unroll
    for (int k = 0; k < kIngestPer; ++k) {
        const int64_t i = i0 + k * 256 + tid;
        if (i >= n) break;
        uint32_t st = 0, sh = 0;
        if ((c[k] >> 24) != 0) {
            st = sh = c[k];
            if (hsp && !(rgb_to_hsp_clear(c[k], &st) && hsp_to_rgb_clear(st, &sh))) {
                const int e = atomicAdd(&nunclear, 1);
                at[e] = uint16_t(k * 256 + tid);
                unclear[e] = c[k];
            }
        }
        if (stored) stored[i] = st;
        if (shown) shown[i] = sh;
    }
    __syncthreads();
    for (int e = tid; e < nunclear; e += 256) {
        const int64_t i = i0 + at[e];
        const uint32_t st = rgb_to_hsp(unclear[e]);
        if (stored) stored[i] = st;
        if (shown) shown[i] = hsp_to_rgb(st);
    }
}

// -------------------------------------------------------------- union-find
__device__ __forceinline__ int lds_find(int *L, int x) {
    int p = L[x];
    while (p != x) {
        x = p;
        p = L[x];
    }
    return x;
}
__device__ void lds_unite(int *L, int a, int b) {
    for (;;) {
        a = lds_find(L, a);
        b = lds_find(L, b);
        if (a == b) return;
        if (a < b) {
            const int old = atomicMin(&L[b], a);
            if (old == b) return;
            b = old;
        } else {
            const int old = atomicMin(&L[a], b);
            if (old == a) return;
            a = old;
        }
    }
}
__device__ __forceinline__ int g_load(const int *L, int x) {
    return __hip_atomic_load(L + x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ int g_find(int *L, int x) {
    int p = g_load(L, x);
    while (p != x) {
        x = p;
        p = g_load(L, x);
    }
    return x;
}
__device__ void g_unite(int *L, int a, int b) {
    for (;;) {
        a = g_find(L, a);
        b = g_find(L, b);
        if (a == b) return;
        if (a < b) {
            const int old = atomicMin(&L[b], a);
            if (old == b) return;
            b = old;
        } else {
            const int old = atomicMin(&L[a], b);
            if (old == a) return;
            a = old;
        }
    }
}

// First column of the run of mask m that holds column `lane`.
__device__ __forceinline__ int run_start(uint64_t m, int lane) {
    const uint64_t gap = ~m & ((1ull << lane) - 1ull);
    return gap ? 64 - __clzll(static_cast<long long>(gap)) : 0;
}

// A tile's labels.  Each row's presence mask is a ballot, so a pixel's run
// start needs no search, only run starts are union-find nodes, and two rows
// are united once per stretch of columns present in both: about 2 unions per
// run instead of 2 per pixel (2048^2, 1.5 M blob pixels: 72 us with every
// pixel a node in 64 x 16 tiles).
template <int ROWS, int NT>
__global__ __launch_bounds__(NT) void k_ccl_local(const uint32_t *__restrict__ rgba, int W, int H,
                                                           int *__restrict__ labels) {
    constexpr int kWaves = NT / 64, kPer = ROWS / kWaves;
    __shared__ int L[ROWS * TW];  // at run starts: the parent
    __shared__ uint64_t mask[ROWS];
    const int tx0 = blockIdx.x * TW, ty0 = blockIdx.y * ROWS;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, x = tx0 + lane;
    uint32_t c[kPer];
    for (int k = 0; k < kPer; ++k) {
        const int y = ty0 + wave + k * kWaves;
        c[k] = (x < W && y < H) ? rgba[int64_t(y) * W + x] : 0u;
    }
    for (int k = 0; k < kPer; ++k) {
        const int r = wave + k * kWaves;
        const bool fg = (c[k] >> 24) != 0;
        const uint64_t m = __ballot(fg);
        if (lane == 0) mask[r] = m;
        if (fg && run_start(m, lane) == lane) L[r * TW + lane] = r * TW + lane;
    }
    __syncthreads();
    for (int k = 0; k < kPer; ++k) {
        const int r = wave + k * kWaves;
        if (r == 0) continue;
        const uint64_t m = mask[r], up = mask[r - 1], both = m & up;
        if (((both & ~(both << 1)) >> lane) & 1u)
            lds_unite(L, r * TW + run_start(m, lane), (r - 1) * TW + run_start(up, lane));
    }
    __syncthreads();
    for (int k = 0; k < kPer; ++k) {
        const int r = wave + k * kWaves, y = ty0 + r;
        if (x >= W || y >= H) continue;
        int lab = -1;
        if ((c[k] >> 24) != 0) {
            const int root = lds_find(L, r * TW + run_start(mask[r], lane));
            lab = (ty0 + root / TW) * W + tx0 + root % TW;
        }
        labels[int64_t(y) * W + x] = lab;
    }
}

// Merge across the right and bottom edge of every tile, once per stretch of
// pairs present on both sides (the pairs of a stretch are united inside the
// tiles already).
__global__ __launch_bounds__(128) void k_ccl_merge(int W, int H, int *labels) {
    const int tiles_x = (W + TW - 1) / TW;
    const int tile = blockIdx.x;
    const int tx0 = (tile % tiles_x) * TW, ty0 = (tile / tiles_x) * TH;
    // threads 0..TH-1: right edge rows; TH..TH+TW-1: bottom edge columns
    const int t = threadIdx.x;
    int a, step, prev;  // the pair (a, a + step); the pair before it (a - prev, ...) in the tile, prev 0: none
    if (t < TH) {
        const int x = tx0 + TW - 1, y = ty0 + t;
        if (x + 1 >= W || y >= H) return;
        a = y * W + x;
        step = 1;
        prev = t > 0 ? W : 0;
    } else if (t < TH + TW) {
        const int x = tx0 + (t - TH), y = ty0 + TH - 1;
        if (x >= W || y + 1 >= H) return;
        a = y * W + x;
        step = W;
        prev = t > TH ? 1 : 0;
    } else {
        return;
    }
    // presence only: links never turn a label negative
    if (labels[a] < 0 || labels[a + step] < 0) return;
    if (prev && labels[a - prev] >= 0 && labels[a - prev + step] >= 0) return;
    g_unite(labels, a, a + step);
}

// Every pixel to its root.  The links are all in place, so what another
// pixel's thread may just have written is an ancestor too and cached reads do.
__global__ __launch_bounds__(256) void k_ccl_flatten(int64_t n, int *labels) {
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const auto load = [&](int64_t k) {
        return __hip_atomic_load(labels + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    };
    const int own = load(i);
    if (own < 0) return;
    int x = own, p = load(own);
    while (p != x) {
        x = p;
        p = load(x);
    }
    if (x != own) labels[i] = x;
}

// ------------------------------------------------------------ compaction
// Blob numbers follow the order of the components' smallest pixel index:
// count roots per block, scan, rank inside the block.
__global__ __launch_bounds__(256) void k_root_count(const int *__restrict__ labels, int64_t n,
                                                    int *__restrict__ bcount) {
    __shared__ int part[4];
    const int64_t base = int64_t(blockIdx.x) * kScanBlock;
    int cnt = 0;
    for (int l = threadIdx.x; l < kScanBlock; l += 256) {
        const int64_t i = base + l;
        if (i < n && labels[i] == int(i)) ++cnt;
    }
    for (int off = 32; off > 0; off >>= 1) cnt += __shfl_down(cnt, off, 64);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = cnt;
    __syncthreads();
    if (threadIdx.x == 0) bcount[blockIdx.x] = part[0] + part[1] + part[2] + part[3];
}

// Single-workgroup exclusive scan of nb ints into boff; total into boff[nb].
__global__ __launch_bounds__(1024) void k_scan_small(const int *__restrict__ in, int nb, int *__restrict__ out) {
    __shared__ int buf[1024];
    __shared__ int carry;
    if (threadIdx.x == 0) carry = 0;
    __syncthreads();
    for (int base = 0; base < nb; base += 1024) {
        const int i = base + threadIdx.x;
        int v = i < nb ? in[i] : 0;
        buf[threadIdx.x] = v;
        __syncthreads();
        for (int off = 1; off < 1024; off <<= 1) {
            const int t = threadIdx.x >= off ? buf[threadIdx.x - off] : 0;
            __syncthreads();
            buf[threadIdx.x] += t;
            __syncthreads();
        }
        if (i < nb) out[i] = carry + buf[threadIdx.x] - v;
        __syncthreads();
        if (threadIdx.x == 1023) carry += buf[1023];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[nb] = carry;
}

// Up to this many blocks each adds up the counts of the blocks before it
// itself (kSum; 32 loads per thread at most), without the scan's launch: a call
// on 8,192 blocks takes 49 us, on two more with the scan 52.
constexpr int kSumBlocks = 8192;
// Up to this many pixels one workgroup numbers the roots alone.  Calls of 64^2
// and 64 x 65 pixels take 17 us, the wait for the count; at this limit the one
// workgroup takes 20, the two launches past it 18.
constexpr int kOneCount = 16 * kScanBlock;

// Numbers the roots of pixels [blockIdx.x kScanBlock, ...): bcount holds the
// blocks' counts (kSum) or their scan; the last block writes the total to
// *total (host memory) and boff_total.
template <bool kSum>
__global__ __launch_bounds__(256) void k_root_ids(const int *__restrict__ labels, int64_t n,
                                                  const int *__restrict__ bcount, int *__restrict__ root_id,
                                                  int *__restrict__ boff_total, int *__restrict__ total) {
    __shared__ int wcount[4 * (kScanBlock / 256)];
    __shared__ int part[4];
    const int64_t base = int64_t(blockIdx.x) * kScanBlock;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int running;
    if (kSum) {
        int o = 0;
        for (int j = threadIdx.x; j < int(blockIdx.x); j += 256) o += bcount[j];
        for (int off = 32; off > 0; off >>= 1) o += __shfl_down(o, off, 64);
        if (lane == 0) part[wave] = o;
        __syncthreads();
        running = part[0] + part[1] + part[2] + part[3];
    } else {
        running = bcount[blockIdx.x];
    }
    // pass over the block in 4 chunks of 256; ranks in row-major order
    for (int chunk = 0; chunk < kScanBlock / 256; ++chunk) {
        const int64_t i = base + chunk * 256 + threadIdx.x;
        const bool root = i < n && labels[i] == int(i);
        const uint64_t ball = __ballot(root);
        const int below = __popcll(ball & ((1ull << lane) - 1ull));
        if (lane == 0) wcount[chunk * 4 + wave] = __popcll(ball);
        __syncthreads();
        int before = running;
        for (int w = 0; w < wave; ++w) before += wcount[chunk * 4 + w];
        if (root) root_id[i] = before + below;
        running += wcount[chunk * 4 + 0] + wcount[chunk * 4 + 1] + wcount[chunk * 4 + 2] + wcount[chunk * 4 + 3];
    }
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) {
        *boff_total = running;
        if (total) __hip_atomic_store(total, running, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// The same by one workgroup (n <= kOneCount), no counts needed.
__global__ __launch_bounds__(1024) void k_root_ids_one(const int *__restrict__ labels, int n, int *__restrict__ root_id,
                                                       int *__restrict__ boff_total, int *__restrict__ total) {
    constexpr int kChunks = kOneCount / 1024;
    __shared__ int wcount[kChunks][16];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint64_t ball[kChunks];
    for (int k = 0; k < kChunks; ++k) {
        const int i = k * 1024 + int(threadIdx.x);
        ball[k] = __ballot(i < n && labels[i] == i);
        if (lane == 0) wcount[k][wave] = __popcll(ball[k]);
    }
    __syncthreads();
    int running = 0;
    for (int k = 0; k < kChunks; ++k) {
        int before = running;
        for (int w = 0; w < 16; ++w) {
            before += w < wave ? wcount[k][w] : 0;
            running += wcount[k][w];
        }
        if ((ball[k] >> lane) & 1u)
            root_id[k * 1024 + threadIdx.x] = before + __popcll(ball[k] & ((1ull << lane) - 1ull));
    }
    if (threadIdx.x == 0) {
        *boff_total = running;
        if (total) __hip_atomic_store(total, running, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// Words of pinned host memory that a kernel writes a result into: one page
// for the process, a slot held from the launch to the wait.  slot() < 0 when
// all are held or there is none (then the result is copied).
class HostWords {
    static constexpr int kSlots = 64, kStride = 16;  // 64-byte slots
    std::mutex mu;
    int *page = nullptr;
    uint64_t held = 0;
    bool tried = false;

  public:
    int slot() {
        std::lock_guard<std::mutex> lk(mu);
        if (!tried) {
            tried = true;
            void *p = nullptr;
            if (hipHostMalloc(&p, kSlots * kStride * sizeof(int), hipHostMallocPortable | hipHostMallocMapped) == hipSuccess)
                page = static_cast<int *>(p);
            else
                (void)hipGetLastError();
        }
        if (!page || held == ~0ull) return -1;
        const int k = __builtin_ctzll(~held);
        held |= 1ull << k;
        return k;
    }
    volatile int *word(int k) { return page + k * kStride; }
    void release(int k) {
        std::lock_guard<std::mutex> lk(mu);
        held &= ~(1ull << k);
    }
};
HostWords g_words;

// Per-blob sums in two levels: each block covers a tile of 64 columns, one
// wave per row.  A row's stretches of one blob are summed across the lanes
// (colours as packed prefix sums, positions in closed form) and each adds one
// entry into a small open-addressed LDS table of the tile's blobs, which is
// then flushed with one set of global atomics per (tile, blob).  Device
// atomics on this GPU are performed past the L2: square tiles meet few blobs,
// so there are few flushes (2048^2, 1,200 blobs: 97 us with bands of 4,096
// consecutive pixels and an entry per pixel).
constexpr int kStatSlots = 256;
constexpr int kStatRows = 32;  // of a tile; an image of one tile: up to 64

struct StatTable {  // sums within the tile
    int key[kStatSlots];
    uint32_t sum[7][kStatSlots];  // count, x, y, c0..c3
    int box[4][kStatSlots];       // x1 y1 x2 y2
};

// Slot of blob b in the table (inserting it), or -1 when the table is full.
__device__ __forceinline__ int stat_slot(StatTable &T, int b) {
    int h = int((uint32_t(b) * 2654435761u) >> 24);  // 8 bits: [0, 256)
    for (int probe = 0; probe < kStatSlots; ++probe) {
        const int k = atomicCAS(&T.key[h], -1, b);
        if (k == -1 || k == b) return h;
        h = (h + 1) & (kStatSlots - 1);
    }
    return -1;
}

// Adds v (count, x, y, c0..c3 within the tile at x0, y0) to blob b's totals.
__device__ __forceinline__ void stat_add_global(amh_blob_stat *p, const uint32_t v[7], int x0, int y0, int x1, int y1,
                                                int x2, int y2) {
    using u64 = unsigned long long;
    atomicAdd((u64 *)&p->count, u64(v[0]));
    atomicAdd((u64 *)&p->sum_x, u64(v[0]) * u64(x0) + v[1]);
    atomicAdd((u64 *)&p->sum_y, u64(v[0]) * u64(y0) + v[2]);
    for (int k = 0; k < 4; ++k) atomicAdd((u64 *)&p->sum_c[k], u64(v[3 + k]));
    atomicMin(&p->x1, x0 + x1);
    atomicMin(&p->y1, y0 + y1);
    atomicMax(&p->x2, x0 + x2);
    atomicMax(&p->y2, y0 + y2);
}

__device__ __forceinline__ void stat_init(amh_blob_stat &z) {
    z.count = z.sum_x = z.sum_y = 0;
    z.sum_c[0] = z.sum_c[1] = z.sum_c[2] = z.sum_c[3] = 0;
    z.x1 = z.y1 = 0x7FFFFFFF;
    z.x2 = z.y2 = -1;
    z.first = -1;
}

// Inclusive sum over the wave's lanes.
template <int CTRL, int ROWS>
__device__ __forceinline__ uint32_t dpp_add(uint32_t v) {
    return v + uint32_t(__builtin_amdgcn_update_dpp(0, int(v), CTRL, ROWS, 0xF, false));
}
__device__ __forceinline__ uint32_t wave_prefix(uint32_t v) {
    v = dpp_add<0x111, 0xF>(v);
    v = dpp_add<0x112, 0xF>(v);
    v = dpp_add<0x114, 0xF>(v);
    v = dpp_add<0x118, 0xF>(v);
    v = dpp_add<0x142, 0xA>(v);  // lane 15 -> row 1, lane 47 -> row 3
    return dpp_add<0x143, 0xC>(v);  // lane 31 -> rows 2 and 3
}

// init: the only block starts the totals itself.
template <int NT>
__global__ __launch_bounds__(NT) void k_blob_stats(const int *__restrict__ labels,
                                                             const uint32_t *__restrict__ stored, int W, int H,
                                                             int rows, const int *__restrict__ root_id,
                                                             int *__restrict__ bop, amh_blob_stat *__restrict__ st,
                                                             int nblobs, bool init) {
    __shared__ StatTable T;
    for (int h = threadIdx.x; h < kStatSlots; h += NT) {
        T.key[h] = -1;
        for (int k = 0; k < 7; ++k) T.sum[k][h] = 0u;
        T.box[0][h] = T.box[1][h] = 0x7FFFFFFF;
        T.box[2][h] = T.box[3][h] = -1;
    }
    if (init) {
        for (int b = threadIdx.x; b < nblobs; b += NT) stat_init(st[b]);
        __threadfence();
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int x0 = int(blockIdx.x) * 64, y0 = int(blockIdx.y) * rows, x = x0 + lane;
    constexpr int kWaves = NT / 64;
    constexpr int kBatch = 2 * kStatRows / kWaves < 8 ? 2 * kStatRows / kWaves : 8;  // rows of a wave loaded together
    for (int r0 = wave; r0 < rows; r0 += kBatch * kWaves) {
        int lab[kBatch], blob[kBatch];
        uint32_t col[kBatch];
        for (int k = 0; k < kBatch; ++k) {
            const int r = r0 + kWaves * k, y = y0 + r;
            const bool in = r < rows && x < W && y < H;
            const int64_t i = in ? int64_t(y) * W + x : 0;
            const int l = labels[i];
            col[k] = stored[i];
            lab[k] = in ? l : -1;
        }
        for (int k = 0; k < kBatch; ++k) blob[k] = root_id[max(lab[k], 0)];
        for (int k = 0; k < kBatch; ++k) {
            const int r = r0 + kWaves * k, y = y0 + r;
            if (r >= rows) break;  // uniform over the wave
            const int b = lab[k] >= 0 ? blob[k] : -1;
            if (x < W && y < H) bop[int64_t(y) * W + x] = b;
            if (lab[k] >= 0 && lab[k] == y * W + x) st[b].first = lab[k];
            if (!__any(b >= 0)) continue;
            const int before = __builtin_amdgcn_update_dpp(-2, b, 0x138, 0xF, 0xF, false);  // lane - 1
            const int after = __builtin_amdgcn_update_dpp(-2, b, 0x130, 0xF, 0xF, false);   // lane + 1
            const uint64_t heads = __ballot(lane == 0 || before != b) & ((2ull << lane) - 1ull);
            const int s = 63 - __clzll(static_cast<long long>(heads));
            const uint32_t c = b >= 0 ? col[k] : 0u;
            // two channels per word: 64 x 255 < 2^16
            const uint32_t rb = wave_prefix(c & 0x00FF00FFu), ga = wave_prefix((c >> 8) & 0x00FF00FFu);
            const uint32_t rb0 = uint32_t(__shfl(int(rb), max(s - 1, 0), 64));
            const uint32_t ga0 = uint32_t(__shfl(int(ga), max(s - 1, 0), 64));
            if (b < 0 || !(lane == 63 || after != b)) continue;  // the last lane of each stretch adds it
            const uint32_t drb = rb - (s > 0 ? rb0 : 0u), dga = ga - (s > 0 ? ga0 : 0u), len = uint32_t(lane - s + 1);
            const uint32_t v[7] = {len, len * uint32_t(s + lane) / 2, len * uint32_t(r), drb & 0xFFFFu, dga & 0xFFFFu,
                                   drb >> 16, dga >> 16};
            const int h = stat_slot(T, b);
            if (h < 0) {  // more blobs in the tile than slots: straight to memory
                stat_add_global(st + b, v, x0, y0, s, r, lane, r);
                continue;
            }
            for (int q = 0; q < 7; ++q) atomicAdd(&T.sum[q][h], v[q]);
            atomicMin(&T.box[0][h], s);
            atomicMin(&T.box[1][h], r);
            atomicMax(&T.box[2][h], lane);
            atomicMax(&T.box[3][h], r);
        }
    }
    __syncthreads();
    for (int h = threadIdx.x; h < kStatSlots; h += NT) {
        const int b = T.key[h];
        if (b < 0) continue;
        uint32_t v[7];
        for (int k = 0; k < 7; ++k) v[k] = T.sum[k][h];
        stat_add_global(st + b, v, x0, y0, T.box[0][h], T.box[1][h], T.box[2][h], T.box[3][h]);
    }
}

__global__ void k_stats_init(amh_blob_stat *st, int nb) {
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b < nb) stat_init(st[b]);
}

// ----------------------------------------------------- grouping by blob
// Stable counting sort of pixel indices by blob number.  Per band of kBand
// consecutive pixels and blob: the count (k_group_hist), its scan along the
// bands (k_group_colscan; the table is blob-major, so a blob's bands are
// consecutive), the blobs' starts (k_first_scan), and the placing
// (k_group_scatter).  A band's blobs are looked up in an LDS table with room
// for as many as it has pixels; a wave's equal blobs are grouped with ballots
// first.  (2048^2, 1,200 blobs: 250 us with a block-major table of
// 1,024-pixel bands, device atomics per pixel and one wave placing each
// band.)
constexpr int kBand = 2048, kBandT = 256;
constexpr int kBandPer = kBand / kBandT;  // 64-pixel chunks per wave, consecutive

struct BandTable {
    int key[kBand];
    __device__ __forceinline__ int slot(int b) {
        int h = int((uint32_t(b) * 2654435761u) >> 21);  // 11 bits: [0, kBand)
        for (;;) {  // at most kBand different blobs: there is always a place
            const int k = atomicCAS(&key[h], -1, b);
            if (k == -1 || k == b) return h;
            h = (h + 1) & (kBand - 1);
        }
    }
};
static_assert(kBand == 1 << 11, "slot() takes 11 bits");

// The lanes of the wave with this lane's b: their first, their number and
// this lane's rank among them (b < 0: alone, 0, 0).
struct SameLanes {
    int lead, total, rank;
};
__device__ __forceinline__ SameLanes same_lanes(int b) {
    const int lane = threadIdx.x & 63;
    SameLanes s = {lane, 0, 0};
    uint64_t todo = __ballot(b >= 0);
    while (todo) {
        const int leader = __ffsll((unsigned long long)todo) - 1;
        const uint64_t same = __ballot(b == __builtin_amdgcn_readlane(b, leader));
        if ((same >> lane) & 1u) {
            s.lead = leader;
            s.total = int(__popcll(same));
            s.rank = int(__popcll(same & ((1ull << lane) - 1ull)));
        }
        todo &= ~same;
    }
    return s;
}

__global__ __launch_bounds__(256) void k_group_zero(int *__restrict__ p, int64_t n) {
    const int64_t stride = int64_t(gridDim.x) * 256;
    for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < n; i += stride) p[i] = 0;
}

__global__ __launch_bounds__(kBandT) void k_group_hist(const int *__restrict__ bop, int64_t n, int nbands,
                                                       int *__restrict__ hist) {
    __shared__ BandTable T;
    __shared__ int cnt[kBand];
    for (int k = threadIdx.x; k < kBand; k += kBandT) {
        T.key[k] = -1;
        cnt[k] = 0;
    }
    __syncthreads();
    int b[kBandPer];
    for (int j = 0; j < kBandPer; ++j) {
        const int64_t i = int64_t(blockIdx.x) * kBand + j * kBandT + threadIdx.x;
        b[j] = i < n ? bop[i] : -1;
    }
    for (int j = 0; j < kBandPer; ++j) {
        const SameLanes s = same_lanes(b[j]);
        if (s.total > 0 && s.rank == 0) atomicAdd(&cnt[T.slot(b[j])], s.total);
    }
    __syncthreads();
    for (int k = threadIdx.x; k < kBand; k += kBandT)
        if (T.key[k] >= 0) hist[int64_t(T.key[k]) * nbands + blockIdx.x] = cnt[k];
}

// One workgroup per blob: hist[b][band] becomes the number of b's pixels in
// earlier bands, and count[b] the blob's total.
__global__ __launch_bounds__(256) void k_group_colscan(int *__restrict__ hist, int nbands,
                                                       int64_t *__restrict__ count) {
    __shared__ int wsum[4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int *row = hist + int64_t(blockIdx.x) * nbands;
    int carry = 0;
    for (int base = 0; base < nbands; base += 256) {
        const int k = base + int(threadIdx.x);
        const int v = k < nbands ? row[k] : 0;
        const int incl = int(wave_prefix(uint32_t(v)));
        if (lane == 63) wsum[wave] = incl;
        __syncthreads();
        int before = carry;
        for (int w = 0; w < wave; ++w) before += wsum[w];
        if (k < nbands) row[k] = before + incl - v;
        carry += wsum[0] + wsum[1] + wsum[2] + wsum[3];
        __syncthreads();
    }
    if (threadIdx.x == 0) count[blockIdx.x] = carry;
}

// Blob starts: exclusive scan of the counts in place, first[nblobs] = total.
__global__ __launch_bounds__(1024) void k_first_scan(int nblobs, int64_t *__restrict__ first) {
    __shared__ int64_t wsum[16];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int64_t carry = 0;
    for (int base = 0; base < nblobs; base += 1024) {
        const int b = base + int(threadIdx.x);
        const int64_t cnt = b < nblobs ? first[b] : 0;
        int64_t incl = cnt;
        for (int off = 1; off < 64; off <<= 1) {
            const int64_t t = __shfl_up(incl, off, 64);
            if (lane >= off) incl += t;
        }
        if (lane == 63) wsum[wave] = incl;
        __syncthreads();
        int64_t before = carry;
        for (int w = 0; w < 16; ++w) {
            before += w < wave ? wsum[w] : 0;
            carry += wsum[w];
        }
        if (b < nblobs) first[b] = before + incl - cnt;
        __syncthreads();
    }
    if (threadIdx.x == 0) first[nblobs] = carry;
}

// A band's pixels into the list.  Each wave takes consecutive pixels; its
// blobs' places follow the counts of the waves before it, so the order is the
// pixels'.
__global__ __launch_bounds__(kBandT) void k_group_scatter(const int *__restrict__ bop, int64_t n, int nbands,
                                                          const int *__restrict__ hist,
                                                          const int64_t *__restrict__ first, int *__restrict__ list) {
    __shared__ BandTable T;
    __shared__ uint32_t cnt[2][kBand];  // 16 bits per wave: counts, then running places
    __shared__ int64_t start[kBand];
    for (int k = threadIdx.x; k < kBand; k += kBandT) {
        T.key[k] = -1;
        cnt[0][k] = cnt[1][k] = 0u;
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t w0 = int64_t(blockIdx.x) * kBand + wave * (64 * kBandPer);
    uint32_t *const mine = cnt[wave / 2];
    const int shift = 16 * (wave & 1);
    int b[kBandPer], slot[kBandPer];
    SameLanes s[kBandPer];
    for (int j = 0; j < kBandPer; ++j) {
        const int64_t i = w0 + 64 * j + lane;
        b[j] = i < n ? bop[i] : -1;
    }
    for (int j = 0; j < kBandPer; ++j) {
        s[j] = same_lanes(b[j]);
        slot[j] = -1;
        if (s[j].total > 0 && s[j].rank == 0) {
            slot[j] = T.slot(b[j]);
            atomicAdd(&mine[slot[j]], uint32_t(s[j].total) << shift);
        }
    }
    __syncthreads();
    for (int k = threadIdx.x; k < kBand; k += kBandT) {
        const int key = T.key[k];
        if (key < 0) continue;
        start[k] = first[key] + hist[int64_t(key) * nbands + blockIdx.x];
        const uint32_t c01 = cnt[0][k], c23 = cnt[1][k];
        const uint32_t c0 = c01 & 0xFFFFu, c1 = c01 >> 16, c2 = c23 & 0xFFFFu;
        cnt[0][k] = c0 << 16;
        cnt[1][k] = (c0 + c1) | ((c0 + c1 + c2) << 16);
    }
    __syncthreads();
    for (int j = 0; j < kBandPer; ++j) {
        int64_t at = 0;
        if (slot[j] >= 0) {
            const uint32_t old = atomicAdd(&mine[slot[j]], uint32_t(s[j].total) << shift);
            at = start[slot[j]] + ((old >> shift) & 0xFFFFu);
        }
        at = __shfl(at, s[j].lead, 64);
        if (b[j] >= 0) list[at + s[j].rank] = int(w0 + 64 * j + lane);
    }
}

// The whole grouping by one workgroup: few pixels and blobs, the counts per
// wave and blob in LDS.  Five launches cost more than the work here: 4,096
// pixels of 10 blobs take 8 us, 4,097 take 23; of 1,024 blobs 32 us, one pixel or
// blob more 70.  (More blobs than this do not fit the LDS.)
constexpr int kOnePixels = 4096, kOneBlobs = 1024, kOneT = 1024, kOneWaves = kOneT / 64;

__global__ __launch_bounds__(kOneT) void k_group_one(const int *__restrict__ bop, int n, int nblobs,
                                                     int64_t *__restrict__ first, int *__restrict__ list) {
    __shared__ int cnt[kOneWaves][kOneBlobs];
    __shared__ int wsum[kOneWaves];
    constexpr int kPer = kOnePixels / kOneT;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, w0 = wave * (64 * kPer);
    for (int k = threadIdx.x; k < kOneWaves * kOneBlobs; k += kOneT) (&cnt[0][0])[k] = 0;
    int b[kPer];
    SameLanes s[kPer];
    for (int j = 0; j < kPer; ++j) {
        const int i = w0 + 64 * j + lane;
        b[j] = i < n ? bop[i] : -1;
    }
    __syncthreads();
    for (int j = 0; j < kPer; ++j) {
        s[j] = same_lanes(b[j]);
        // (this wave's own counts, by another lane in the next turn)
        if (s[j].total > 0 && s[j].rank == 0) cnt[wave][b[j]] += s[j].total;
        wave_order();
    }
    __syncthreads();
    {   // thread b: blob b's total, its start, and each wave's first place
        const int k = int(threadIdx.x);
        int c[kOneWaves], total = 0;
        for (int w = 0; w < kOneWaves; ++w) {
            c[w] = k < nblobs ? cnt[w][k] : 0;
            total += c[w];
        }
        const int incl = int(wave_prefix(uint32_t(total)));
        if (lane == 63) wsum[wave] = incl;
        __syncthreads();
        int at = incl - total, all = 0;
        for (int w = 0; w < kOneWaves; ++w) {
            at += w < wave ? wsum[w] : 0;
            all += wsum[w];
        }
        if (k < nblobs) {
            first[k] = at;
            for (int w = 0; w < kOneWaves; ++w) {
                cnt[w][k] = at;
                at += c[w];
            }
        }
        if (k == 0) first[nblobs] = all;
    }
    __syncthreads();
    for (int j = 0; j < kPer; ++j) {
        int at = 0;
        if (s[j].total > 0 && s[j].rank == 0) {
            at = cnt[wave][b[j]];
            cnt[wave][b[j]] = at + s[j].total;
        }
        wave_order();
        at = __shfl(at, s[j].lead, 64);
        if (b[j] >= 0) list[at + s[j].rank] = w0 + 64 * j + lane;
    }
}

// Grouping with many blobs: a stable LSD radix sort of the pixels by blob
// number (8-bit digits, as many passes as the blob numbers need), so the
// memory is O(pixels + blobs) whatever the blob count.  Pixels without a
// blob get key nblobs and sort last.  Per pass: a digit histogram per block
// of kGrpTile pixels, an exclusive scan of the digit-major histograms, and a
// scatter that ranks equal digits in pixel order with ballots (stable).
constexpr int kGrpTile = 256 * 8;

__device__ __forceinline__ uint32_t grp_key(bool from_bop, const int *__restrict__ bop,
                                            const uint32_t *__restrict__ kin, int64_t e, int nblobs) {
    if (!from_bop) return kin[e];
    const int b = bop[e];
    return b >= 0 ? uint32_t(b) : uint32_t(nblobs);
}

__global__ __launch_bounds__(256) void k_grp_hist(bool from_bop, const int *__restrict__ bop,
                                                  const uint32_t *__restrict__ kin, int64_t n, int nblobs, int shift,
                                                  int nblk, int *__restrict__ hist) {
    __shared__ int h[256];
    h[threadIdx.x] = 0;
    __syncthreads();
    const int64_t b0 = int64_t(blockIdx.x) * kGrpTile;
    for (int j = 0; j < kGrpTile / 256; ++j) {
        const int64_t e = b0 + j * 256 + threadIdx.x;
        if (e < n) atomicAdd(&h[(grp_key(from_bop, bop, kin, e, nblobs) >> shift) & 255u], 1);
    }
    __syncthreads();
    hist[int64_t(threadIdx.x) * nblk + blockIdx.x] = h[threadIdx.x];
}

// Stable scatter of one pass.  `last`: values go to `list` and only those of
// real blobs (their places are below the number of blob pixels).
__global__ __launch_bounds__(256) void k_grp_scatter(bool from_bop, const int *__restrict__ bop,
                                                     const uint32_t *__restrict__ kin,
                                                     const int32_t *__restrict__ vin, int64_t n, int nblobs,
                                                     int shift, int nblk, const int *__restrict__ off, bool last,
                                                     uint32_t *__restrict__ kout, int32_t *__restrict__ vout) {
    __shared__ int base[256];
    __shared__ int cnt[4][256];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    base[t] = off[int64_t(t) * nblk + blockIdx.x];
    const uint64_t below = (1ull << lane) - 1ull;
    const int64_t b0 = int64_t(blockIdx.x) * kGrpTile;
    for (int j = 0; j < kGrpTile / 256; ++j) {
        for (int w = 0; w < 4; ++w) cnt[w][t] = 0;
        __syncthreads();
        const int64_t e = b0 + j * 256 + t;
        const bool ok = e < n;
        const uint32_t k = ok ? grp_key(from_bop, bop, kin, e, nblobs) : 0u;
        const int32_t v = ok ? (from_bop ? int32_t(e) : vin[e]) : 0;
        const int d = int((k >> shift) & 255u);
        uint64_t same = __ballot(ok);
        for (int bit = 0; bit < 8; ++bit) {
            const uint64_t bb = __ballot((d >> bit) & 1);
            same &= ((d >> bit) & 1) ? bb : ~bb;
        }
        const int rank = int(__popcll(same & below));
        if (ok && rank == 0) cnt[wave][d] = int(__popcll(same));
        __syncthreads();
        int before = 0;
        for (int w = 0; w < wave; ++w) before += cnt[w][d];
        if (ok) {
            const int pos = base[d] + before + rank;
            if (!last) {
                kout[pos] = k;
                vout[pos] = v;
            } else if (k < uint32_t(nblobs)) {
                kout[pos] = k;
                vout[pos] = v;
            }
        }
        __syncthreads();
        int tot = 0;
        for (int w = 0; w < 4; ++w) tot += cnt[w][t];
        base[t] += tot;
        __syncthreads();
    }
}

// Per blob, from the sorted keys of its pixels (places [0, *total)): the
// start and end of its run; absent blobs keep start = end = 0.
__global__ void k_grp_bounds_total(const uint32_t *__restrict__ key, const unsigned long long *__restrict__ ptotal,
                                   int *__restrict__ start, int *__restrict__ end) {
    const int64_t p = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    const int64_t total = int64_t(*ptotal);
    if (p >= total) return;
    const uint32_t k = key[p];
    if (p == 0 || key[p - 1] != k) start[k] = int(p);
    if (p == total - 1 || key[p + 1] != k) end[k] = int(p + 1);
}

__global__ void k_grp_counts(const int *__restrict__ start, const int *__restrict__ end, int nblobs,
                             int64_t *__restrict__ count) {
    const int b = int(blockIdx.x) * blockDim.x + threadIdx.x;
    if (b < nblobs) count[b] = end[b] - start[b];
}

// Counts the pixels that have a blob.
__global__ void k_grp_present(const int *__restrict__ bop, int64_t n, unsigned long long *__restrict__ total) {
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    const bool has = i < n && bop[i] >= 0;
    const uint64_t m = __ballot(has);
    if ((threadIdx.x & 63) == 0 && m) atomicAdd(total, (unsigned long long)__popcll(m));
}

struct GroupLayout {
    bool radix;
    int nblk;                   // table: pixel bands; radix: sort tiles
    int passes;
    size_t hist, k0, v0, k1, v1, hoff, sums, offs, start, end, total, bytes;
};

GroupLayout group_layout(int64_t n, int64_t nblobs) {
    GroupLayout L{};
    auto al = [](size_t v) { return (v + 255) & ~size_t(255); };
    const int64_t tblk = (n + kBand - 1) / kBand;
    const int64_t nb = nblobs > 0 ? nblobs : 1;
    // the per-(blob, band) table when it is at most 2 ints per pixel
    if (tblk * nb <= 2 * std::max<int64_t>(n, 1)) {
        L.radix = false;
        L.nblk = int(tblk);
        L.bytes = size_t(tblk) * size_t(nb) * sizeof(int);
        return L;
    }
    L.radix = true;
    L.nblk = int((n + kGrpTile - 1) / kGrpTile);
    int bits = 1;
    while ((int64_t(1) << bits) <= nblobs) ++bits;  // keys 0..nblobs
    L.passes = (bits + 7) / 8;
    const size_t hn = size_t(256) * size_t(std::max(L.nblk, 1));
    size_t o = 0;
    L.k0 = o; o = al(o + size_t(n) * 4);
    L.v0 = o; o = al(o + size_t(n) * 4);
    L.k1 = o; o = al(o + size_t(n) * 4);
    L.v1 = o; o = al(o + size_t(n) * 4);
    L.hist = o; o = al(o + hn * 4);
    L.hoff = o; o = al(o + (hn + 1) * 4);
    L.sums = o; o = al(o + size_t(scan::blocks(int64_t(hn))) * 4);
    L.offs = o; o = al(o + (size_t(scan::blocks(int64_t(hn))) + 1) * 4);
    L.start = o; o = al(o + size_t(nb) * 4);
    L.end = o; o = al(o + size_t(nb) * 4);
    L.total = o; o = al(o + 8);
    L.bytes = o;
    return L;
}

int group_radix(const GroupLayout &L, const int32_t *bop, int64_t n, int nblobs, char *ws, int64_t *first,
                int32_t *list, hipStream_t s) {
    uint32_t *k[2] = {reinterpret_cast<uint32_t *>(ws + L.k0), reinterpret_cast<uint32_t *>(ws + L.k1)};
    int32_t *v[2] = {reinterpret_cast<int32_t *>(ws + L.v0), reinterpret_cast<int32_t *>(ws + L.v1)};
    int *hist = reinterpret_cast<int *>(ws + L.hist), *hoff = reinterpret_cast<int *>(ws + L.hoff);
    int *sums = reinterpret_cast<int *>(ws + L.sums), *offs = reinterpret_cast<int *>(ws + L.offs);
    int *start = reinterpret_cast<int *>(ws + L.start), *end = reinterpret_cast<int *>(ws + L.end);
    unsigned long long *total = reinterpret_cast<unsigned long long *>(ws + L.total);
    const int64_t hn = int64_t(256) * L.nblk;
    int cur = 0;
    for (int p = 0; p < L.passes; ++p) {
        const bool from_bop = p == 0, last = p + 1 == L.passes;
        hipLaunchKernelGGL(k_grp_hist, dim3(uint32_t(L.nblk)), dim3(256), 0, s, from_bop, bop, k[cur], n, nblobs,
                           8 * p, L.nblk, hist);
        scan::exclusive(hist, hn, sums, offs, hoff, s);
        hipLaunchKernelGGL(k_grp_scatter, dim3(uint32_t(L.nblk)), dim3(256), 0, s, from_bop, bop, k[cur], v[cur], n,
                           nblobs, 8 * p, L.nblk, hoff, last, k[cur ^ 1], last ? list : v[cur ^ 1]);
        cur ^= 1;
    }
    // runs of the sorted keys -> counts -> first[] (exclusive scan)
    if (int r = check_hip(hipMemsetAsync(ws + L.start, 0, L.total + 8 - L.start, s), "amh_group_pixels memset"))
        return r;
    const uint32_t gn = uint32_t((n + 255) / 256);
    hipLaunchKernelGGL(k_grp_present, dim3(gn), dim3(256), 0, s, bop, n, total);
    // the blob pixels are the first `total` places; bounds over all n places
    // would read the keys of blobless pixels, which the last pass skipped
    hipLaunchKernelGGL(k_grp_bounds_total, dim3(gn), dim3(256), 0, s, k[cur], total, start, end);
    hipLaunchKernelGGL(k_grp_counts, dim3(uint32_t((nblobs + 255) / 256)), dim3(256), 0, s, start, end, nblobs,
                       first);
    return AMH_OK;
}

// ------------------------------------------------------------ chain build
// Row y of every chain (thread.cpp:803-848).
__global__ void k_build_row(int y, int h, int64_t wtot, int nchains, const int64_t *__restrict__ off,
                            const int32_t *__restrict__ cw, const int32_t *__restrict__ cblob,
                            const uint32_t *__restrict__ exy, const int32_t *__restrict__ plist,
                            const int64_t *__restrict__ bfirst, int W, uint64_t seed,
                            uint64_t *__restrict__ pts) {
    const int64_t a = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (a >= wtot) return;
    int lo = 0, hi = nchains - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (off[mid] <= a) lo = mid; else hi = mid - 1;
    }
    const int c = lo;
    const int64_t x = a - off[c];
    const int b = cblob[int64_t(c) * h + y];
    int64_t n;
    int64_t first = 0;
    if (b >= 0) {
        first = bfirst[b];
        n = bfirst[b + 1] - first;
    } else {
        n = 1;
    }
    uint64_t pt;
    if (x < n) {
        if (b >= 0) {
            const int p = plist[first + x];
            pt = make_pt(uint32_t(p % W), uint32_t(p / W), 0, 0, HAS_PIXEL | HAS_FLUID);
        } else {
            const uint32_t e = exy[int64_t(c) * h + y];
            pt = make_pt(e & 0xFFFFu, e >> 16, 0, 0, HAS_FLUID);
        }
    } else {
        // duplicate of a shuffled copy (thread.cpp:837-848)
        const uint64_t key = mix64(seed ^ (uint64_t(c) << 32) ^ uint64_t(y));
        const uint32_t q = feistel_perm(uint32_t(x % n), uint32_t(n), key);
        uint32_t px, py, fl;
        if (b >= 0) {
            const int p = plist[first + q];
            px = uint32_t(p % W);
            py = uint32_t(p / W);
            fl = HAS_PIXEL;
        } else {
            const uint32_t e = exy[int64_t(c) * h + y];
            px = e & 0xFFFFu;
            py = e >> 16;
            fl = 0;
        }
        const uint64_t r = mix64(key ^ (uint64_t(x) * 0x9E3779B97F4A7C15ull));
        pt = make_pt(px, py, uint32_t(r & 255u), uint32_t((r >> 8) & 255u), fl);
    }
    pts[int64_t(y) * wtot + a] = pt;
}

int check_frame(int32_t W, int32_t H, const char *what) {
    if (W <= 0 || H <= 0 || W > 65535 || H > 65535 || int64_t(W) * H >= (int64_t(1) << 31)) {
        set_error("%s: invalid frame size %dx%d", what, W, H);
        return AMH_E_ARG;
    }
    return AMH_OK;
}

}  // namespace

extern "C" int amh_ingest_frame(const uint32_t *rgba, int32_t W, int32_t H, int32_t hsp, uint32_t *stored,
                                uint32_t *shown, void *stream) {
    if (int r = check_frame(W, H, "amh_ingest_frame")) return r;
    if (!rgba || (!stored && !shown)) {
        set_error("amh_ingest_frame: NULL buffer");
        return AMH_E_ARG;
    }
    const int64_t n = int64_t(W) * H;
    hipLaunchKernelGGL(k_ingest, dim3(uint32_t((n + 256 * kIngestPer - 1) / (256 * kIngestPer))), dim3(256), 0,
                       static_cast<hipStream_t>(stream), rgba, n, hsp, stored, shown);
    AMH_LAUNCH_CHECK("amh_ingest_frame");
    return AMH_OK;
}

extern "C" int amh_segment(const uint32_t *rgba, int32_t W, int32_t H, int32_t *labels, void *stream) {
    if (int r = check_frame(W, H, "amh_segment")) return r;
    if (!rgba || !labels) {
        set_error("amh_segment: NULL buffer");
        return AMH_E_ARG;
    }
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (W <= TW && H <= 2 * TH) {  // one tile: its labels are final
        hipLaunchKernelGGL((k_ccl_local<2 * TH, 1024>), dim3(1), dim3(1024), 0, s, rgba, W, H, labels);
        AMH_LAUNCH_CHECK("amh_segment");
        return AMH_OK;
    }
    const int tx = (W + TW - 1) / TW, ty = (H + TH - 1) / TH;
    hipLaunchKernelGGL((k_ccl_local<TH, 512>), dim3(tx, ty), dim3(512), 0, s, rgba, W, H, labels);
    hipLaunchKernelGGL(k_ccl_merge, dim3(tx * ty), dim3(128), 0, s, W, H, labels);
    const int64_t n = int64_t(W) * H;
    hipLaunchKernelGGL(k_ccl_flatten, dim3(uint32_t((n + 255) / 256)), dim3(256), 0, s, n, labels);
    AMH_LAUNCH_CHECK("amh_segment");
    return AMH_OK;
}

extern "C" size_t amh_blob_workspace_bytes(int32_t W, int32_t H) {
    const int64_t n = int64_t(W) * H;
    const int64_t nb = (n + kScanBlock - 1) / kScanBlock;
    return size_t(n) * sizeof(int) + size_t(2 * nb + 2) * sizeof(int);
}

extern "C" int amh_blob_count(const int32_t *labels, int32_t W, int32_t H, void *ws, int32_t *nblobs, void *stream) {
    if (int r = check_frame(W, H, "amh_blob_count")) return r;
    if (!labels || !ws || !nblobs) {
        set_error("amh_blob_count: NULL argument");
        return AMH_E_ARG;
    }
    hipStream_t s = static_cast<hipStream_t>(stream);
    const int64_t n = int64_t(W) * H;
    const int nb = int((n + kScanBlock - 1) / kScanBlock);
    int *root_id = static_cast<int *>(ws);
    int *bcount = root_id + n;
    int *boff = bcount + nb;
    const int slot = g_words.slot();
    struct Release {
        int slot;
        ~Release() {
            if (slot >= 0) g_words.release(slot);
        }
    } release{slot};
    int *const word = slot >= 0 ? const_cast<int *>(g_words.word(slot)) : nullptr;
    if (n <= kOneCount) {
        hipLaunchKernelGGL(k_root_ids_one, dim3(1), dim3(1024), 0, s, labels, int(n), root_id, boff + nb, word);
    } else {
        hipLaunchKernelGGL(k_root_count, dim3(nb), dim3(256), 0, s, labels, n, bcount);
        if (nb <= kSumBlocks) {
            hipLaunchKernelGGL(k_root_ids<true>, dim3(nb), dim3(256), 0, s, labels, n, bcount, root_id, boff + nb, word);
        } else {
            hipLaunchKernelGGL(k_scan_small, dim3(1), dim3(1024), 0, s, bcount, nb, boff);
            hipLaunchKernelGGL(k_root_ids<false>, dim3(nb), dim3(256), 0, s, labels, n, boff, root_id, boff + nb, word);
        }
    }
    AMH_LAUNCH_CHECK("amh_blob_count");
    int total = 0;
    if (!word)
        if (int r = check_hip(hipMemcpyAsync(&total, boff + nb, sizeof(int), hipMemcpyDeviceToHost, s), "D2H count"))
            return r;
    if (int r = check_hip(hipStreamSynchronize(s), "amh_blob_count sync")) return r;
    if (word) total = *g_words.word(slot);
    *nblobs = total;
    return AMH_OK;
}

extern "C" int amh_blob_stats(const int32_t *labels, const uint32_t *stored, int32_t W, int32_t H, void *ws,
                              int32_t nblobs, int32_t *bop, amh_blob_stat *st, void *stream) {
    if (int r = check_frame(W, H, "amh_blob_stats")) return r;
    if (!labels || !stored || !ws || !bop || (nblobs > 0 && !st) || nblobs < 0) {
        set_error("amh_blob_stats: invalid argument");
        return AMH_E_ARG;
    }
    hipStream_t s = static_cast<hipStream_t>(stream);
    const bool one = W <= 64 && H <= 2 * kStatRows;
    const int rows = one ? H : kStatRows;
    if (nblobs > 0 && !one)
        hipLaunchKernelGGL(k_stats_init, dim3((nblobs + 255) / 256), dim3(256), 0, s, st, int(nblobs));
    const dim3 grid(uint32_t((W + 63) / 64), uint32_t((H + rows - 1) / rows));
    const int *root_id = static_cast<const int *>(ws);
    if (one)  // the one workgroup's rows side by side: its chain of loads sets the time
        amh::launch_timed("k_blob_stats", k_blob_stats<1024>, grid, dim3(1024), 0, s, labels, stored, int(W), int(H),
                          rows, root_id, bop, st, int(nblobs), true);
    else
        amh::launch_timed("k_blob_stats", k_blob_stats<256>, grid, dim3(256), 0, s, labels, stored, int(W), int(H),
                          rows, root_id, bop, st, int(nblobs), false);
    AMH_LAUNCH_CHECK("amh_blob_stats");
    return AMH_OK;
}

extern "C" size_t amh_group_workspace_bytes(int32_t npixels, int32_t nblobs) {
    return group_layout(npixels > 0 ? npixels : 0, nblobs > 0 ? nblobs : 0).bytes;
}

extern "C" int amh_group_pixels(const int32_t *bop, int32_t npixels, int32_t nblobs, void *ws, size_t ws_bytes,
                                int64_t *first, int32_t *list, void *stream) {
    if (!bop || !first || !list || npixels < 0 || nblobs < 0 ||
        ws_bytes < amh_group_workspace_bytes(npixels, nblobs) || (!ws && ws_bytes)) {
        set_error("amh_group_pixels: invalid argument");
        return AMH_E_ARG;
    }
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (nblobs == 0) return check_hip(hipMemsetAsync(first, 0, sizeof(int64_t), s), "amh_group_pixels");
    const int64_t n = npixels;
    const GroupLayout L = group_layout(n, nblobs);
    if (L.radix) {
        if (int r = group_radix(L, bop, n, int(nblobs), static_cast<char *>(ws), first, list, s)) return r;
        hipLaunchKernelGGL(k_first_scan, dim3(1), dim3(1024), 0, s, int(nblobs), first);
        AMH_LAUNCH_CHECK("amh_group_pixels");
        return AMH_OK;
    }
    if (n > 0 && n <= kOnePixels && nblobs <= kOneBlobs) {
        hipLaunchKernelGGL(k_group_one, dim3(1), dim3(kOneT), 0, s, bop, int(n), int(nblobs), first, list);
        AMH_LAUNCH_CHECK("amh_group_pixels");
        return AMH_OK;
    }
    const int nbands = L.nblk;
    int *hist = static_cast<int *>(ws);
    const int64_t cells = int64_t(nbands) * nblobs;
    hipLaunchKernelGGL(k_group_zero, dim3(uint32_t(std::min<int64_t>((cells + 255) / 256, 4096))), dim3(256), 0, s, hist,
                       cells);
    hipLaunchKernelGGL(k_group_hist, dim3(nbands), dim3(kBandT), 0, s, bop, n, nbands, hist);
    hipLaunchKernelGGL(k_group_colscan, dim3(uint32_t(nblobs)), dim3(256), 0, s, hist, nbands, first);
    hipLaunchKernelGGL(k_first_scan, dim3(1), dim3(1024), 0, s, int(nblobs), first);
    hipLaunchKernelGGL(k_group_scatter, dim3(nbands), dim3(kBandT), 0, s, bop, n, nbands, hist, first, list);
    AMH_LAUNCH_CHECK("amh_group_pixels");
    return AMH_OK;
}

extern "C" int amh_build_chains(const amh_chain_build *a, uint64_t *pts, void *stream) {
    if (!a || !pts || a->nkeys <= 0 || a->nchains <= 0 || a->wtot <= 0 || !a->chain_off_dev || !a->chain_w_dev ||
        !a->chain_blob_dev || !a->empty_xy_dev || !a->pixel_list_dev || !a->blob_first_dev || a->frame_width <= 0) {
        set_error("amh_build_chains: invalid argument");
        return AMH_E_ARG;
    }
    hipStream_t s = static_cast<hipStream_t>(stream);
    const uint32_t blocks = uint32_t((a->wtot + 255) / 256);
    for (int y = 0; y < a->nkeys; ++y) {
        hipLaunchKernelGGL(k_build_row, dim3(blocks), dim3(256), 0, s, y, a->nkeys, a->wtot, a->nchains,
                           a->chain_off_dev, a->chain_w_dev, a->chain_blob_dev, a->empty_xy_dev,
                           a->pixel_list_dev[y], a->blob_first_dev[y], a->frame_width, a->seed, pts);
    }
    AMH_LAUNCH_CHECK("amh_build_chains");
    return AMH_OK;
}

// Host-callable colour conversions with the kernels' arithmetic.
extern "C" uint32_t amh_rgb_to_hsp(uint32_t rgba) { return rgb_to_hsp(rgba); }
extern "C" uint32_t amh_hsp_to_rgb(uint32_t hspa) { return hsp_to_rgb(hspa); }
extern "C" void amh_rgb2hsp(double r, double g, double b, double *h, double *s, double *p) { rgb2hsp(r, g, b, h, s, p); }
extern "C" void amh_hsp2rgb(double h, double s, double p, double *r, double *g, double *b) { hsp2rgb(h, s, p, r, g, b); }
