// Frame rendering on the atom path: morph::get_pixels(t) -> draw_atoms
// (morph.cpp:1302-1421) over get_pixels(blob, t) (morph.cpp:452-678).
//
// Per frame:
//   prepare  per atom: trajectory point and colour at t (FP64, the
//            reference's operation order), bilinear taps; its taps counted
//            into the 16 x 16 pixel tiles they fall in.
//   place    the atoms' numbers into the tiles' lists (starts: the scan of
//            the counts).
//   splat    one workgroup per tile, one thread per pixel: the tile's taps
//            are summed in LDS (count, sum n, sum c*n with n = the integer
//            bilinear weight numerator) for one blob per pixel at a time, in
//            increasing blob order, and each resolved colour is composited
//            "over" in that order; background, RGBA8 out.
//   composite  (inward feather only) the splat leaves each pixel's resolved
//            blobs as a list instead, since the feather of a pixel asks
//            whether its neighbours, in other tiles too, hold the same blob;
//            a second kernel feathers and composites them.
// Composite order equals the reference's (blob order); sums are exact, so
// nothing depends on the order the atoms land in.
//
// The sums stay in LDS because device-wide 64-bit atomics are performed past
// the L2: with five of them per tap into per-pixel accumulators in memory
// (and a second, scanned list for the other blobs of a pixel) a frame took
// 1,518 us at 2048^2 with 1.7 M atoms, 261 us at 1001 x 777 with feather 2;
// in tiles it takes 207 and 70 us (kernels at 2048^2: prepare 88, the scan of
// the counts 9, place 36, splat 73 us).
#include <mutex>
#include <type_traits>

#include "colour.h"
#include "common.h"
#include "../../include/atomorph_hip.h"
#include "scan.h"
#include "shade.h"

using namespace amh;
using namespace amh::shade;

namespace {

constexpr int kT = 256;
constexpr int kTile = 16;             // pixels per side of an image tile
constexpr int kTilePx = kTile * kTile;  // one thread of the splat per pixel
static_assert(kTilePx == kT, "one thread per pixel");
constexpr int kFewTiles = 4096;       // up to this many tiles blocks count, scan and place atoms per tile in LDS (k_place)
constexpr int kManyTiles = 16384;     // up to this many, larger blocks count them there
constexpr int kNoBlob = 0x7FFFFFFF;
// The tiles' lists are indexed by 32-bit sums of the atoms' taps, four of an
// atom at most (kEnd is none of them).
constexpr int64_t kMaxAtoms = 0x3FFFFFFF;
constexpr uint32_t kEnd = 0xFFFFFFFFu;

// --------------------------------------------------------------- prepare
struct Rec {       // one atom's splat, 16 bytes
    uint32_t xy;   // x | y << 16 of the base tap
    uint32_t fm;   // x_fract | y_fract << 8 | tap mask << 16 (mask 0: not drawn)
    uint32_t col;  // RGBA8
    int32_t blob;  // composite index
};

// The image tiles and their lists.
struct Tiles {
    int32_t ntx, nty;
    uint32_t *taps;     // [tiles] taps that fall in the tile
    uint32_t *entries;  // [tiles] atoms listed so far
    uint32_t *start;    // [tiles + 1] scan of taps: a tile lists at most one atom per tap
    uint32_t *list;     // [<= 4 atoms] atom numbers
};

// The taps of `mask` (bit k: tap (k & 1, k >> 1) of the base pixel x, y) that
// fall in tile (x / 16 + (j & 1), y / 16 + (j >> 1)).
__device__ __forceinline__ uint32_t taps_in(uint32_t mask, uint32_t x, uint32_t y, int j) {
    const uint32_t right = (x % kTile == kTile - 1) ? 10u : 0u, below = (y % kTile == kTile - 1) ? 12u : 0u;
    return mask & ((j & 1) ? right : ~right) & ((j & 2) ? below : ~below);
}
__device__ __forceinline__ int tile_of(uint32_t x, uint32_t y, int j, int ntx) {
    return int(y / kTile + (j >> 1)) * ntx + int(x / kTile + (j & 1));
}

// What bounds it: the instructions of the PERLIN fade's 16 noise octaves per
// atom (1.7 M atoms: 246 us with one noise at a time and selects for the
// gradients, 90 us with both together from tables).  The taps are counted per
// tile in the block's LDS, TILES counters of 16 bits, then one atomic per
// tile and block: refined chains scatter, so that grouping a wave's lanes by
// tile (TILES = 0, one atomic per distinct tile) takes up to 64 turns, and on
// few tiles the atomics queue at the same counters.  11,000 atoms on 70
// tiles: 17.8 us grouped, 4.9 in LDS; 300,000 on 3,087: 21.7 and 10; 1.7 M on
// 16,384: 110 and 90, in blocks of 1,024 that share the 32 KB.  A row of tiles
// further 1.7 M atoms take 82 us grouped against 70 here where neighbours lie
// together, 140 against 117 scattered; counters for more tiles than that in LDS
// have not been measured.
template <int NT, int TILES>
__global__ __launch_bounds__(NT) void k_prepare(amh_render R, Frame F, Rec *__restrict__ recs, Tiles B) {
    __shared__ PerlinTab tab;
    __shared__ uint4 counters[TILES ? TILES / 8 : 1];  // 16 bits per tile
    static_assert(4 * NT < 1 << 16, "a block's taps fit 16 bits");
    const int64_t a = int64_t(blockIdx.x) * NT + threadIdx.x;
    const bool in = a < R.wtot;
    // the points first: their loads overlap the tables' and the chain search
    const int64_t al = in ? a : 0;
    const uint64_t p1 = R.pts_dev[int64_t(F.fk) * R.wtot + al];
    const uint64_t p2 = R.pts_dev[int64_t(F.fnext) * R.wtot + al];
    uint64_t tk[4] = {p1, p1, p2, p2};
    traj_keys(R, F, al, tk);
    if (R.fading == kPerlin) stage_perlin(R.lag_perm_dev, R.slope_perm_dev, tab, threadIdx.x, NT);
    const int tiles = B.ntx * B.nty;
    if (TILES)
        for (int k = threadIdx.x; k < (tiles + 7) / 8; k += NT) counters[k] = uint4{0u, 0u, 0u, 0u};
    __syncthreads();
    const int c = block_chain(R.chain_off_dev, R.nchains, a);
    uint32_t mask = 0, X = 0, Y = 0;
    if (in) {
        Rec rec = {0u, 0u, 0u, -1};
        const int W = R.width, H = R.height;
        const int b = R.rank_dev[int64_t(F.fk) * R.nchains + c];
        const bool h1 = pt_flags(p1) & HAS_PIXEL, h2 = pt_flags(p2) & HAS_PIXEL;
        if (b >= 0 && (h1 || h2)) {
            // colours at both ends (morph.cpp:495-522); a missing end fades from /
            // to the other end's colour with alpha 0
            uint32_t c1 = key_px(R.keys_dev, F.fk, W, H, pt_x(p1), pt_y(p1));
            uint32_t c2 = key_px(R.keys_dev, F.fnext, W, H, pt_x(p2), pt_y(p2));
            if (!h2) c2 = c1 & 0x00FFFFFFu;
            else if (!h1) c1 = c2 & 0x00FFFFFFu;
            uint32_t qxf, qyf;
            traj_point(R, F, a, p1, p2, X, Y, qxf, qyf, tk);
            const uint32_t col = atom_colour(R, F, p1, c1, c2, tab);
            // guards and taps (morph.cpp:552-589); taps outside the image are
            // dropped (draw_atoms skips pos >= W*H)
            const int x = int(X), y = int(Y), xf = int(qxf), yf = int(qyf);
            if (x < W && y < H) {
                if ((255 - xf) * (255 - yf) > 0) mask |= 1u;
                if (x + 1 < W && xf * (255 - yf) > 0) mask |= 2u;
                if (y + 1 < H && (255 - xf) * yf > 0) mask |= 4u;
                if (x + 1 < W && y + 1 < H && xf * yf > 0) mask |= 8u;
            }
            if (mask) rec = Rec{X | (Y << 16), qxf | (qyf << 8) | (mask << 16), col, b};
        }
        recs[a] = rec;
    }
    if (TILES) {
        uint32_t *cnt = reinterpret_cast<uint32_t *>(counters);
        for (int j = 0; j < 4; ++j) {
            const uint32_t m = taps_in(mask, X, Y, j);
            if (!m) continue;
            const int t = tile_of(X, Y, j, B.ntx);
            atomicAdd(&cnt[t / 2], uint32_t(__popc(m)) << (t % 2 * 16));
        }
        __syncthreads();
        for (int k = threadIdx.x; k < (tiles + 7) / 8; k += NT) {
            const uint4 c = counters[k];
            if ((c.x | c.y | c.z | c.w) == 0) continue;
            const uint32_t w[4] = {c.x, c.y, c.z, c.w};
            for (int q = 0; q < 8; ++q) {
                const uint32_t n = w[q / 2] >> (q % 2 * 16) & 0xFFFFu;
                if (n) atomicAdd(&B.taps[8 * k + q], n);
            }
        }
        return;
    }
    const int lane = threadIdx.x & 63;
    for (int j = 0; j < 4; ++j) {
        const uint32_t m = taps_in(mask, X, Y, j);
        const int t = m ? tile_of(X, Y, j, B.ntx) : -1;
        const int w = int(__popc(m));
        uint64_t todo = __ballot(m != 0);
        if (!todo) continue;
        const uint64_t w0 = __ballot(w & 1), w1 = __ballot(w & 2), w2 = __ballot(w & 4);
        while (todo) {
            const int leader = __ffsll((unsigned long long)todo) - 1;
            const uint64_t same = __ballot(t == __builtin_amdgcn_readlane(t, leader));
            if (lane == leader)
                atomicAdd(&B.taps[t], uint32_t(__popcll(same & w0) + 2 * __popcll(same & w1) + 4 * __popcll(same & w2)));
            todo &= ~same;
        }
    }
}

// The atoms' numbers into their tiles' lists, in no fixed order (the sums are
// exact).  kFew: every block scans the tap counts in LDS (block 0 stores the
// starts) and takes ranks within the block from LDS counters, as in k_prepare;
// otherwise B.start holds the scan already and a wave's lanes are grouped.
// (With the counting in LDS, eight 64^2 frames 239 -> 191 us, a frame of 3,087
// tiles 94 -> 65.)  Every block scans all tiles, so that this loses before its
// limit: of 4,096 tiles and of 4,225 (and two launches of 4.6 us for the scan)
// 300,000 neighbouring atoms take 24 and 7 us, scattered ones 66 and 43; 1.7 M
// neighbouring ones 104 and 22, scattered ones 185 and 209.
template <bool kFew>
__global__ __launch_bounds__(kT) void k_place(const Rec *__restrict__ recs, int64_t n, Tiles B) {
    const int64_t a = int64_t(blockIdx.x) * kT + threadIdx.x;
    const uint2 r = *reinterpret_cast<const uint2 *>(&recs[a < n ? a : 0]);
    const uint32_t X = r.x & 0xFFFFu, Y = r.x >> 16, mask = a < n ? r.y >> 16 : 0u;
    if constexpr (kFew) {
        __shared__ uint32_t start[kFewTiles + 1], cnt[kFewTiles], wsum[kT / 64];
        const int tiles = B.ntx * B.nty;
        scan::block_exclusive(tiles, [&](int k) { return B.taps[k]; }, start, wsum);
        if (blockIdx.x == 0)
            for (int k = threadIdx.x; k <= tiles; k += kT) B.start[k] = start[k];
        for (int k = threadIdx.x; k < tiles; k += kT) cnt[k] = 0;
        __syncthreads();
        int t[4];
        uint32_t rank[4];
        for (int j = 0; j < 4; ++j) {
            t[j] = taps_in(mask, X, Y, j) ? tile_of(X, Y, j, B.ntx) : -1;
            rank[j] = t[j] >= 0 ? atomicAdd(&cnt[t[j]], 1u) : 0u;
        }
        __syncthreads();
        for (int k = threadIdx.x; k < tiles; k += kT)
            if (cnt[k]) cnt[k] = start[k] + atomicAdd(&B.entries[k], cnt[k]);
        __syncthreads();
        for (int j = 0; j < 4; ++j)
            if (t[j] >= 0) B.list[cnt[t[j]] + rank[j]] = uint32_t(a);
        return;
    }
    const int lane = threadIdx.x & 63;
    const uint64_t below = (1ull << lane) - 1ull;
    int t[4], lead[4];  // the wave's lanes grouped by tile, per neighbour tile
    uint32_t pre[4], total[4];
    for (int j = 0; j < 4; ++j) {
        t[j] = taps_in(mask, X, Y, j) ? tile_of(X, Y, j, B.ntx) : -1;
        lead[j] = lane;
        pre[j] = total[j] = 0u;
        uint64_t todo = __ballot(t[j] >= 0);
        while (todo) {
            const int leader = __ffsll((unsigned long long)todo) - 1;
            const uint64_t same = __ballot(t[j] == __builtin_amdgcn_readlane(t[j], leader));
            if ((same >> lane) & 1u) {
                lead[j] = leader;
                pre[j] = uint32_t(__popcll(same & below));
            }
            if (lane == leader) total[j] = uint32_t(__popcll(same));
            todo &= ~same;
        }
    }
    uint32_t base[4], first[4];
    for (int j = 0; j < 4; ++j) {
        base[j] = total[j] > 0u ? atomicAdd(&B.entries[t[j]], total[j]) : 0u;
        first[j] = B.start[max(t[j], 0)];
    }
    for (int j = 0; j < 4; ++j) {
        const uint32_t b = __shfl(base[j], lead[j], 64);
        if (t[j] >= 0) B.list[first[j] + b + pre[j]] = uint32_t(a);
    }
}

// ------------------------------------------------------------ composite
struct Px {  // one resolved (pixel, blob) colour
    uint32_t r, g, b, a;
};

// morph.cpp:591-623 with exact integer sums: round(sum c*n / sum n), alpha
// times min(1, count / density).  The quotients are floor((2 s + sn) / (2 sn))
// through one FP64 reciprocal: all operands are integers below 2^53, so the
// estimate is at most one off and its remainder, exact in a fused
// multiply-add, says which way (four 64-bit integer divisions took the splat
// 110 registers).
template <class T>
__device__ __forceinline__ Px resolve(uint32_t cnt, T sn, const T s[4], int density) {
    const double n = double(sn), d = 2.0 * n, inv = 1.0 / d;
    uint32_t v[4];
    for (int k = 0; k < 4; ++k) {
        const double num = fma(2.0, double(s[k]), n);
        const int q = int(num * inv);
        const double rem = fma(-double(q), d, num);
        v[k] = uint32_t(q + (rem >= d ? 1 : 0) - (rem < 0.0 ? 1 : 0));
    }
    const double w = density > 0 ? double(cnt) / double(density) : 0.0;
    if (!(w >= 1.0)) v[3] = narrow8(round(w * (double(s[3]) / n)));
    return Px{v[0], v[1], v[2], v[3]};
}

// With feather: the resolved blobs of a pixel, in increasing blob order.  The
// first is kept per pixel; the others are a chain of Ov, in the splat's
// numbering of the tile's taps (a (pixel, blob) pair has at least one tap).
struct Ov {
    int32_t blob;
    uint32_t col;
    uint32_t next;  // kEnd: last
};
struct Resolved {
    int32_t *blob;  // [npx] kNoBlob: none
    uint32_t *col;
    uint32_t *next;
    Ov *ov;         // [<= 4 atoms]
};

// Is blob b among the further blobs of pixel q?
__device__ __forceinline__ bool chained(const Resolved &V, int64_t q, int b) {
    for (uint32_t i = V.next[q]; i != kEnd; i = V.ov[i].next)
        if (V.ov[i].blob == b) return true;
    return false;
}

// Inward feather (morph.cpp:625-674): the peel layer of pixel (x, y) in
// blob b is d - 1, d = L1 distance to the nearest pixel outside the blob
// (coordinates 0 and 65535 count as blob borders).  Returns d (> feather:
// untouched).
__device__ int feather_depth(int x, int y, int W, int H, int F, int b, const Resolved &V) {
    int best = F + 1;
    best = min(best, x + 1);
    best = min(best, y + 1);
    best = min(best, 65536 - x);
    best = min(best, 65536 - y);
    for (int r = 1; r < best; ++r) {
        // the 4 r pixels at L1 distance r, one of each quadrant at a time, so
        // that their first blobs are loaded together
        for (int i = 0; i < r; ++i) {
            const int dx[4] = {i, r - i, -i, i - r}, dy[4] = {r - i, -i, i - r, i};
            int64_t q[4];
            int v[4];
            bool in = true;
            for (int k = 0; k < 4; ++k) {
                const int qx = x + dx[k], qy = y + dy[k];
                const bool ok = qx >= 0 && qy >= 0 && qx < W && qy < H;
                in = in && ok;
                q[k] = ok ? int64_t(qy) * W + qx : 0;
                v[k] = V.blob[q[k]];
            }
            for (int k = 0; k < 4; ++k) in = in && (v[k] == b || (v[k] < b && chained(V, q[k], b)));
            if (!in) return r;
        }
    }
    return best;
}

// "Over" in increasing blob order (morph.cpp:1357-1380).  Without blending
// the first colour is only taken apart when a second follows: alone, it comes
// back from the division by 255 and the rounding as it was.
struct Over {
    double r = 0, g = 0, b = 0, a = 0;
    uint32_t one = 0;
    int n = 0;
    __device__ void add(uint32_t c) {
        if (n++ == 0) {
            one = c;
            return;
        }
        if (n == 2) {
            r = (one & 255u) / 255.0;
            g = ((one >> 8) & 255u) / 255.0;
            b = ((one >> 16) & 255u) / 255.0;
            a = (one >> 24) / 255.0;
        }
        const double sr = (c & 255u) / 255.0, sg = ((c >> 8) & 255u) / 255.0;
        const double sb = ((c >> 16) & 255u) / 255.0, sa = (c >> 24) / 255.0;
        r = sa * sr + (1.0 - sa) * r;
        g = sa * sg + (1.0 - sa) * g;
        b = sa * sb + (1.0 - sa) * b;
        a = a + (1.0 - a) * sa;
    }
    __device__ uint32_t colour() const {
        if (n < 2) return one;
        return rgba_pack(narrow8(round(r * 255.0)), narrow8(round(g * 255.0)), narrow8(round(b * 255.0)),
                         narrow8(round(a * 255.0)));
    }
};

// The same with the alpha-weighted sums that blending takes.
struct Blend {
    double r = 0, g = 0, b = 0, a = 0, rs = 0, gs = 0, bs = 0, as = 0;
    int n = 0;
    __device__ void add(uint32_t c) {
        const double sr = (c & 255u) / 255.0, sg = ((c >> 8) & 255u) / 255.0;
        const double sb = ((c >> 16) & 255u) / 255.0, sa = (c >> 24) / 255.0;
        as += sa;
        rs += sr * sa;
        gs += sg * sa;
        bs += sb * sa;
        if (n == 0) {
            r = sr; g = sg; b = sb; a = sa;
        } else {
            r = sa * sr + (1.0 - sa) * r;
            g = sa * sg + (1.0 - sa) * g;
            b = sa * sb + (1.0 - sa) * b;
            a = a + (1.0 - a) * sa;
        }
        ++n;
    }
};

// The folded pixel over the background (morph.cpp:1381-1401, 1405-1417).
__device__ __forceinline__ uint32_t finish(const amh_render &R, const Blend &fold, uint32_t bg) {
    if (fold.n == 0) return bg;
    double r = fold.r, g = fold.g, b = fold.b, a = fold.a;
    if (R.blend_blobs) {
        r = fold.rs / fold.as;
        g = fold.gs / fold.as;
        b = fold.bs / fold.as;
    }
    if (R.keep_background) {
        const double bgr = double(bg & 255u) / 255.0, bgg = double((bg >> 8) & 255u) / 255.0;
        const double bgb = double((bg >> 16) & 255u) / 255.0, bga = double(bg >> 24) / 255.0;
        r = a * r + (1.0 - a) * bgr;
        g = a * g + (1.0 - a) * bgg;
        b = a * b + (1.0 - a) * bgb;
        a = bga + (1.0 - bga) * a;
    }
    return rgba_pack(narrow8(round(r * 255.0)), narrow8(round(g * 255.0)), narrow8(round(b * 255.0)),
                     narrow8(round(a * 255.0)));
}

// Per-pixel sums of a tile in LDS: taps, sum n and sum c * n per channel.
// Wide: any number of taps.  Packed: a tile of at most kPackedAtoms atoms, of
// which each gives a pixel one tap at most, so sum n < 2^24, the taps fit in
// 8 bits and sum c * n in 32: three atomics per tap instead of five.
constexpr int kPackedAtoms = 255;
static_assert(255ull * 65025 * kPackedAtoms < 1ull << 32 && 65025 * kPackedAtoms < 1 << 24, "packed sums");

struct PackedSums {
    using T = uint32_t;
    uint32_t cn[kTilePx];                         // taps << 24 | sum n
    unsigned long long rg[kTilePx], ba[kTilePx];  // two channels each
    __device__ __forceinline__ void clear(int p) {
        cn[p] = 0u;
        rg[p] = ba[p] = 0ull;
    }
    __device__ __forceinline__ void add(int p, uint32_t n, uint32_t col) {
        atomicAdd(&cn[p], (1u << 24) | n);
        atomicAdd(&rg[p], (unsigned long long)(ch(col, 0) * n) | ((unsigned long long)(ch(col, 1) * n) << 32));
        atomicAdd(&ba[p], (unsigned long long)(ch(col, 2) * n) | ((unsigned long long)(ch(col, 3) * n) << 32));
    }
    __device__ __forceinline__ uint32_t get(int p, T &sn, T s[4]) const {
        const uint32_t v = cn[p];
        sn = v & 0xFFFFFFu;
        s[0] = T(rg[p]);
        s[1] = T(rg[p] >> 32);
        s[2] = T(ba[p]);
        s[3] = T(ba[p] >> 32);
        return v >> 24;
    }
};
struct WideSums {
    using T = uint64_t;
    unsigned long long cn[kTilePx], s[4][kTilePx];  // taps << 40 | sum n
    __device__ __forceinline__ void clear(int p) {
        cn[p] = 0ull;
        for (int k = 0; k < 4; ++k) s[k][p] = 0ull;
    }
    __device__ __forceinline__ void add(int p, uint32_t n, uint32_t col) {
        atomicAdd(&cn[p], (1ull << 40) | n);
        for (int k = 0; k < 4; ++k) atomicAdd(&s[k][p], (unsigned long long)(ch(col, k) * n));
    }
    __device__ __forceinline__ uint32_t get(int p, T &sn, T v[4]) const {
        sn = cn[p] & ((1ull << 40) - 1);
        for (int k = 0; k < 4; ++k) v[k] = s[k][p];
        return uint32_t(cn[p] >> 40);
    }
};

// f(pixel of the tile at x0, y0, weight numerator, atom) for every tap in the
// tile of its n atoms; each thread's first atom is `mine`.
template <class F>
__device__ __forceinline__ void for_taps(const Rec *__restrict__ recs, const uint32_t *__restrict__ list, int n,
                                         const Rec &mine, int x0, int y0, const F &f) {
    for (int e = threadIdx.x; e < n; e += kT) {
        Rec r = e == int(threadIdx.x) ? mine : recs[list[e]];
        // opaque, so that the taps' products are not kept for all passes
        // (they took 108 registers; without them eight waves fit)
        asm volatile("" : "+v"(r.xy), "+v"(r.fm), "+v"(r.col));
        const uint32_t xf = r.fm & 255u, yf = (r.fm >> 8) & 255u, mask = r.fm >> 16;
        const int lx = int(r.xy & 0xFFFFu) - x0, ly = int(r.xy >> 16) - y0;
        for (int k = 0; k < 4; ++k) {
            const int px = lx + (k & 1), py = ly + (k >> 1);
            if (!((mask >> k) & 1u) || uint32_t(px) >= uint32_t(kTile) || uint32_t(py) >= uint32_t(kTile)) continue;
            f(py * kTile + px, ((k & 1) ? xf : 255u - xf) * ((k >> 1) ? yf : 255u - yf), r);
        }
    }
}

// Calls emit(blob, colour) for every blob of this thread's pixel in
// increasing blob order.  one: the blob of every atom of the tile, or -1: then
// each pass sums, per pixel, the taps of one blob (bcur) and finds the next
// larger one that touches the pixel (bnext) on the way.
template <class Sums, class Emit>
__device__ __forceinline__ void tile_blobs(Sums &acc, int *bcur, int *bnext, const Rec *__restrict__ recs,
                                           const uint32_t *__restrict__ list, int n, const Rec &mine, int one, int x0,
                                           int y0, int density, const Emit &emit) {
    const int tid = threadIdx.x;
    const auto give = [&](int b) {
        typename Sums::T sn, s[4];
        const uint32_t cnt = acc.get(tid, sn, s);
        if (cnt) {
            const Px q = resolve(cnt, sn, s, density);
            emit(b, rgba_pack(q.r, q.g, q.b, q.a));
        }
    };
    acc.clear(tid);
    if (one >= 0) {
        __syncthreads();
        for_taps(recs, list, n, mine, x0, y0, [&](int p, uint32_t w, const Rec &r) { acc.add(p, w, r.col); });
        __syncthreads();
        give(one);
        return;
    }
    bnext[tid] = kNoBlob;
    __syncthreads();
    for_taps(recs, list, n, mine, x0, y0, [&](int p, uint32_t, const Rec &r) { atomicMin(&bnext[p], r.blob); });
    __syncthreads();
    for (;;) {
        const int b = bnext[tid];
        bcur[tid] = b;
        bnext[tid] = kNoBlob;
        acc.clear(tid);
        if (!__syncthreads_or(b != kNoBlob)) break;
        for_taps(recs, list, n, mine, x0, y0, [&](int p, uint32_t w, const Rec &r) {
            const int cur = bcur[p];
            if (r.blob == cur) acc.add(p, w, r.col);
            else if (r.blob > cur) atomicMin(&bnext[p], r.blob);
        });
        __syncthreads();
        give(b);
    }
}

// One workgroup per tile, one thread per pixel.  A tile's loads are one
// dependent chain (counters, list, atoms), so each mode holds only the
// registers it needs and eight workgroups fit a CU; then the LDS atomics and
// the tap arithmetic bound it.  Hence the packed sums, and with them the single
// pass over a tile whose atoms are all of one blob: 109 us at 2048^2 with 110
// registers and five sums, 94 with 54 registers, 73 with these.  They serve
// blobs' rims, sparse blobs and frames in motion; a tile filled by a blob at
// rest holds 256 atoms and more, and takes the wide sums in two passes.
// Leaves the tile's counters at zero for the next frame.
enum SplatMode {
    kPlain,    // no background, no blending
    kOver,     // over the background, or blending
    kFeather,  // the resolved colours go to V for k_composite
};
template <SplatMode kMode>
__global__ __launch_bounds__(kT) void k_splat(amh_render R, Frame F, const Rec *__restrict__ recs, Tiles B, Resolved V,
                                              uint32_t *__restrict__ out) {
    __shared__ union {
        PackedSums packed;
        WideSums wide;
    } acc;
    __shared__ int bcur[kTilePx], bnext[kTilePx];
    __shared__ std::conditional_t<kMode == kOver, PerlinTab, char> tab;
    __shared__ uint32_t nov;
    __shared__ int some;
    const int tile = int(blockIdx.x), tid = int(threadIdx.x);
    const int x0 = (tile % B.ntx) * kTile, y0 = (tile / B.ntx) * kTile;
    const int x = x0 + tid % kTile, y = y0 + tid / kTile;
    const bool inside = x < R.width && y < R.height;
    const int64_t p = int64_t(y) * R.width + x;
    const int n = int(B.entries[tile]);
    const uint32_t s0 = B.start[tile];
    std::conditional_t<kMode == kOver, Blend, Over> fold;
    uint32_t last = kEnd;  // kFeather: the pixel's last chained Ov
    bool first = true;
    if constexpr (kMode == kOver)
        if (R.keep_background && R.fading == kPerlin) stage_perlin(R.lag_perm_dev, R.slope_perm_dev, tab, tid, kT);
    if (n > 0) {
        const uint32_t *list = B.list + s0;
        Rec mine = {0u, 0u, 0u, 0};
        if (tid < n) mine = recs[list[tid]];
        if (tid == 0) {
            nov = 0;
            some = mine.blob;
        }
        __syncthreads();
        if (tid == 0) {  // every thread has read them
            B.entries[tile] = 0;
            B.taps[tile] = 0;
        }
        const auto emit = [&](int b, uint32_t c) {
            if constexpr (kMode == kFeather) {
                if (first) {
                    V.blob[p] = b;
                    V.col[p] = c;
                } else {
                    const uint32_t o = s0 + atomicAdd(&nov, 1u);
                    V.ov[o] = Ov{b, c, kEnd};
                    if (last == kEnd) V.next[p] = o;
                    else V.ov[last].next = o;
                    last = o;
                }
                first = false;
            } else {
                const bool texture = R.show_blobs != 1 && R.show_blobs != 2;
                if (!texture && R.blob_rgba_dev) c = R.blob_rgba_dev[int64_t(F.fk) * R.nblobs + b];
                if (c >> 24) fold.add(c);
            }
        };
        if (n <= kPackedAtoms) {
            const int one = __syncthreads_or(tid < n && mine.blob != some) ? -1 : some;
            tile_blobs(acc.packed, bcur, bnext, recs, list, n, mine, one, x0, y0, R.density, emit);
        } else {
            tile_blobs(acc.wide, bcur, bnext, recs, list, n, mine, -1, x0, y0, R.density, emit);
        }
    } else if (kMode == kOver) {
        __syncthreads();  // the noise tables
    }
    if (!inside) return;
    if constexpr (kMode == kFeather) {
        if (first) V.blob[p] = kNoBlob;
        if (last == kEnd) V.next[p] = kEnd;
    } else if constexpr (kMode == kOver) {
        out[p] = finish(R, fold, R.keep_background ? background(R, F, x, y, tab) : 0u);
    } else {
        out[p] = fold.colour();
    }
}

// Feather and composite of the resolved blobs (texture blobs only: the other
// modes are not feathered).
__global__ __launch_bounds__(kT) void k_composite(amh_render R, Frame F, Resolved V, uint32_t *__restrict__ out) {
    __shared__ PerlinTab tab;
    if (R.keep_background && R.fading == kPerlin)
        stage_perlin(R.lag_perm_dev, R.slope_perm_dev, tab, threadIdx.x, kT);
    __syncthreads();
    const int W = R.width, H = R.height;
    const int64_t p = int64_t(blockIdx.x) * kT + threadIdx.x;
    if (p >= int64_t(W) * H) return;
    const int x = int(p % W), y = int(p / W);
    Blend fold;
    Ov o = {V.blob[p], V.col[p], V.next[p]};
    while (o.blob != kNoBlob) {
        const int d = feather_depth(x, y, W, H, R.feather, o.blob, V);
        uint32_t c = o.col;
        if (d <= R.feather)
            c = (c & 0x00FFFFFFu) | (narrow8(round(double(c >> 24) * (double(d) / double(R.feather + 1)))) << 24);
        if (c >> 24) fold.add(c);
        if (o.next == kEnd) break;
        o = V.ov[o.next];
    }
    out[p] = finish(R, fold, R.keep_background ? background(R, F, x, y, tab) : 0u);
}

// ------------------------------------------------------------ workspace
struct Layout {
    int64_t npx, tiles;
    int32_t ntx, nty;
    size_t taps, entries, start, sums, offs, recs, list, ov, blob, col, next, total;
};
Layout layout(int32_t W, int32_t H, int64_t wtot) {
    Layout L;
    L.npx = int64_t(W) * H;
    L.ntx = (W + kTile - 1) / kTile;
    L.nty = (H + kTile - 1) / kTile;
    L.tiles = int64_t(L.ntx) * L.nty;
    const size_t n = size_t(wtot > 0 ? wtot : 1), nt = size_t(L.tiles), nb = size_t(scan::blocks(L.tiles));
    auto al = [](size_t v) { return (v + 255) & ~size_t(255); };
    size_t o = 0;
    L.taps = o;  // the counters first: they stay at zero between frames
    L.entries = o + 4 * nt;
    o = al(o + 8 * nt);
    L.start = o; o = al(o + 4 * (nt + 1));
    L.sums = o;
    L.offs = o + 4 * nb;
    o = al(o + 4 * (2 * nb + 1));
    // per atom: its record, 4 list entries, 4 chained blobs
    L.recs = o;
    L.list = o + sizeof(Rec) * n;
    L.ov = L.list + 16 * n;
    o = al(L.ov + 4 * sizeof(Ov) * n);
    L.blob = o;
    L.col = o + 4 * size_t(L.npx);
    L.next = o + 8 * size_t(L.npx);
    o += 12 * size_t(L.npx);
    // The size asked of callers: 52 bytes per pixel and 80 per atom, eight
    // arrays.  It decides which frames amh_render_frame_noalloc takes.
    const size_t px = size_t(L.npx), pb = size_t(scan::blocks(L.npx));
    L.total = 2 * al(4 * px) + al(4 * (px + 1)) + 2 * al(4 * (pb + 1)) + al(40 * px) + al(16 * n) + al(64 * n);
    if (L.total < o) L.total = o;
    return L;
}

Tiles tiles_of(char *ws, const Layout &L) {
    return Tiles{L.ntx, L.nty, reinterpret_cast<uint32_t *>(ws + L.taps), reinterpret_cast<uint32_t *>(ws + L.entries),
                 reinterpret_cast<uint32_t *>(ws + L.start), reinterpret_cast<uint32_t *>(ws + L.list)};
}

}  // namespace

extern "C" size_t amh_render_workspace_bytes(int32_t W, int32_t H, int64_t wtot) {
    return layout(W, H, wtot).total;
}

extern "C" int amh_render_workspace_init(void *ws, size_t ws_bytes, int32_t W, int32_t H, int64_t wtot,
                                         void *stream) {
    const Layout L = layout(W, H, wtot);
    if (!ws || ws_bytes < L.total || W <= 0 || H <= 0) {
        set_error("amh_render_workspace_init: invalid argument");
        return AMH_E_ARG;
    }
    hipStream_t s = static_cast<hipStream_t>(stream);
    char *base = static_cast<char *>(ws);
    return check_hip(hipMemsetAsync(base, 0, L.total, s), "amh_render_workspace_init");
}

namespace {

bool render_args_ok(const amh_render *R) {
    return R && R->width > 0 && R->height > 0 && R->nkeys > 0 && R->nchains >= 0 && R->keys_dev &&
           !(R->wtot > 0 && (!R->pts_dev || !R->chain_off_dev || !R->chain_w_dev || !R->rank_dev)) &&
           !(R->fading == kPerlin && (!R->lag_perm_dev || !R->slope_perm_dev)) && R->width <= 65535 &&
           R->height <= 65535 && R->wtot >= 0 && R->wtot <= kMaxAtoms;
}

// The frame itself, on a workspace laid out by `L` whose tile counters are
// zero; leaves them at zero.
int render_frame_on(const amh_render *R, double t, char *base, const Layout &L, uint32_t *out, hipStream_t s);

}  // namespace

extern "C" int amh_render_frame(const amh_render *R, double t, void *ws, size_t ws_bytes, uint32_t *out,
                                void *stream) {
    if (!render_args_ok(R) || !ws || !out) {
        set_error("amh_render_frame: invalid argument");
        return AMH_E_ARG;
    }
    const Layout L = layout(R->width, R->height, R->wtot);
    if (ws_bytes < L.total) {
        set_error("amh_render_frame: workspace %zu < %zu bytes", ws_bytes, L.total);
        return AMH_E_ARG;
    }
    return render_frame_on(R, t, static_cast<char *>(ws), L, out, static_cast<hipStream_t>(stream));
}

// ------------------------------------------- allocation-free frame render
// The same frame render for callers that cannot allocate (code under HIP
// graph capture, serving loops, harnesses that forbid hipMalloc): the
// workspace is a fixed array in device memory, one per GPU, held until the
// process ends.  Every call on a GPU shares it, so calls that overlap on one
// GPU race; each call clears the parts that must start clean with a fill
// kernel (no memset node, which graph capture would record).
namespace {

constexpr size_t kScratchBytes = size_t(96) << 20;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void *g_scratch_ptr[kMaxDevices] = {};

// The device address of `scratch` on the current device.  The array's name
// is only a host-side stand-in, so kernels and copies get this pointer.
int scratch_ptr(char **out) {
    int dev = -1;
    if (int r = check_hip(hipGetDevice(&dev), "amh_render_frame_noalloc: hipGetDevice")) return r;
    if (dev < 0 || dev >= kMaxDevices) {
        set_error("amh_render_frame_noalloc: device %d beyond %d", dev, kMaxDevices);
        return AMH_E_ARG;
    }
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void *p = nullptr;
        if (int r = check_hip(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)),
                              "amh_render_frame_noalloc: hipGetSymbolAddress"))
            return r;
        g_scratch_ptr[dev] = p;
    }
    *out = static_cast<char *>(g_scratch_ptr[dev]);
    return AMH_OK;
}

// The tile counters := 0.
__global__ __launch_bounds__(kT) void k_ws_reset(uint32_t *__restrict__ counters, int64_t n) {
    const int64_t i = int64_t(blockIdx.x) * kT + threadIdx.x;
    if (i < n) counters[i] = 0u;
}

}  // namespace

extern "C" size_t amh_render_noalloc_max_bytes(void) { return kScratchBytes; }

extern "C" int amh_render_frame_noalloc(const amh_render *R, double t, uint32_t *out, void *stream) {
    if (!render_args_ok(R) || !out) {
        set_error("amh_render_frame_noalloc: invalid argument");
        return AMH_E_ARG;
    }
    const Layout L = layout(R->width, R->height, R->wtot);
    if (L.total > kScratchBytes) {
        set_error("amh_render_frame_noalloc: %dx%d with %lld atoms needs %zu bytes of workspace, more than the "
                  "%zu this entry point holds; use amh_render_frame",
                  R->width, R->height, (long long)R->wtot, L.total, kScratchBytes);
        return AMH_E_ARG;
    }
    char *base = nullptr;
    if (int r = scratch_ptr(&base)) return r;
    hipStream_t s = static_cast<hipStream_t>(stream);
    hipLaunchKernelGGL(k_ws_reset, dim3(uint32_t((2 * L.tiles + kT - 1) / kT)), dim3(kT), 0, s,
                       reinterpret_cast<uint32_t *>(base + L.taps), 2 * L.tiles);
    AMH_LAUNCH_CHECK("amh_render_frame_noalloc");
    return render_frame_on(R, t, base, L, out, s);
}

namespace {
int render_frame_on(const amh_render *R, double t, char *base, const Layout &L, uint32_t *out, hipStream_t s) {
    amh::ProfScope whole_("render_frame", s);
    Rec *recs = reinterpret_cast<Rec *>(base + L.recs);
    const Tiles B = tiles_of(base, L);
    const Resolved V = {reinterpret_cast<int32_t *>(base + L.blob), reinterpret_cast<uint32_t *>(base + L.col),
                        reinterpret_cast<uint32_t *>(base + L.next), reinterpret_cast<Ov *>(base + L.ov)};

    // morph::normalize_time / get_frame_key (morph.cpp:404-450, 460-464)
    Frame F;
    double integ;
    F.tn = modf(t, &integ);
    if (F.tn < 0.0) F.tn += 1.0;
    const size_t fk = size_t(F.tn * R->nkeys);
    amh_render Rc = *R;
    if (fk >= size_t(R->nkeys) || R->wtot == 0) {
        // nothing to draw: the background only
        Rc.wtot = 0;
    }
    F.fk = int(fk < size_t(R->nkeys) ? fk : 0);
    F.fnext = (F.fk + 1) % R->nkeys;
    const double dt = 1.0 / double(R->nkeys);
    F.tl = fmax(0.0, (F.tn - (double(F.fk) * dt)) / dt);
    const auto launch = [&](const char *name, auto kernel, int64_t threads, auto... args) {  // workgroups of kT
        amh::launch_timed(name, kernel, dim3(uint32_t((threads + kT - 1) / kT)), dim3(kT), 0, s, args...);
    };
    if (Rc.wtot > 0) {
        if (L.tiles <= kFewTiles) launch("k_prepare", k_prepare<kT, kFewTiles>, Rc.wtot, Rc, F, recs, B);
        else if (L.tiles <= kManyTiles)
            amh::launch_timed("k_prepare", k_prepare<1024, kManyTiles>, dim3(uint32_t((Rc.wtot + 1023) / 1024)),
                              dim3(1024), 0, s, Rc, F, recs, B);
        else launch("k_prepare", k_prepare<kT, 0>, Rc.wtot, Rc, F, recs, B);
        if (L.tiles <= kFewTiles) {
            launch("k_place", k_place<true>, Rc.wtot, recs, Rc.wtot, B);
        } else {
            scan::exclusive(B.taps, L.tiles, reinterpret_cast<uint32_t *>(base + L.sums),
                            reinterpret_cast<uint32_t *>(base + L.offs), B.start, s);
            launch("k_place", k_place<false>, Rc.wtot, recs, Rc.wtot, B);
        }
    }
    const bool texture = Rc.show_blobs != 1 && Rc.show_blobs != 2;
    if (texture && Rc.feather > 0) {
        launch("k_splat", k_splat<kFeather>, L.tiles * kT, Rc, F, recs, B, V, out);
        launch("k_composite", k_composite, L.npx, Rc, F, V, out);
    } else if (Rc.keep_background || Rc.blend_blobs) {
        launch("k_splat", k_splat<kOver>, L.tiles * kT, Rc, F, recs, B, V, out);
    } else {
        launch("k_splat", k_splat<kPlain>, L.tiles * kT, Rc, F, recs, B, V, out);
    }
    AMH_LAUNCH_CHECK("amh_render_frame");
    return AMH_OK;
}
}  // namespace

// ------------------------------------------------- frames on a kept handle
// The render arguments and the workspace checked and kept for many frames.
// A frame is three or four launches, which are cheaper enqueued one by one
// than as a captured graph with a launch for the frame's time before it:
// eight 64^2 frames took 290 us replayed and 228 us enqueued, two 2048^2
// frames 494 and 478 us.
struct amh_render_graph_s {
    amh_render R;
    char *ws;
    Layout L;
};

extern "C" int amh_render_graph_create(void **graph, const amh_render *R, void *ws, size_t ws_bytes, void *stream) {
    if (!graph || !render_args_ok(R) || !ws || !stream) {
        set_error("amh_render_graph_create: invalid argument (a created stream is required)");
        return AMH_E_ARG;
    }
    *graph = nullptr;
    const Layout L = layout(R->width, R->height, R->wtot);
    if (ws_bytes < L.total) {
        set_error("amh_render_graph_create: workspace %zu < %zu bytes", ws_bytes, L.total);
        return AMH_E_ARG;
    }
    *graph = new amh_render_graph_s{*R, static_cast<char *>(ws), L};
    return AMH_OK;
}

extern "C" int amh_render_graph_frame(void *graph, double t, uint32_t *out, void *stream) {
    amh_render_graph_s *g = static_cast<amh_render_graph_s *>(graph);
    if (!g || !out) {
        set_error("amh_render_graph_frame: invalid argument");
        return AMH_E_ARG;
    }
    return render_frame_on(&g->R, t, g->ws, g->L, out, static_cast<hipStream_t>(stream));
}

extern "C" int amh_render_graph_destroy(void *graph) {
    amh_render_graph_s *g = static_cast<amh_render_graph_s *>(graph);
    if (!g) return AMH_OK;
    (void)hipDeviceSynchronize();  // frames may still be queued on the caller's stream
    delete g;
    return AMH_OK;
}
