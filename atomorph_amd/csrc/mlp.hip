// The learned proposal's MLP on the CDNA4 matrix cores.
//
// 8 -> 128 -> 128 -> 128 -> 128 -> 2, exact GELU after each hidden layer.
// Parameters are kept as FP32 masters (Adam state beside them) and as
// bfloat16 images in the order the matrix operands are read; every product
// takes bfloat16 operands and accumulates in FP32.  Inference (k_mlp_fused)
// and the training step (k_train: forward, backward and weight gradients)
// are one kernel each, with the activations in registers and LDS.
// The packed parameter layout (W row-major [in][out] then b, per layer) is
// the one the oracle and the host API use.
#include "common.h"
#include "../../include/atomorph_hip.h"

#include <cmath>
#include <cstring>
#include <vector>

using amh::check_hip;
using amh::set_error;

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int kIn = 8, kH = 128, kOut = 2;
constexpr int kDims[6] = {kIn, kH, kH, kH, kH, kOut};  // (constant indices only: in a kernel others read scratch)
constexpr int kParams = 50946;
constexpr int kLayers = 5;

__host__ __device__ constexpr size_t w_off(int l) {
    return l == 0 ? 0 : w_off(l - 1) + size_t(kDims[l - 1]) * kDims[l] + kDims[l];
}
__host__ __device__ constexpr size_t b_off(int l) { return w_off(l) + size_t(kDims[l]) * kDims[l + 1]; }
static_assert(b_off(4) + kOut == kParams, "parameter layout");

// FP32 -> bfloat16 bits, round to nearest even (v_cvt_pk_bf16_f32)
__device__ __forceinline__ uint16_t to_bf16(float f) { return __builtin_bit_cast(uint16_t, static_cast<__bf16>(f)); }
// erf by Abramowitz & Stegun, Handbook of Mathematical Functions (1964),
// formula 7.1.26: for x >= 0, erf x = 1 - (a1 t + a2 t^2 + a3 t^3 + a4 t^4 +
// a5 t^5) exp(-x^2) with t = 1 / (1 + p x), |error| <= 1.5e-7; odd in x.
// About a third of the instructions of erff, and the GELUs (4 x 128 per
// row) are what bounds the fused forward; the activations are rounded to
// bfloat16 (2^-8 relative) right after.
__device__ __forceinline__ float erf_as(float x) {
    const float ax = fabsf(x);
    const float t = __builtin_amdgcn_rcpf(fmaf(0.3275911f, ax, 1.0f));
    float poly = fmaf(t, 1.061405429f, -1.453152027f);
    poly = fmaf(t, poly, 1.421413741f);
    poly = fmaf(t, poly, -0.284496736f);
    poly = fmaf(t, poly, 0.254829592f);
    poly *= t;
    const float y = fmaf(-poly, __expf(-ax * ax), 1.0f);
    return copysignf(y, x);
}
__device__ __forceinline__ float gelu(float z) { return z * fmaf(0.5f, erf_as(z * 0.70710678118654752f), 0.5f); }
// gelu(z) and its derivative d = cdf + z pdf; erf's exponential exp(-z^2 / 2)
// is the density's too.
__device__ __forceinline__ float gelu_and_d(float z, float &d) {
    const float ax = fabsf(z * 0.70710678118654752f);
    const float t = __builtin_amdgcn_rcpf(fmaf(0.3275911f, ax, 1.0f));
    float poly = fmaf(t, 1.061405429f, -1.453152027f);
    poly = fmaf(t, poly, 1.421413741f);
    poly = fmaf(t, poly, -0.284496736f);
    poly = fmaf(t, poly, 0.254829592f);
    poly *= t;
    const float e = __expf(-ax * ax);
    const float cdf = 0.5f * (1.0f + copysignf(fmaf(-poly, e, 1.0f), z));
    d = fmaf(z, e * 0.39894228040143268f, cdf);
    return z * cdf;
}

// ---------------------------------------------------------- plain product
// c[M][N] = a[M][K] b[K][N], operands rounded to bfloat16, FP32 out: for
// amh_mlp_gemm_test alone, which pins the operand and accumulator layout of the
// 32x32x16 instruction that k_mlp_fused rests on.  Block tile 64 x 64 (2 x 2
// waves of 32 x 32), K staged 32 at a time in LDS as As[m][k] and Bs[n][k], so
// each lane's operand is 16 contiguous bytes: lane l holds row/column l % 32
// and k = 8 * (l / 32) + 0..7; the accumulator's register r of lane l is
// row 8 * (r / 4) + 4 * (l / 32) + r % 4, column l % 32.
constexpr int kBM = 64, kBN = 64, kBK = 32, kPadK = kBK + 8;

__global__ __launch_bounds__(256) void k_gemm(const float *__restrict__ a, const float *__restrict__ b,
                                              float *__restrict__ c, int M, int N, int K) {
    __shared__ __attribute__((aligned(16))) uint16_t As[kBM][kPadK];
    __shared__ __attribute__((aligned(16))) uint16_t Bs[kBN][kPadK];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int m0 = blockIdx.x * kBM, n0 = blockIdx.y * kBN;
    floatx16 acc;
    for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
    const int sr = t >> 2, sk = (t & 3) * 8, m = m0 + sr, n = n0 + sr;  // staging: row sr, k sk..sk+7
    for (int k0 = 0; k0 < K; k0 += kBK) {
        alignas(16) uint16_t va[8], vb[8];
        for (int j = 0; j < 8; ++j) {
            const int k = k0 + sk + j;
            va[j] = (m < M && k < K) ? to_bf16(a[int64_t(m) * K + k]) : uint16_t(0);
            vb[j] = (n < N && k < K) ? to_bf16(b[int64_t(k) * N + n]) : uint16_t(0);
        }
        *reinterpret_cast<uint4 *>(&As[sr][sk]) = *reinterpret_cast<const uint4 *>(va);
        *reinterpret_cast<uint4 *>(&Bs[sr][sk]) = *reinterpret_cast<const uint4 *>(vb);
        __syncthreads();
        for (int ks = 0; ks < kBK; ks += 16) {
            const int kk = ks + 8 * (lane >> 5);
            const bf16x8 fa = *reinterpret_cast<const bf16x8 *>(&As[wm * 32 + (lane & 31)][kk]);
            const bf16x8 fb = *reinterpret_cast<const bf16x8 *>(&Bs[wn * 32 + (lane & 31)][kk]);
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa, fb, acc, 0, 0, 0);
        }
        __syncthreads();
    }
    const int col = n0 + wn * 32 + (lane & 31);
    for (int r = 0; r < 16; ++r) {
        const int row = m0 + wm * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
        if (row < M && col < N) c[int64_t(row) * N + col] = acc[r];
    }
}

// ------------------------------------------------------- training images
typedef float floatx4 __attribute__((ext_vector_type(4)));

// The weights as A operands of v_mfma_f32_16x16x32_bf16 (lane l: row l % 16, k =
// 8 (l / 16) + 0..7), for products whose B operand is the accumulator of the
// layer before: k slot j of lane group g in K step ks is feature
// 32 ks + 16 (j / 4) + 4 g + j % 4.  The seven products of the step in their
// order: forward Z^T = W^T A^T of layers 1 (its K padded 8 -> 128 with zeros)
// to 4, backward dA^T = W dZ^T of layers 4 to 2; then layer 5's two products,
// its 2 outputs padded with zeros.
constexpr int kProducts = 7;
struct TrainImage {
    uint16_t w[kProducts][8][4][64][8];
    uint16_t w5f[4][64][8];
    uint16_t w5b[8][64][8];
};

__device__ __forceinline__ int k_step(int f) { return f / 32; }
__device__ __forceinline__ int k_group(int f) { return f % 16 / 4; }
__device__ __forceinline__ int k_slot(int f) { return 4 * (f % 32 / 16) + f % 4; }

// Parameter i's bfloat16 value v into the images that hold it.
template <int l>
__device__ __forceinline__ void put_layer(TrainImage *T, int i, uint16_t v) {
    constexpr int dout = kDims[l + 1], size = kDims[l] * dout;
    const int k = i - int(w_off(l));
    if (k < 0 || k >= size) return;
    const int in = k / dout, out = k % dout;
    if constexpr (l == 0) {  // (the inputs are not an accumulator: feature k in slot k of group 0)
        T->w[0][out / 16][0][out % 16][in] = v;
    } else if constexpr (l < kLayers - 1) {
        T->w[l][out / 16][k_step(in)][16 * k_group(in) + out % 16][k_slot(in)] = v;
        T->w[7 - l][in / 16][k_step(out)][16 * k_group(out) + in % 16][k_slot(out)] = v;
    } else {
        T->w5f[k_step(in)][16 * k_group(in) + out][k_slot(in)] = v;
        T->w5b[in / 16][in % 16][out] = v;
    }
}
__device__ __forceinline__ void put_image(TrainImage *T, int i, uint16_t v) {
    put_layer<0>(T, i, v);
    put_layer<1>(T, i, v);
    put_layer<2>(T, i, v);
    put_layer<3>(T, i, v);
    put_layer<4>(T, i, v);
}

// New parameters: the bfloat16 copies, and no Adam state.
__global__ void k_set_params(const float *__restrict__ p, uint16_t *__restrict__ pb, TrainImage *__restrict__ T,
                             float *__restrict__ m, float *__restrict__ v, int n) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    pb[i] = to_bf16(p[i]);
    put_image(T, i, pb[i]);
    m[i] = v[i] = 0.0f;
}

// Adam (Kingma & Ba 2015) on the FP32 masters; refreshes the bfloat16 copies.
__global__ void k_adam(float *__restrict__ p, uint16_t *__restrict__ pb, TrainImage *__restrict__ T,
                       const float *__restrict__ g, float *__restrict__ m, float *__restrict__ v, int n, float lr,
                       float b1, float b2, float eps, float c1, float c2) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.0f - b1) * gi;
    const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float pi = p[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    p[i] = pi;
    pb[i] = to_bf16(pi);
    put_image(T, i, pb[i]);
}

// ------------------------------------------------------- fused forward
// Inference in one kernel with the activations kept in registers: each wave
// computes 32 rows at a time as Z^T = W^T A^T, so the accumulator of one
// layer (lane = row l % 32, registers = output features) is already the
// next layer's B operand once its K order is permuted to match:
//   MFMA k = 16 ks + 8 (l / 32) + j  <->  feature feat(ks, l / 32, j)
// and the weights are staged into LDS in that order (A operands, 16 bytes
// per lane).  Layer 1 pads K 8 -> 16 with zeros, the output layer pads its
// 2 rows to 32.  LDS: 4 + 3 x 32 + 8 KB of weights, 2 KB of biases.
__host__ __device__ constexpr int feat(int ks, int h, int j) {
    return 32 * (ks / 2) + 16 * (ks % 2) + 8 * (j / 4) + 4 * h + (j % 4);
}
struct FusedLds {
    bf16x8 w1[4][64];
    bf16x8 wh[3][4][8][64];
    bf16x8 w5[8][64];
    float b[4][kH];
    float b5[kOut];
};
constexpr size_t kFusedLds = sizeof(FusedLds);
static_assert(kFusedLds % 16 == 0, "LDS image copied in 16-byte units");

__device__ __forceinline__ bf16x8 pack8(const uint16_t *v) {
    bf16x8 r;
    __builtin_memcpy(&r, v, 16);
    return r;
}

// The LDS image of the weights in MFMA operand order (built once per
// parameter change into global memory; the fused kernel copies it).
__global__ __launch_bounds__(256) void k_fused_stage(const uint16_t *__restrict__ pb, const float *__restrict__ p,
                                                    FusedLds *__restrict__ S) {
    const int t = blockIdx.x * 256 + threadIdx.x, nt = gridDim.x * 256;
    for (int e = t; e < 4 * 64; e += nt) {
        const int mb = e / 64, l = e % 64, lh = l >> 5, lm = l & 31;
        uint16_t v[8];
        for (int j = 0; j < 8; ++j) v[j] = lh == 0 ? pb[w_off(0) + j * kH + mb * 32 + lm] : uint16_t(0);
        S->w1[mb][l] = pack8(v);
    }
    for (int e = t; e < 3 * 4 * 8 * 64; e += nt) {
        const int li = e / (4 * 8 * 64), mb = (e / (8 * 64)) % 4, ks = (e / 64) % 8, l = e % 64;
        const int lh = l >> 5, lm = l & 31;
        uint16_t v[8];
        for (int j = 0; j < 8; ++j) v[j] = pb[w_off(li + 1) + size_t(feat(ks, lh, j)) * kH + mb * 32 + lm];
        S->wh[li][mb][ks][l] = pack8(v);
    }
    for (int e = t; e < 8 * 64; e += nt) {
        const int ks = e / 64, l = e % 64, lh = l >> 5, lm = l & 31;
        uint16_t v[8];
        for (int j = 0; j < 8; ++j) v[j] = lm < kOut ? pb[w_off(4) + size_t(feat(ks, lh, j)) * kOut + lm] : uint16_t(0);
        S->w5[ks][l] = pack8(v);
    }
    for (int e = t; e < 4 * kH; e += nt) S->b[e / kH][e % kH] = p[b_off(e / kH) + e % kH];
    if (t < kOut) S->b5[t] = p[b_off(4) + t];
}

constexpr int kFusedThreads = 1024;  // 16 waves (4 per SIMD, <= 128 registers each) share one copy of the weights

// Bias + GELU of one 32-feature output block (accumulator layout: feature
// 8*(r/4) + 4*h + r%4 of block mb) -> the two B operands it feeds.
__device__ __forceinline__ void gelu_block(const floatx16 &acc, const float *__restrict__ bias, int mb, int h,
                                           bf16x8 &lo, bf16x8 &hi) {
    uint16_t v[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) v[r] = to_bf16(gelu(acc[r] + bias[mb * 32 + 8 * (r >> 2) + 4 * h + (r & 3)]));
    lo = pack8(v);
    hi = pack8(v + 8);
}

__global__ __launch_bounds__(kFusedThreads) void k_mlp_fused(const float *__restrict__ x, int64_t n,
                                                  const FusedLds *__restrict__ image, float *__restrict__ out) {
    extern __shared__ __attribute__((aligned(16))) char lds_raw[];
    FusedLds &S = *reinterpret_cast<FusedLds *>(lds_raw);
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6, h = lane >> 5, m = lane & 31;
    {
        const uint4 *src = reinterpret_cast<const uint4 *>(image);
        uint4 *dst = reinterpret_cast<uint4 *>(lds_raw);
        for (size_t e = t; e < kFusedLds / 16; e += kFusedThreads) dst[e] = src[e];
    }
    __syncthreads();

    const int64_t tiles = (n + 31) / 32;
    constexpr int kWaves = kFusedThreads / 64;
    // (a last turn that is not full leaves every workgroup some waves, not
    // some workgroups none: 229k rows, 1.75 turns, 87 -> 73 us.  GELU, 94 of
    // a SIMD's cycles for 64 values, bounds the rest.)
    for (int64_t tile = int64_t(wave) * gridDim.x + blockIdx.x; tile < tiles; tile += int64_t(gridDim.x) * kWaves) {
        const int64_t row = tile * 32 + m;
        uint16_t xin[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) xin[j] = (h == 0 && row < n) ? to_bf16(x[row * kIn + j]) : uint16_t(0);
        const bf16x8 xa = pack8(xin);
        // Layer 1 (K = 8 in one MFMA), two output blocks at a time: each
        // pair is finished (bias, GELU) before the next starts, so only two
        // accumulators are live.
        bf16x8 B[8], Bn[8];
#pragma unroll
        for (int mp = 0; mp < 2; ++mp) {
            floatx16 a0, a1;
#pragma unroll
            for (int r = 0; r < 16; ++r) a0[r] = a1[r] = 0.0f;
            a0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(S.w1[2 * mp][lane], xa, a0, 0, 0, 0);
            a1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(S.w1[2 * mp + 1][lane], xa, a1, 0, 0, 0);
            gelu_block(a0, S.b[0], 2 * mp, h, B[4 * mp], B[4 * mp + 1]);
            gelu_block(a1, S.b[0], 2 * mp + 1, h, B[4 * mp + 2], B[4 * mp + 3]);
            __builtin_amdgcn_sched_barrier(0);  // keep the pairs apart: bounded register use
        }
        // Hidden layers 2-4: B (this layer's input) -> Bn, then swap.
#pragma unroll 1
        for (int li = 0; li < 3; ++li) {
#pragma unroll
            for (int mp = 0; mp < 2; ++mp) {
                floatx16 a0, a1;
#pragma unroll
                for (int r = 0; r < 16; ++r) a0[r] = a1[r] = 0.0f;
#pragma unroll
                for (int ks = 0; ks < 8; ++ks) {
                    a0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(S.wh[li][2 * mp][ks][lane], B[ks], a0, 0, 0, 0);
                    a1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(S.wh[li][2 * mp + 1][ks][lane], B[ks], a1, 0, 0, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
                gelu_block(a0, S.b[li + 1], 2 * mp, h, Bn[4 * mp], Bn[4 * mp + 1]);
                gelu_block(a1, S.b[li + 1], 2 * mp + 1, h, Bn[4 * mp + 2], Bn[4 * mp + 3]);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int ks = 0; ks < 8; ++ks) B[ks] = Bn[ks];
        }
        floatx16 o;
#pragma unroll
        for (int r = 0; r < 16; ++r) o[r] = 0.0f;
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) o = __builtin_amdgcn_mfma_f32_32x32x16_bf16(S.w5[ks][lane], B[ks], o, 0, 0, 0);
        if (h == 0 && row < n) {  // rows 0 and 1 of the output block: registers 0 and 1
            out[row * kOut + 0] = o[0] + S.b5[0];
            out[row * kOut + 1] = o[1] + S.b5[1];
        }
    }
}

// --------------------------------------------------------- training step
// Forward, backward and weight gradients of kTrainRows rows per workgroup and
// turn, 16 per wave: Z^T = W^T A^T, so a layer's accumulator (lane = row,
// registers = features) is the next product's B operand, forward and
// backward, and never leaves the registers.  GELU' of the four hidden layers
// waits there too, in FP32, from the forward pass for the backward.  The
// weight gradients dW = A^T dZ contract over the rows: each layer's A and dZ
// are put into LDS as bfloat16 (what the product rounds them to) with the
// rows of a feature consecutive, and each wave computes 32 columns of dW.
// Bias gradients are FP32 sums of the unrounded dZ.  Each workgroup leaves
// its partial gradient (stored in its first turn, added to in later ones) and
// loss for k_train_reduce.
//
// One wave per SIMD (512 registers).  The layers are loops, not unrolled: at
// the trainer's 16,384 rows each CU has one turn of one workgroup, which
// would wait for 68 KB of straight-line code (78 us; as loops 69, and 43 with
// the weights' registers named, see below).  GELU' moves through the four
// register arrays by copies.  What is left is about a third of it VALU work,
// the rest the layers' dependent chain and the 52 MB of partials.  The step
// with k_train_reduce (12 us, at the memory's rate) takes 55 us; with one
// tiled product per layer and direction, atomics for the split weight
// gradients and the activations in memory it took 708.
constexpr int kTrainRows = 64, kTrainThreads = 256;
constexpr int kRowPad = kTrainRows + 8;  // 144 bytes per feature: 16 lanes' 16-byte reads hit distinct banks
constexpr int kPart = kParams + 1;       // partial gradient, then the loss

struct TrainLds {
    bf16x8 w[8][4][64];          // the current product's weights
    uint16_t a[4][kH][kRowPad];  // A1..A4
    uint16_t dz[kH][kRowPad];    // the current layer's dZ
    uint16_t x[16][kRowPad];     // the inputs (rows 8..15 zero)
    uint16_t d5[16][kRowPad];    // dZ5 (rows 2..15 zero)
    float b[4][kH];
    float db[4][4][kH];          // per wave: bias gradients of the hidden layers
    float db5[4][kOut];
    float loss[4];
};
static_assert(sizeof(TrainLds) <= 160 * 1024, "one workgroup per CU");

__device__ __forceinline__ floatx4 mfma16(const bf16x8 &a, const bf16x8 &b, const floatx4 &c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// Sum over each row of 16 lanes, in its last lane.
template <int CTRL>
__device__ __forceinline__ float row_shr(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, false));
}
__device__ __forceinline__ float row_sum(float v) {
    v += row_shr<0x111>(v);
    v += row_shr<0x112>(v);
    v += row_shr<0x114>(v);
    v += row_shr<0x118>(v);
    return v;
}

// A layer's 32 values of this lane (its row, features 16 mb + 4 g + r) ->
// B operands, and into LDS with the rows of a feature consecutive.
__device__ __forceinline__ void to_operands(const float (&v)[32], bf16x8 (&B)[4], uint16_t (*lds)[kRowPad], int g,
                                            int row) {
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        uint16_t q[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            q[j] = to_bf16(v[8 * s + j]);
            lds[32 * s + 16 * (j / 4) + 4 * g + j % 4][row] = q[j];
        }
        B[s] = pack8(q);
    }
}

__global__ __launch_bounds__(kTrainThreads) __attribute__((amdgpu_waves_per_eu(1, 1))) void k_train(
    const float *__restrict__ x, const float *__restrict__ t, int n, const TrainImage *__restrict__ T,
    const float *__restrict__ p, float *__restrict__ part) {
    extern __shared__ __attribute__((aligned(16))) char lds_raw[];
    TrainLds &S = *reinterpret_cast<TrainLds *>(lds_raw);
    const int tid = threadIdx.x, wave = tid >> 6;
    for (int e = tid; e < 16 * kRowPad; e += kTrainThreads) (&S.x[0][0])[e] = (&S.d5[0][0])[e] = 0;
    constexpr int kStride = kH * kH + kH;  // from one hidden layer's biases to the next's
    for (int e = tid; e < 4 * kH; e += kTrainThreads) S.b[e / kH][e % kH] = p[b_off(0) + e / kH * kStride + e % kH];
    for (int e = tid; e < 16 * kH; e += kTrainThreads) (&S.db[0][0][0])[e] = 0.0f;
    const float b50 = p[b_off(4)], b51 = p[b_off(4) + 1];
    const bf16x8 *w5f = reinterpret_cast<const bf16x8 *>(T->w5f), *w5b = reinterpret_cast<const bf16x8 *>(T->w5b);
    // the products' weights pass through S.w; each is loaded into registers
    // during the product before
    // (eight named registers: an array here went to scratch memory, whose
    // stores waited for the loads)
    static_assert(sizeof(S.w) == 8 * 16 * kTrainThreads, "eight 16-byte loads per thread");
    uint4 pre0, pre1, pre2, pre3, pre4, pre5, pre6, pre7;
    const auto prefetch = [&](int k) {
        const uint4 *src = reinterpret_cast<const uint4 *>(T->w[k]) + tid;
        pre0 = src[0], pre1 = src[kTrainThreads], pre2 = src[2 * kTrainThreads], pre3 = src[3 * kTrainThreads];
        src += 4 * kTrainThreads;
        pre4 = src[0], pre5 = src[kTrainThreads], pre6 = src[2 * kTrainThreads], pre7 = src[3 * kTrainThreads];
    };
    const auto stage = [&] {
        uint4 *dst = reinterpret_cast<uint4 *>(S.w) + tid;
        dst[0] = pre0, dst[kTrainThreads] = pre1, dst[2 * kTrainThreads] = pre2, dst[3 * kTrainThreads] = pre3;
        dst += 4 * kTrainThreads;
        dst[0] = pre4, dst[kTrainThreads] = pre5, dst[2 * kTrainThreads] = pre6, dst[3 * kTrainThreads] = pre7;
    };

    const floatx4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    float *out = part + size_t(blockIdx.x) * kPart;
    float loss = 0.0f, db50 = 0.0f, db51 = 0.0f;
    const float inv_n = 1.0f / float(n);
    prefetch(0);
    __syncthreads();

    const int tiles = (n + kTrainRows - 1) / kTrainRows;
#pragma unroll 1
    for (int tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        const int lane = tid & 63, g = lane >> 4, c = lane & 15;
        const int lr = 16 * wave + c;  // this lane's row of the workgroup's rows
        const int64_t row = int64_t(tile) * kTrainRows + lr;
        const bool valid = row < n, again = tile != int(blockIdx.x);
        // a weight gradient of this turn into the workgroup's partial
        const auto put = [&](uint32_t at, float v) { out[at] = again ? out[at] + v : v; };
        bf16x8 B[4];
        {
            uint16_t q[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) q[j] = (g == 0 && valid) ? to_bf16(x[row * kIn + j]) : uint16_t(0);
            if (g == 0)
#pragma unroll
                for (int j = 0; j < 8; ++j) S.x[j][lr] = q[j];
            B[0] = pack8(q);
#pragma unroll
            for (int j = 0; j < 8; ++j) q[j] = 0;
            B[1] = B[2] = B[3] = pack8(q);
        }
        float gd[4][32];  // gelu' of hidden layers 1..4 (the newest in gd[3])
#pragma unroll
        for (int k = 0; k < 32; ++k) gd[1][k] = gd[2][k] = gd[3][k] = 0.0f;
#pragma unroll 1
        for (int l = 0; l < 4; ++l) {
            stage();
            prefetch(l + 1);
            __syncthreads();
#pragma unroll
            for (int k = 0; k < 32; ++k) {
                gd[0][k] = gd[1][k];
                gd[1][k] = gd[2][k];
                gd[2][k] = gd[3][k];
            }
            float a[32];
#pragma unroll
            for (int mb = 0; mb < 8; mb += 4) {
                floatx4 z[4] = {zero, zero, zero, zero};
#pragma unroll
                for (int ks = 0; ks < 4; ++ks)
#pragma unroll
                    for (int q = 0; q < 4; ++q) z[q] = mfma16(S.w[mb + q][ks][lane], B[ks], z[q]);
#pragma unroll
                for (int q = 0; q < 4; ++q)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int k = 4 * (mb + q) + r;
                        a[k] = gelu_and_d(z[q][r] + S.b[l][16 * (mb + q) + 4 * g + r], gd[3][k]);
                    }
            }
            to_operands(a, B, S.a[l], g, lr);
            __syncthreads();  // S.w is free
        }
        // output, loss, dZ5 (lanes of group 0 hold their row's two values)
        floatx4 o = zero;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) o = mfma16(w5f[ks * 64 + lane], B[ks], o);
        float d0 = 0.0f, d1 = 0.0f;
        if (g == 0 && valid) {
            d0 = o[0] + b50 - t[row * kOut];
            d1 = o[1] + b51 - t[row * kOut + 1];
        }
        loss += (d0 * d0 + d1 * d1) * inv_n;
        d0 *= 2.0f * inv_n;
        d1 *= 2.0f * inv_n;
        db50 += d0;
        db51 += d1;
        uint16_t q5[8] = {to_bf16(d0), to_bf16(d1), 0, 0, 0, 0, 0, 0};
        if (g == 0) {
            S.d5[0][lr] = q5[0];
            S.d5[1][lr] = q5[1];
        }
        const bf16x8 b5 = pack8(q5);  // (zero outside group 0)
        float dz[32];
#pragma unroll
        for (int mb = 0; mb < 8; ++mb) {
            const floatx4 da = mfma16(w5b[mb * 64 + lane], b5, zero);
#pragma unroll
            for (int r = 0; r < 4; ++r) dz[4 * mb + r] = da[r] * gd[3][4 * mb + r];
        }
        __syncthreads();  // S.a and S.d5 are complete
        // dW5 = A4^T dZ5, this wave's 32 rows
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            floatx4 v = zero;
#pragma unroll
            for (int ks = 0; ks < 2; ++ks)
                v = mfma16(*reinterpret_cast<const bf16x8 *>(&S.a[3][32 * wave + 16 * k + c][32 * ks + 8 * g]),
                           *reinterpret_cast<const bf16x8 *>(&S.d5[c][32 * ks + 8 * g]), v);
            if (c < kOut)
#pragma unroll
                for (int r = 0; r < 4; ++r) put(uint32_t(w_off(4)) + (32 * wave + 16 * k + 4 * g + r) * kOut + c, v[r]);
        }
        // dZ of hidden layer l + 1: the gradients of its weights (input: A of
        // layer l, or x) and biases, then the dZ below
#pragma unroll 1
        for (int l = 3; l >= 0; --l) {
            to_operands(dz, B, S.dz, g, lr);
#pragma unroll
            for (int k = 0; k < 32; ++k) {
                const float s = row_sum(dz[k]);
                if (c == 15) atomicAdd(&S.db[wave][l][16 * (k / 4) + 4 * g + k % 4], s);  // (no other adds here)
            }
            if (l > 0) {
                stage();
                prefetch(l > 1 ? 8 - l : 0);  // products 4, 5, 6 are staged at l = 3, 2, 1
            }
            __syncthreads();
            if (l > 0) {
#pragma unroll
                for (int mb = 0; mb < 8; mb += 4) {
                    floatx4 z[4] = {zero, zero, zero, zero};
#pragma unroll
                    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
                        for (int q = 0; q < 4; ++q) z[q] = mfma16(S.w[mb + q][ks][lane], B[ks], z[q]);
#pragma unroll
                    for (int q = 0; q < 4; ++q)
#pragma unroll
                        for (int r = 0; r < 4; ++r) dz[4 * (mb + q) + r] = z[q][r] * gd[2][4 * (mb + q) + r];
                }
#pragma unroll
                for (int k = 0; k < 32; ++k) {
                    gd[2][k] = gd[1][k];
                    gd[1][k] = gd[0][k];
                }
            }
            // dW = A^T dZ over the workgroup's rows, this wave's 32 columns
            bf16x8 bz[2][2];
#pragma unroll
            for (int ks = 0; ks < 2; ++ks)
#pragma unroll
                for (int nb = 0; nb < 2; ++nb)
                    bz[ks][nb] = *reinterpret_cast<const bf16x8 *>(&S.dz[32 * wave + 16 * nb + c][32 * ks + 8 * g]);
            const uint16_t(*a)[kRowPad] = l > 0 ? S.a[l - 1] : S.x;
            uint32_t at = (l == 0 ? uint32_t(w_off(0)) : uint32_t(w_off(1)) + uint32_t(l - 1) * kStride) +
                          uint32_t(4 * g * kH + 32 * wave + c);
            const bool rows = l > 0 || g < 2;
#pragma unroll 2
            for (int mb = 0; mb < (l > 0 ? 8 : 1); ++mb, at += 16 * kH) {
                const bf16x8 a0 = *reinterpret_cast<const bf16x8 *>(&a[16 * mb + c][8 * g]);
                const bf16x8 a1 = *reinterpret_cast<const bf16x8 *>(&a[16 * mb + c][32 + 8 * g]);
#pragma unroll
                for (int nb = 0; nb < 2; ++nb) {
                    const floatx4 v = mfma16(a1, bz[1][nb], mfma16(a0, bz[0][nb], zero));
                    if (rows)
#pragma unroll
                        for (int r = 0; r < 4; ++r) put(at + uint32_t(r * kH + 16 * nb), v[r]);
                }
            }
            __syncthreads();  // S.dz and S.w are free
        }
    }

    loss = row_sum(loss);
    db50 = row_sum(db50);
    db51 = row_sum(db51);
    if ((tid & 63) == 15) {
        S.loss[wave] = loss;
        S.db5[wave][0] = db50;
        S.db5[wave][1] = db51;
    }
    __syncthreads();
    for (int e = tid; e < 4 * kH; e += kTrainThreads) {
        const int l = e / kH, f = e % kH;
        out[b_off(0) + l * kStride + f] = (S.db[0][l][f] + S.db[1][l][f]) + (S.db[2][l][f] + S.db[3][l][f]);
    }
    if (tid < kOut) out[b_off(4) + tid] = (S.db5[0][tid] + S.db5[1][tid]) + (S.db5[2][tid] + S.db5[3][tid]);
    if (tid == 0) out[kParams] = (S.loss[0] + S.loss[1]) + (S.loss[2] + S.loss[3]);
}

// The workgroups' partial gradients summed in FP32, in a fixed order: 64
// parameters per block, a quarter of the partials per wave.
__global__ __launch_bounds__(256) void k_train_reduce(const float *__restrict__ part, int parts,
                                                     float *__restrict__ g, float *__restrict__ grad,
                                                     float *__restrict__ loss) {
    __shared__ float sum[4][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int i = blockIdx.x * 64 + lane;
    float s[8] = {};
    if (i < kPart) {
        int k = wave;
        for (; k + 28 < parts; k += 32)
#pragma unroll
            for (int j = 0; j < 8; ++j) s[j] += part[size_t(k + 4 * j) * kPart + i];
        for (; k < parts; k += 4) s[0] += part[size_t(k) * kPart + i];
    }
    sum[wave][lane] = ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]));
    __syncthreads();
    if (wave != 0 || i >= kPart) return;
    const float v = (sum[0][lane] + sum[1][lane]) + (sum[2][lane] + sum[3][lane]);
    if (i < kParams) {
        g[i] = v;
        if (grad) grad[i] = v;
    } else if (loss) {
        atomicAdd(loss, v);  // (other handles' steps, on other streams, may add to it too)
    }
}

}  // namespace

// ------------------------------------------------------------- handle
struct amh_mlp_s {
    int32_t batch = 0;
    int cus = 0;  // of the device the handle was made on
    void *buf = nullptr;
    float *p = nullptr, *g = nullptr, *m = nullptr, *v = nullptr;  // [kParams]
    uint16_t *pb = nullptr;                                         // bfloat16 copy
    FusedLds *image = nullptr;  // weights in the fused forward's LDS order
    bool image_stale = true;
    TrainImage *train = nullptr;  // weights in the training step's operand order
    float *part = nullptr;        // [workgroups][kPart] partial gradients
    int64_t step = 0;
};

namespace {
// Readies the current device for the fused kernels (110 KB and 137 KB of LDS in
// one workgroup) and counts its CUs.  Each handle asks for itself: handles may
// be made from several threads at once and on several devices.
int fused_kernels(int &cus) {
    const char *what = "amh_mlp_create: the kernels' LDS";
    int dev = 0;
    int r = check_hip(hipGetDevice(&dev), what);
    if (!r) r = check_hip(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev), what);
    if (!r)
        r = check_hip(hipFuncSetAttribute(reinterpret_cast<const void *>(&k_mlp_fused),
                                          hipFuncAttributeMaxDynamicSharedMemorySize, int(kFusedLds)),
                      what);
    if (!r)
        r = check_hip(hipFuncSetAttribute(reinterpret_cast<const void *>(&k_train),
                                          hipFuncAttributeMaxDynamicSharedMemorySize, int(sizeof(TrainLds))),
                      what);
    return r;
}

// Workgroups of the training step on n rows: one per CU at most.
int train_groups(int cus, int n) { return std::min(cus, (n + kTrainRows - 1) / kTrainRows); }

int stage_image(amh_mlp_s *M, hipStream_t s) {
    hipLaunchKernelGGL(k_fused_stage, dim3(64), dim3(256), 0, s, M->pb, M->p, M->image);
    M->image_stale = false;
    return AMH_OK;
}
}  // namespace

extern "C" int amh_mlp_create(void **mlp, int32_t batch_max, void *stream) {
    if (!mlp || batch_max <= 0 || batch_max > (1 << 22)) {
        set_error("amh_mlp_create: invalid argument");
        return AMH_E_ARG;
    }
    int cus = 0;
    if (int r = fused_kernels(cus)) return r;
    amh_mlp_s *M = new amh_mlp_s;
    M->batch = batch_max;
    M->cus = cus;
    const auto al = [](size_t b) { return (b + 255) & ~size_t(255); };
    const size_t vec = al(kParams * 4), half = al(kParams * 2), train = al(sizeof(TrainImage));
    const size_t held = 4 * vec + half + al(kFusedLds) + train;
    if (int r = check_hip(hipMalloc(&M->buf, held + size_t(train_groups(cus, batch_max)) * kPart * 4), "amh_mlp_create")) {
        delete M;
        return r;
    }
    char *q = static_cast<char *>(M->buf);
    const auto take = [&](size_t b) { char *r = q; q += b; return r; };
    M->p = reinterpret_cast<float *>(take(vec));
    M->g = reinterpret_cast<float *>(take(vec));
    M->m = reinterpret_cast<float *>(take(vec));
    M->v = reinterpret_cast<float *>(take(vec));
    M->pb = reinterpret_cast<uint16_t *>(take(half));
    M->image = reinterpret_cast<FusedLds *>(take(al(kFusedLds)));
    M->train = reinterpret_cast<TrainImage *>(take(train));
    M->part = reinterpret_cast<float *>(q);
    if (int r = check_hip(hipMemsetAsync(M->buf, 0, held, static_cast<hipStream_t>(stream)), "amh_mlp_create")) {
        (void)hipFree(M->buf);
        delete M;
        return r;
    }
    *mlp = M;
    return AMH_OK;
}

extern "C" int amh_mlp_destroy(void *mlp) {
    amh_mlp_s *M = static_cast<amh_mlp_s *>(mlp);
    if (!M) return AMH_OK;
    if (M->buf) (void)hipFree(M->buf);
    delete M;
    return AMH_OK;
}

extern "C" int amh_mlp_set_params(void *mlp, const float *host, void *stream) {
    amh_mlp_s *M = static_cast<amh_mlp_s *>(mlp);
    if (!M || !host) { set_error("amh_mlp_set_params: NULL"); return AMH_E_ARG; }
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (int r = check_hip(hipMemcpyAsync(M->p, host, kParams * 4, hipMemcpyHostToDevice, s), "set_params")) return r;
    hipLaunchKernelGGL(k_set_params, dim3((kParams + 255) / 256), dim3(256), 0, s, M->p, M->pb, M->train, M->m, M->v,
                       kParams);
    M->step = 0;
    stage_image(M, s);  // the forward's weight image, now rather than at the first forward
    AMH_LAUNCH_CHECK("amh_mlp_set_params");
    return check_hip(hipStreamSynchronize(s), "set_params");
}

extern "C" int amh_mlp_get_params(void *mlp, float *host, void *stream) {
    amh_mlp_s *M = static_cast<amh_mlp_s *>(mlp);
    if (!M || !host) { set_error("amh_mlp_get_params: NULL"); return AMH_E_ARG; }
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (int r = check_hip(hipMemcpyAsync(host, M->p, kParams * 4, hipMemcpyDeviceToHost, s), "get_params")) return r;
    return check_hip(hipStreamSynchronize(s), "get_params");
}

// Inference: out[n][2] for x[n][8].
extern "C" int amh_mlp_forward(void *mlp, const float *x, int64_t n, float *out, void *stream) {
    amh_mlp_s *M = static_cast<amh_mlp_s *>(mlp);
    if (!M || (n > 0 && (!x || !out)) || n < 0) { set_error("amh_mlp_forward: invalid argument"); return AMH_E_ARG; }
    hipStream_t s = static_cast<hipStream_t>(stream);
    amh::ProfScope ps_("mlp_forward", s);
    if (n == 0) return AMH_OK;
    const int64_t tiles = (n + 31) / 32;
    // from four waves' tiles a workgroup, one per SIMD, on more CUs first
    const uint32_t grid = uint32_t(std::min<int64_t>(M->cus, (tiles + 3) / 4));
    if (M->image_stale) stage_image(M, s);
    hipLaunchKernelGGL(k_mlp_fused, dim3(grid), dim3(kFusedThreads), kFusedLds, s, x, n, M->image, out);
    AMH_LAUNCH_CHECK("amh_mlp_forward");
    return AMH_OK;
}

// Gradient of mean_s sum_o (out - t)^2 over n <= batch samples into the
// handle's gradient buffer (and, if grad != NULL, a copy there); the loss
// is added to *loss_dev when it is not NULL.
extern "C" int amh_mlp_gradients(void *mlp, const float *x, const float *t, int32_t n, float *grad, float *loss_dev,
                                 void *stream) {
    amh_mlp_s *M = static_cast<amh_mlp_s *>(mlp);
    if (!M || !x || !t || n <= 0 || n > M->batch) { set_error("amh_mlp_gradients: invalid argument"); return AMH_E_ARG; }
    hipStream_t s = static_cast<hipStream_t>(stream);
    amh::ProfScope ps_("mlp_gradients", s);
    const int groups = train_groups(M->cus, n);
    hipLaunchKernelGGL(k_train, dim3(uint32_t(groups)), dim3(kTrainThreads), sizeof(TrainLds), s, x, t, int(n),
                       M->train, M->p, M->part);
    hipLaunchKernelGGL(k_train_reduce, dim3((kPart + 63) / 64), dim3(256), 0, s, M->part, groups, M->g, grad, loss_dev);
    AMH_LAUNCH_CHECK("amh_mlp_gradients");
    return AMH_OK;
}

// One Adam step with the handle's gradient buffer (from amh_mlp_gradients).
extern "C" int amh_mlp_adam_step(void *mlp, float lr, void *stream) {
    amh_mlp_s *M = static_cast<amh_mlp_s *>(mlp);
    if (!M || !(lr > 0.0f)) { set_error("amh_mlp_adam_step: invalid argument"); return AMH_E_ARG; }
    hipStream_t s = static_cast<hipStream_t>(stream);
    M->step += 1;
    M->image_stale = true;
    const float b1 = 0.9f, b2 = 0.999f;
    const float c1 = 1.0f - std::pow(b1, float(M->step)), c2 = 1.0f - std::pow(b2, float(M->step));
    hipLaunchKernelGGL(k_adam, dim3((kParams + 255) / 256), dim3(256), 0, s, M->p, M->pb, M->train, M->g, M->m, M->v,
                       kParams, lr, b1, b2, 1e-8f, c1, c2);
    AMH_LAUNCH_CHECK("amh_mlp_adam_step");
    return AMH_OK;
}

// Plain product for the test of the matrix instruction's layouts (k_gemm).
extern "C" int amh_mlp_gemm_test(const float *a, const float *b, float *c, int32_t M, int32_t N, int32_t K,
                                 void *stream) {
    if (!a || !b || !c || M <= 0 || N <= 0 || K <= 0) { set_error("amh_mlp_gemm_test: invalid argument"); return AMH_E_ARG; }
    hipLaunchKernelGGL(k_gemm, dim3(uint32_t((M + kBM - 1) / kBM), uint32_t((N + kBN - 1) / kBN)), dim3(256), 0,
                       static_cast<hipStream_t>(stream), a, b, c, M, N, K);
    AMH_LAUNCH_CHECK("amh_mlp_gemm_test");
    return AMH_OK;
}
