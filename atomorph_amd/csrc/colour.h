// Colour arithmetic of the morph engine, FP64 with the reference's
// operation order (compiled with -ffp-contract=off) so 8-bit results match.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace amh {

__host__ __device__ __forceinline__ uint32_t narrow8(double v) { return uint32_t(int32_t(v)) & 0xFFu; }
__host__ __device__ __forceinline__ uint32_t narrow16(double v) { return uint32_t(int32_t(v)) & 0xFFFFu; }
__host__ __device__ __forceinline__ uint32_t rgba_pack(uint32_t r, uint32_t g, uint32_t b, uint32_t a) {
    return (r & 255u) | ((g & 255u) << 8) | ((b & 255u) << 16) | ((a & 255u) << 24);
}

// Finley's HSP model (color.cpp:71-178, public-domain formulas): perceived
// brightness P = sqrt(.299 R^2 + .587 G^2 + .114 B^2), hue measured within
// the sextant of the largest channel.
__host__ __device__ inline void rgb2hsp(double R, double G, double B, double *H, double *S, double *P) {
    const double wr = 0.299, wg = 0.587, wb = 0.114;
    *P = sqrt(R * R * wr + G * G * wg + B * B * wb);
    if (R == G && R == B) {
        *H = 0.0;
        *S = 0.0;
        return;
    }
    // top: largest channel; after / before: the channels that follow / precede
    // it in R->G->B->R order; hue origins of the two half-sextants.
    double top, after, before, origin_down, origin_up;
    if (R >= G && R >= B) {
        top = R; after = G; before = B; origin_down = 6. / 6.; origin_up = 0. / 6.;
    } else if (G >= R && G >= B) {
        top = G; after = B; before = R; origin_down = 2. / 6.; origin_up = 2. / 6.;
    } else {
        top = B; after = R; before = G; origin_down = 4. / 6.; origin_up = 4. / 6.;
    }
    if (before >= after) {
        *H = origin_down - 1. / 6. * (before - after) / (top - after);
        *S = 1. - after / top;
    } else {
        *H = origin_up + 1. / 6. * (after - before) / (top - before);
        *S = 1. - before / top;
    }
}

__host__ __device__ inline void hsp2rgb(double H, double S, double P, double *R, double *G, double *B) {
    const double w[3] = {0.299, 0.587, 0.114};
    // per sextant: channel index of the largest, middle and smallest value
    int sext;
    if (H < 1. / 6.) sext = 0;
    else if (H < 2. / 6.) sext = 1;
    else if (H < 3. / 6.) sext = 2;
    else if (H < 4. / 6.) sext = 3;
    else if (H < 5. / 6.) sext = 4;
    else sext = 5;
    const int big = (sext == 0 || sext == 5) ? 0 : (sext == 1 || sext == 2) ? 1 : 2;
    const int mid = (sext == 0 || sext == 3) ? 1 : (sext == 1 || sext == 4) ? 0 : 2;
    const int low = 3 - big - mid;
    const double f = (sext & 1) ? 6. * (-H + double(sext + 1) / 6.) : 6. * (H - double(sext) / 6.);
    double c[3];
    const double ratio = 1. - S;  // smallest / largest
    if (ratio > 0.) {
        const double part = 1. + f * (1. / ratio - 1.);
        const double lo = P / sqrt(w[big] / ratio / ratio + w[mid] * part * part + w[low]);
        const double hi = lo / ratio;
        c[low] = lo;
        c[big] = hi;
        c[mid] = lo + f * (hi - lo);
    } else {
        const double hi = sqrt(P * P / (w[big] + w[mid] * f * f));
        c[big] = hi;
        c[mid] = hi * f;
        c[low] = 0.;
    }
    *R = c[0];
    *G = c[1];
    *B = c[2];
}

// color.cpp:31-44
__host__ __device__ inline uint32_t rgb_to_hsp(uint32_t c) {
    double h, s, p;
    rgb2hsp((c & 255u) / 255.0, ((c >> 8) & 255u) / 255.0, ((c >> 16) & 255u) / 255.0, &h, &s, &p);
    return rgba_pack(narrow8(round(h * 255.0)), narrow8(round(s * 255.0)), narrow8(round(p * 255.0)), c >> 24);
}
// color.cpp:46-59 (only the upper bound is clamped)
__host__ __device__ inline uint32_t hsp_to_rgb(uint32_t c) {
    double r, g, b;
    hsp2rgb((c & 255u) / 255.0, ((c >> 8) & 255u) / 255.0, ((c >> 16) & 255u) / 255.0, &r, &g, &b);
    return rgba_pack(narrow8(fmin(round(r * 255.0), 255.0)), narrow8(fmin(round(g * 255.0), 255.0)),
                     narrow8(fmin(round(b * 255.0), 255.0)), c >> 24);
}

// The same two in float, for a colour whose channels all land further than
// kClear from where the 8-bit rounding turns; false where one does not (about
// 1 colour in 30, mostly exact ties), and the double-precision form above
// decides.  Float has to be off by less than kClear = 2.4e-4.  Whole numbers up
// to 255 go in and no rounded terms are subtracted; a rounding is 2^-24 of its
// value, a reciprocal or root (v_rcp, v_rsq, v_sqrt) one ulp, 2^-23.  On the way
// to HSP that comes to 6e-5 at most (P's root).  On the way back the middle
// channel, through three of those and ten roundings, could reach 2.5e-4 if all
// were at their worst and added up; so a test compares the two with the
// double-precision form for every RGB colour and the HSP word it gives, which
// is all that ingest converts.
//
// Measured on one MI355X, 2048x2048 pixels, 36% opaque, both ways: 52 -> 26 us.
// In double precision the dozen divisions and two roots of a pixel bound it.
constexpr float kClear = 1.f / 4096;
__device__ __forceinline__ bool round_clear(float v, uint32_t *out) {
    const float r = rintf(v);
    *out = uint32_t(r);
    return fabsf(v - r) < 0.5f - kClear;
}
__device__ __forceinline__ bool rgb_to_hsp_clear(uint32_t c, uint32_t *hsp) {
    const float R = float(c & 255u), G = float((c >> 8) & 255u), B = float((c >> 16) & 255u);
    uint32_t h = 0, s = 0, p = 0;
    bool clear = round_clear(__builtin_amdgcn_sqrtf(R * R * 0.299f + G * G * 0.587f + B * B * 0.114f), &p);
    if (R != G || R != B) {
        const bool r = R >= G && R >= B, g = G >= R && G >= B;
        const float top = r ? R : g ? G : B, after = r ? G : g ? B : R, before = r ? B : g ? R : G;
        const bool down = before >= after;
        const float origin = r ? (down ? 255.f : 0.f) : g ? 85.f : 170.f;
        const float low = down ? after : before, part = 42.5f * (after - before);
        clear &= round_clear(origin + part * __builtin_amdgcn_rcpf(top - low), &h);
        clear &= round_clear(255.f * (top - low) * __builtin_amdgcn_rcpf(top), &s);
    }
    *hsp = rgba_pack(h, s, p, c >> 24);
    return clear;
}
__device__ __forceinline__ bool hsp_to_rgb_clear(uint32_t c, uint32_t *rgb) {
    const uint32_t h6 = 6 * (c & 255u), sext = min(h6 / 255u, 5u);
    const float f = float((sext & 1) ? 255 * (sext + 1) - h6 : h6 - 255 * sext) * (1.f / 255);
    const float S = float((c >> 8) & 255u), P = float((c >> 16) & 255u);
    const float wbig = (sext == 0 || sext == 5) ? 0.299f : sext < 3 ? 0.587f : 0.114f;
    const float wmid = (sext == 0 || sext == 3) ? 0.587f : (sext == 1 || sext == 4) ? 0.299f : 0.114f;
    const float wlow = 1.f - wbig - wmid;  // (exact to a rounding)
    float lo = 0.f, mid, hi;
    if (S < 255.f) {
        const float grow = 255.f * __builtin_amdgcn_rcpf(255.f - S);  // largest / smallest
        const float part = 1.f + f * S * __builtin_amdgcn_rcpf(255.f - S);
        lo = P * __builtin_amdgcn_rsqf(wbig * grow * grow + wmid * part * part + wlow);
        hi = lo * grow;
        mid = lo * part;
    } else {
        hi = P * __builtin_amdgcn_rsqf(wbig + wmid * f * f);
        mid = hi * f;
    }
    uint32_t a, b, d;
    bool clear = round_clear(fminf(hi, 255.f), &a);
    clear &= round_clear(fminf(mid, 255.f), &b);
    clear &= round_clear(fminf(lo, 255.f), &d);
    const bool r_big = sext == 0 || sext == 5, r_mid = sext == 1 || sext == 4;
    const bool g_big = sext == 1 || sext == 2, g_mid = sext == 0 || sext == 3;
    const bool b_big = sext == 3 || sext == 4;
    *rgb = rgba_pack(r_big ? a : r_mid ? b : d, g_big ? a : g_mid ? b : d, b_big ? a : (sext == 2 || sext == 5) ? b : d,
                     c >> 24);
    return clear;
}

}  // namespace amh
