// One term of the softened pair sums, shared by the batched sums (soft.hip) and the
// centring iteration (centre.hip).
#pragma once
#include "halma_common.h"

namespace halma {

constexpr int kSub = 8;  // terms of a plain FP32 sub-tile

// pair quantities: bit 0 the potential S, bit 1 the gradient a and w
constexpr int kModePot = 1;
constexpr int kModeAcc = 2;
constexpr int kModeBoth = 3;
__host__ __device__ constexpr int n_planes(int mode) {
    return ((mode & kModePot) ? 1 : 0) + ((mode & kModeAcc) ? 4 : 0);
}

struct TestPt {
    float hx, hy, hz, lx, ly, lz;
};

__device__ __forceinline__ TestPt split_test(double x, double y, double z) {
    TestPt t;
    t.hx = static_cast<float>(x);
    t.hy = static_cast<float>(y);
    t.hz = static_cast<float>(z);
    t.lx = static_cast<float>(x - static_cast<double>(t.hx));
    t.ly = static_cast<float>(y - static_cast<double>(t.hy));
    t.lz = static_cast<float>(z - static_cast<double>(t.hz));
    return t;
}

// Kahan-compensated addition: c holds the low part lost so far (s + c is the sum; the
// sequence of s is that of the textbook form, whose compensation is -c)
__device__ __forceinline__ void kahan(float& s, float& c, float v) {
    const float y = v + c;
    const float t = s + y;
    c = y - (t - s);
    s = t;
}

// Error bounds of the softened sums, u = 2^-24 (tests FP64 points; the members as tests lack
// the lo part's share).  A difference is off by 2u (the lo part's rounding or the first
// subtraction's, and the second's), r^2 + eps^2 by 7u, its root by 3.5u, v_rsq_f32 by 1 ulp =
// 2u: 5.5u for 1 / r.  S: 5.5u, at most 8 roundings of a term in its sub-tile (the product's
// included), the Kahan sum 2u, 0.5u for the FP64 sums and the higher orders: 16u = 2^-20.
// a: three times 5.5u, the products of the cube and the mass 3u, the difference 2u, the
// sub-tile 8u, Kahan 2u and 0.5u: 32u = 2^-19 of the sum of |terms|; w less.  The symmetric
// form (soft_sym.hip) has neither the lo part nor Kahan sums: 13u and 26u.

// One pair term added into the plain sub-tile sums ps (planes as n_planes(MODE): the
// potential first when present, then ax, ay, az, w).  FP64 tests (SELF false) subtract
// their lo part after the hi part.
template <int MODE, bool SELF>
__device__ __forceinline__ void pair_term(float* ps, float4 p, const TestPt& t, float e2) {
    const float dx = SELF ? p.x - t.hx : (p.x - t.hx) - t.lx;
    const float dy = SELF ? p.y - t.hy : (p.y - t.hy) - t.ly;
    const float dz = SELF ? p.z - t.hz : (p.z - t.hz) - t.lz;
    const float mn = fminf(fminf(fabsf(dx), fabsf(dy)), fabsf(dz));
    const float d2 = __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, __builtin_fmaf(dx, dx, e2)));
    const float inv = mn != 0.0f ? __builtin_amdgcn_rsqf(d2) : 0.0f;
    constexpr int A = (MODE & kModePot) ? 1 : 0;
    if (MODE & kModePot) ps[0] = __builtin_fmaf(p.w, inv, ps[0]);
    if (MODE & kModeAcc) {
        const float w = p.w * (inv * (inv * inv));
        ps[A + 0] = __builtin_fmaf(w, dx, ps[A + 0]);
        ps[A + 1] = __builtin_fmaf(w, dy, ps[A + 1]);
        ps[A + 2] = __builtin_fmaf(w, dz, ps[A + 2]);
        ps[A + 3] += w;
    }
}

}  // namespace halma
