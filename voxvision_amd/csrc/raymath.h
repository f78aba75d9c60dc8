// The traversal's box and plane tests without IEEE divisions.
//
// The exact tests (hit_box, hit_plane in voxgpu.hip; geom-sse.c:84-142)
// divide by a direction component: three divisions per box test, up to
// three per inner node and one per pending child taken from the stack.  On
// gfx950 a correctly rounded division is 45 cycles of a SIMD per wave
// (measured; an fma is 2.3, a min, max or compare 4), and the traversal
// kernels are bound by VALU issue.  The functions here give the same bits
// for less: a ray's reciprocals y = RN(1 / d) are taken once, and a / d is
//
//   q0 = RN(a y),   r = RN(a - q0 d),   q = RN(q0 + r y)
//
// which is the correctly rounded quotient.  Let D < 2^24 be d's significand
// as an integer, and count in ulps of a / d.  |a / d - q0| <= 1.5, so the
// remainder a - q0 d is an integer of at most 25 bits in units of
// ulp(q0) ulp(d): r is off by one unit at most (1 / D in the quotient).  y
// is off by 2^-24 relative, 1.5 / D in r y.  So the value that the last
// line rounds is within 2.5 / D (and a relative 2^-23 of that) of a / d.  A
// quotient lies R / (2 D) away from the nearest midpoint of two floats for
// an integer R >= 1, so only quotients with R <= 5 could be rounded the
// other way; tests/test_raymath.py runs all of those (every D, every R up
// to 6) and finds none.  The remainder's last bit is 2^-47 |a| at least, so
// nothing underflows or overflows for
//
//   2^-60 <= |d| <= 2^30  and  2^-89 <= |a| <= 2^62
//
// (then 2^-119 <= |a / d| <= 2^122).  d = 0 gets y = 0, which makes every
// quotient a zero, as the box test takes it; a = 0 gives a zero.
//
// A ray is `plain` when its direction is in that range (or zero, but not in
// all components), and its origin is at most 2^60 in magnitude; a tree is
// plain when its boxes, centres and voxels are finite, at most 2^60 in
// magnitude and not inverted.  Then every point the traversal computes
// from it is finite: a box's entry point lies in the box, and a plane
// point is kept only inside the node's box.  For other rays and trees, and
// where a distance a is nonzero but below 2^-89, the caller takes the exact
// tests (kUndecided).
#pragma once
#include <math.h>
#include <stdint.h>
#include <string.h>

// The tests are written with & and | on conditions, not && and ||: every
// lane evaluates everything (a branch costs the wave more than the rest of
// the test).
namespace raymath {

__host__ __device__ inline float fused(float a, float b, float c) {
    return __builtin_fmaf(a, b, c);
}
__host__ __device__ inline float max3(float a, float b, float c) {
    return fmaxf(fmaxf(a, b), c);
}
// the middle one of x, lo, hi for lo <= hi: x clamped to [lo, hi]
__host__ __device__ inline float clamp(float x, float lo, float hi) {
#ifdef __HIP_DEVICE_COMPILE__
    return __builtin_amdgcn_fmed3f(x, lo, hi);
#else
    return fminf(fmaxf(x, lo), hi);
#endif
}
__host__ __device__ inline uint32_t bits(float x) {
    uint32_t u;
    memcpy(&u, &x, sizeof(u));
    return u;
}
// an order of |a| in which zero comes last: all ones for +-0, else
// 2 bits(|a|) - 1
__host__ __device__ inline uint32_t size_key(float a) {
    return (bits(a) << 1) - 1u;
}
constexpr uint32_t kZeroKey = 0xffffffffu;
// keys below this: 0 < |a| < 2^-89
constexpr uint32_t kTinyKey = ((127u - 89u) << 24) - 1u;

__host__ __device__ inline uint32_t min3(uint32_t a, uint32_t b, uint32_t c) {
    const uint32_t m = a < b ? a : b;
    return m < c ? m : c;
}

__host__ __device__ inline bool plain_axis(float o, float d) {
    const float m = fabsf(d);
    return (fabsf(o) <= 0x1p60f) & ((m == 0.0f) | ((m >= 0x1p-60f) & (m <= 0x1p30f)));
}

// y of the scheme above (an IEEE division, once per ray and axis)
__host__ __device__ inline float reciprocal(float d) {
    return d == 0.0f ? 0.0f : 1.0f / d;
}

// a / d, correctly rounded (see the ranges above)
__host__ __device__ inline float quotient(float a, float d, float y) {
    const float q0 = a * y;
    return fused(fused(-q0, d, a), y, q0);
}

enum Verdict { kMiss = 0, kHit = 1, kUndecided = 2 };

// hit_box for a plain ray and box: the clamped origin is the middle one of
// three (v_med3), the three maxima of the shuffle network are one value,
// and an origin inside the box shows in the smallest of the distances'
// keys, which also tells the tiny ones.
__host__ __device__ inline Verdict box_entry(
    const float (&lo)[3], const float (&hi)[3], const float (&o)[3],
    const float (&d)[3], const float (&y)[3], float (&e)[3]) {
    float f[3], s[3], t[3];
    for (int i = 0; i < 3; ++i) {
        f[i] = clamp(o[i], lo[i], hi[i]);
        s[i] = f[i] - o[i];
        t[i] = quotient(s[i], d[i], y[i]);
    }
    const uint32_t key = min3(size_key(s[0]), size_key(s[1]), size_key(s[2]));
    const float m = max3(t[0], t[1], t[2]);
    const bool inside = key == kZeroKey;
    bool in = true;
    for (int i = 0; i < 3; ++i) {
        const float h = m == t[i] ? f[i] : fused(m, d[i], o[i]);
        e[i] = inside ? o[i] : h;
        in = in & (h >= lo[i]) & (h <= hi[i]);
    }
    if (key < kTinyKey) return kUndecided;
    return inside | ((m > 0.0f) & in) ? kHit : kMiss;
}

// hit_plane for the plane through c normal to axis i, a plain ray from o
// and the box [lo, hi]; a is set to the plane's distance c - o[i] (a size
// key below kTinyKey: the answer is not to be used).  A direction parallel
// to the plane misses it: the exact test's point is then infinite or not a
// number in some component that the box test rejects.
__host__ __device__ inline bool plane_point(
    const float (&lo)[3], const float (&hi)[3], const float (&o)[3],
    const float (&d)[3], const float (&y)[3], float c, int i, float &a,
    float (&p)[3]) {
    a = c - o[i];
    const float k = quotient(a, d[i], y[i]);
    bool in = k > 0.0f;
    for (int j = 0; j < 3; ++j) {
        p[j] = fused(k, d[j], o[j]);
        in = in & (p[j] >= lo[j]) & (p[j] <= hi[j]);
    }
    return in;
}

}  // namespace raymath
