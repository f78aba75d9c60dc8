// Division of 31-bit unsigned integers by a divisor fixed per launch, as
// one 32x32->64 multiply and a shift (Granlund and Montgomery, "Division
// by invariant integers using multiplication", PLDI 1994, theorem 4.2 with
// N = 31): for 1 <= d < 2^31, l = ceil(log2 d) and m = ceil(2^(31+l) / d),
// floor(n / d) = floor(n * m / 2^(31+l)) for every 0 <= n < 2^31, and m
// fits in 32 bits.  The GPU has no integer divide instruction; this
// replaces the tens of instructions of a generic 32-bit division.
#pragma once
#include <stdint.h>

struct FastDiv {
    uint32_t d;  // the divisor
    uint32_t m;  // ceil(2^s / d)
    uint32_t s;  // 31 + ceil(log2 d)

    // n / d for n < 2^31
    __host__ __device__ inline uint32_t div(uint32_t n) const {
        return (uint32_t)(((uint64_t)n * m) >> s);
    }
};

// d in [1, 2^31)
static inline FastDiv make_fastdiv(uint32_t d) {
    uint32_t l = 0;
    while ((1ull << l) < d) ++l;
    FastDiv f;
    f.d = d;
    f.s = 31u + l;
    f.m = (uint32_t)(((1ull << f.s) + d - 1ull) / d);
    return f;
}

// The same for every 32-bit dividend (figure 4.1 of that paper): one more
// subtraction and shift, since the multiplier takes 33 bits.  For sample
// numbers, of which a volume may hold up to 2^32 - 1.
struct FastDiv32 {
    uint32_t d;       // the divisor
    uint32_t m;       // the multiplier less 2^32
    uint32_t s1, s2;  // shifts

    __host__ __device__ inline uint32_t div(uint32_t n) const {
        const uint32_t t = (uint32_t)(((uint64_t)n * m) >> 32);
        return (t + ((n - t) >> s1)) >> s2;
    }
};

// d in [1, 2^32)
static inline FastDiv32 make_fastdiv32(uint32_t d) {
    uint32_t l = 0;
    while (l < 32 && (1ull << l) < d) ++l;
    FastDiv32 f;
    f.d = d;
    f.m = (uint32_t)((((1ull << l) - d) << 32) / d + 1);
    f.s1 = l < 1 ? l : 1;
    f.s2 = l > 1 ? l - 1 : 0;
    return f;
}
