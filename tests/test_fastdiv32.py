"""The division of all 32-bit numbers that the raw selection uses
(voxvision_amd/csrc/fastdiv.h, FastDiv32), compiled for the host with g++ and
checked against the / operator: every divisor up to 3000, the powers of two
and their neighbours, the largest divisors and random ones, each at the
multiples around it, both ends of the range and random numerators."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CHECK = r"""
#define __host__
#define __device__
#include "fastdiv.h"
#include <stdio.h>

static uint64_t rng = 88172645463325252ull;
static uint32_t next(void) {
    rng ^= rng << 13; rng ^= rng >> 7; rng ^= rng << 17;
    return (uint32_t)(rng >> 11);
}
static long bad;
static void one(const FastDiv32 &f, uint32_t n) {
    if (f.div(n) == n / f.d) return;
    if (!bad++) printf("d %u n %u got %u\n", f.d, n, f.div(n));
}
static void check(uint32_t d) {
    const FastDiv32 f = make_fastdiv32(d);
    const uint32_t top = 0xffffffffu, last = top / d * d;
    for (uint32_t k = 0; k < 3; k++) {
        one(f, k);
        one(f, top - k);
        one(f, d - 1 + k);
        one(f, last - 1 + k);
    }
    for (int i = 0; i < 64; i++) {
        one(f, next());
        one(f, (uint32_t)(next() % ((uint64_t)top / d + 1)) * d + next() % 3 - 1);
    }
}
int main(void) {
    for (uint32_t d = 1; d <= 3000; d++) check(d);
    for (int l = 1; l < 32; l++)
        for (int k = -1; k < 2; k++) check((1u << l) + k);
    for (uint32_t k = 0; k < 100; k++) check(0xffffffffu - k);
    for (int i = 0; i < 100000; i++) {
        const uint32_t d = next() >> (next() % 32);
        check(d ? d : 1);
    }
    printf("bad %ld\n", bad);
    return bad != 0;
}
"""


def test_every_dividend(tmp_path):
    src, exe = tmp_path / "check.cpp", tmp_path / "check"
    src.write_text(CHECK)
    r = subprocess.run(["g++", "-O2", "-I",
                        os.path.join(ROOT, "voxvision_amd", "csrc"), str(src),
                        "-o", str(exe)], capture_output=True, text=True)
    if r.returncode:
        pytest.fail(r.stderr)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
