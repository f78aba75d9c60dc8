// Distance bounds on a grid over a tree's box, for ball queries.
//
// Every cell of the grid holds two bounds for all points in it: L2, at most
// the squared distance to the nearest voxel, and U2, at least that distance
// squared.  A ball query whose centre lies in the cell is then answered by
// two comparisons unless rr = r * r lies between them: rr < L2, no voxel
// comes closer than r; rr > U2, one does.  The answers are those of the
// search (box_ball, geom-sse.c:144-149, on the voxels' boxes), bit for bit:
//
// The search's squared distance to a voxel's box is (dx^2 + dy^2) + dz^2
// with d = RN(f - c) for a clamped coordinate f: at most 2^-21 relative off
// the exact one.  A cell's bounds come from the same computation for the
// cell's centre: D2 for some voxel, and low2 such that no voxel is nearer;
// their roots are within 2^-20 relative of exact distances.  A point that grid_cell puts in a
// cell lies within half = sqrt(3) (1/2 + 2^-12) h + 2^-20 S of the computed
// centre, h the cell's edge and S the largest coordinate of the box: the
// index is floor(RN(RN(c - x0) * inv)), at most 2^-15 cells off for 128
// cells an axis, and the centre at most 4 ulp(S).  By the triangle
// inequality the exact distance to the nearest voxel is in
// [sqrt(low2) - half, sqrt(D2) + half]; L2 and U2 are the squares moved
// outward by 2^-17
// relative, rounded outward to the 16 bits that are kept.  Squares neither
// underflow nor overflow for boxes within 2^60 and cells of 2^-30 and more;
// other trees get no grid.
//
// The search also asks that the ball touches every box above the voxel.  In a
// tree whose boxes hold what is below them it does then (the clamp, and with
// it each computed distance, is monotone in the box); the grid of another
// tree decides nothing.
#pragma once
#include <math.h>
#include <stddef.h>
#include <stdint.h>
#include <string.h>

namespace ballgrid {

struct Grid {
    // L2 in the low half, U2 in the high half, as the upper halves of their
    // float bits; null: no grid
    const uint32_t *cells;
    float x0[3], x1[3];  // the tree's box
    float h, inv;        // edge of a cell and its reciprocal
    float half;          // see above
    uint32_t n[3];
};

constexpr uint32_t kMaxAxis = 128;  // cells along the longest axis

// The grid of a plain tree of `nodes` records over the box [lo, hi]; false
// when there is to be none.  At most kMaxAxis cells an axis, cubes no
// smaller than the smallest voxel edge, at most 8 cells a node.
inline bool grid_shape(const float lo[3], const float hi[3],
                       const float voxel[3], size_t nodes, Grid &g) {
    if (nodes < 2) return false;
    float E = 0.0f, S = 0.0f;
    for (int i = 0; i < 3; ++i) {
        if (!(fabsf(lo[i]) <= 0x1p60f) || !(fabsf(hi[i]) <= 0x1p60f) ||
            !(lo[i] <= hi[i]))
            return false;
        E = fmaxf(E, hi[i] - lo[i]);
        S = fmaxf(S, fmaxf(fabsf(lo[i]), fabsf(hi[i])));
    }
    float h = fmaxf(E / (float)kMaxAxis, fminf(voxel[0], fminf(voxel[1], voxel[2])));
    if (!(h >= 0x1p-30f) || !(h <= 0x1p60f)) return false;
    for (;; h *= 1.05f) {
        size_t cells = 1;
        g.h = h;
        g.inv = 1.0f / h;
        for (int i = 0; i < 3; ++i) {
            const float k = ceilf((hi[i] - lo[i]) * g.inv);
            g.n[i] = k < 1.0f ? 1u : k > (float)kMaxAxis ? kMaxAxis : (uint32_t)k;
            cells *= g.n[i];
        }
        if (cells <= 8 * nodes) break;
    }
    for (int i = 0; i < 3; ++i) {
        g.x0[i] = lo[i];
        g.x1[i] = hi[i];
    }
    g.half = 1.7320509f * (0.5f + 0x1p-12f) * h + 0x1p-20f * S;
    g.cells = nullptr;
    return true;
}

inline size_t grid_cells(const Grid &g) {
    return (size_t)g.n[0] * g.n[1] * g.n[2];
}

__host__ __device__ inline uint32_t float_bits(float x) {
    uint32_t u;
    memcpy(&u, &x, sizeof(u));
    return u;
}
__host__ __device__ inline float bits_float(uint32_t u) {
    float x;
    memcpy(&x, &u, sizeof(x));
    return x;
}

__host__ __device__ inline float grid_centre(const Grid &g, int axis, uint32_t i) {
    return g.x0[axis] + ((float)i + 0.5f) * g.h;
}

// How near (squared) a search for the voxel nearest to a cell's centre has
// to look when it has one at the squared distance D2: all of it within four
// cells, and a fifth of the rest less.  Far from the voxels the exact
// distance decides few queries, and its search looks at most of the tree
// (the 256^3 CT scene's grid: 2.0 ms without this, 1.3 with it, 0.58 with
// grid_kernel's start from the middle of its cells as well).
__host__ __device__ inline float grid_low(const Grid &g, float D2) {
    const float D = sqrtf(D2);
    const float low = D > 4.0f * g.h ? D - 0.2f * (D - 4.0f * g.h) : D;
    return D2 < INFINITY ? low * low : D2;
}

// A cell from the squared distance D2 of its centre to some voxel and a
// squared distance low2 <= D2 within which no voxel is.
__host__ __device__ inline uint32_t grid_pack(const Grid &g, float low2, float D2) {
    const float L = sqrtf(fminf(low2, D2)) * (1.0f - 0x1p-18f) - g.half;
    const float U = sqrtf(D2) * (1.0f + 0x1p-18f) + g.half;
    const float L2 = L > 0x1p-40f ? L * L * (1.0f - 0x1p-17f) : 0.0f;
    const float U2 = U * U * (1.0f + 0x1p-17f);
    return (float_bits(L2) >> 16) | ((float_bits(U2) + 0xffffu) & 0xffff0000u);
}

// The cell of a point, or false for a point that is not in the box (or not
// a number).
__host__ __device__ inline bool grid_cell(const Grid &g, float x, float y,
                                          float z, size_t &cell) {
    const bool in = (x >= g.x0[0]) & (x <= g.x1[0]) & (y >= g.x0[1]) &
                    (y <= g.x1[1]) & (z >= g.x0[2]) & (z <= g.x1[2]);
    if (!in) return false;
    auto at = [](float v, uint32_t n) {
        const uint32_t i = (uint32_t)v;  // v >= 0
        return i < n ? i : n - 1u;
    };
    const uint32_t ix = at((x - g.x0[0]) * g.inv, g.n[0]);
    const uint32_t iy = at((y - g.x0[1]) * g.inv, g.n[1]);
    const uint32_t iz = at((z - g.x0[2]) * g.inv, g.n[2]);
    cell = ((size_t)ix * g.n[1] + iy) * g.n[2] + iz;
    return true;
}

enum Verdict { kMiss = 0, kHit = 1, kUndecided = 2 };

// A cell that decides nothing: L2 zero, U2 infinite.
constexpr uint32_t kNoBounds = 0x7f800000u;

__host__ __device__ inline Verdict grid_verdict(uint32_t cell, float rr) {
    if (rr < bits_float(cell << 16)) return kMiss;
    if (rr > bits_float(cell & 0xffff0000u)) return kHit;
    return kUndecided;
}

}  // namespace ballgrid
