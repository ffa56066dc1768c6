// device_dense.h - bodies of the dense path's kernels that evaluate the SDF at given points,
// templated on it.  The tape interpreter's kernels (kernels.hip) and the kernels of programs
// compiled at run time by hiprtc instantiate the same bodies, so both paths run identical
// per-point code around their SDF.  What else the dense path does (device_bricks.h) is
// compiled once, in the library: in every program's module it took half of the 130 ms that
// compiling one takes otherwise.
//
// A slab's corner lattice is handled in bricks of 4 x 4 x 4 points.  sign_words evaluates
// every point and keeps `value > 0`, one 64-bit word per brick; bricks whose cells change
// sign are listed (k_find_bricks), and contour_bricks needs the values at just the corners
// of those cells.  sign_words keeps the values it takes (4 bytes a point beside a whole
// program each), brick by brick, so that a brick's lie in few lines; where the sign is
// decided without the value (the Mandelbulb's early signs) they are evaluated then.
#pragma once
#ifndef __HIPCC_RTC__
#include <hip/hip_runtime.h>
#include <stdint.h>
#endif

#include "dense_args.h"

namespace s2m {

// One lattice point per thread: 256-thread blocks of 16 x 4 x 4 points, each wave a
// 4 x 4 x 4 block (lanes close together, so data-dependent loops diverge less than along
// a row), grid (ceil(nx / 16), ceil(ny / 4), ceil(planes / 4)).
template <class F>
__device__ __forceinline__ void eval_lattice_point(F sdf, const float* __restrict__ cx,
                                                   const float* __restrict__ cy,
                                                   const float* __restrict__ cz, uint32_t nx,
                                                   uint32_t ny, uint32_t lz0, uint32_t nzl, uint32_t pitch,
                                                   float* __restrict__ lat)
{
    const uint32_t l = threadIdx.x & 63u, w = threadIdx.x >> 6;
    const uint32_t ix = blockIdx.x * 16u + w * 4u + (l & 3u);
    const uint32_t iy = blockIdx.y * 4u + ((l >> 2) & 3u);
    const uint32_t iz = blockIdx.z * 4u + (l >> 4);
    if (ix >= nx || iy >= ny || iz >= nzl) return;
    lat[((size_t)iz * ny + iy) * pitch + ix] = sdf(cx[ix], cy[iy], cz[lz0 + iz]);
}

// A NaN result is stored as the canonical quiet NaN (0x7fc00000): which NaN operand an
// instruction propagates, and so the sign and payload of a NaN result, differ between
// kernels that compute the same value (the dense and the tile-sparse path), so vertex
// positions and normals that are NaN are written with one bit pattern on every path.
__device__ __forceinline__ float canonical_nan(float v) { return v != v ? __builtin_nanf("") : v; }

// normalize(g) written to o[3..5] (dualcontour.wgsl:171): g / length(g).
__device__ __forceinline__ void write_unit(float* o, float gx, float gy, float gz)
{
    const float len = sqrtf((gx * gx + gy * gy) + gz * gz);
    o[3] = canonical_nan(gx / len);
    o[4] = canonical_nan(gy / len);
    o[5] = canonical_nan(gz / len);
}

__device__ __forceinline__ uint32_t clamp_to(uint32_t i, uint32_t n) { return i < n ? i : n - 1u; }

// Where the values of brick (bx, by, bz), counted from (bx0, by0), start: 16 per lattice plane of
// the slab in it, bricks of one layer after each other.
__device__ __forceinline__ size_t brick_vals(const BrickArgs& a, uint32_t bx, uint32_t by, uint32_t bz)
{
    const uint32_t planes = a.nzl - 4u * bz < 4u ? a.nzl - 4u * bz : 4u;
    return 16u * ((size_t)bz * 4u * a.nby * a.nbx + ((size_t)by * a.nbx + bx) * planes);
}

// Sign of an SDF at a point as that of its value, without a test on whole bricks.
template <class F>
struct PointSign {
    F sdf;
    static constexpr bool kBricks = false;   // brick() decides whole bricks
    static constexpr bool kValue = true;     // operator() returns the value itself, which is kept
    __device__ float operator()(float x, float y, float z) const { return sdf(x, y, z); }
    __device__ int brick(float, float, float, float, float, float) const { return -1; }
};

// One wave per run of a.run bricks along x (blocks of 4 waves: 4 brick rows), grid
// (ceil(nbx / run), ceil(nby / 4), nbz).  A wave takes one brick at a time, one point per
// lane (lanes close together run data-dependent loops alike), so the run's coordinates
// are loaded once and its words leave in one store.  S::brick decides a whole brick from
// its box (0 / 1: every point <= 0 / > 0; -1: undecided); lane b tests brick b.  Points past
// the lattice's end repeat its last point (no cell uses them).
template <class S>
__device__ __forceinline__ void sign_words(const S& sign, const BrickArgs& a)
{
    const uint32_t l = threadIdx.x & 63u, w = threadIdx.x >> 6;
    const uint32_t b0 = blockIdx.x * a.run, by = blockIdx.y * 4u + w, bz = blockIdx.z;
    if (by >= a.nby) return;
    const float xr = a.cx[clamp_to((a.bx0 + b0) * 4u + l, a.nx)];
    const float y = a.cy[clamp_to((a.by0 + by) * 4u + ((l >> 2) & 3u), a.ny)];
    const float z = a.cz[a.lz0 + clamp_to(bz * 4u + (l >> 4), a.nzl)];
    const uint32_t nb = min(a.run, a.nbx - b0);
    const size_t row = ((size_t)bz * a.nby + by) * a.nbx + b0;
    const uint32_t planes16 = 16u * min(a.nzl - 4u * bz, 4u);  // values of a brick
    float* const vals = S::kValue ? a.vals + brick_vals(a, b0, by, bz) : nullptr;
    uint64_t word = 0;  // lane b: brick b's
    uint32_t todo = (1u << nb) - 1u;
    if constexpr (S::kBricks) {
        // the tables ascend or descend but for neighbours a rounding apart: min and max of all four
        const int xb = (int)(l & 15u) * 4;
        const float x0 = __shfl(xr, xb, 64), x1 = __shfl(xr, xb + 1, 64), x2 = __shfl(xr, xb + 2, 64),
                    x3 = __shfl(xr, xb + 3, 64);
        const float y0 = __shfl(y, 0, 64), y1 = __shfl(y, 4, 64), y2 = __shfl(y, 8, 64), y3 = __shfl(y, 12, 64);
        const float z0 = __shfl(z, 0, 64), z1 = __shfl(z, 16, 64), z2 = __shfl(z, 32, 64), z3 = __shfl(z, 48, 64);
        const int d = sign.brick(fminf(fminf(x0, x1), fminf(x2, x3)), fmaxf(fmaxf(x0, x1), fmaxf(x2, x3)),
                                 fminf(fminf(y0, y1), fminf(y2, y3)), fmaxf(fmaxf(y0, y1), fmaxf(y2, y3)),
                                 fminf(fminf(z0, z1), fminf(z2, z3)), fmaxf(fmaxf(z0, z1), fmaxf(z2, z3)));
        word = d > 0 ? ~0ull : 0ull;
        todo &= (uint32_t)__ballot(d < 0);
    }
    while (todo) {
        const uint32_t b = (uint32_t)__builtin_ctz(todo);
        todo &= todo - 1u;
        const float x = __shfl(xr, (int)(b * 4u + (l & 3u)), 64);
        const float v = sign(x, y, z);
        const uint64_t m = __ballot(v > 0.0f);
        if (l == b) word = m;
        if constexpr (S::kValue) {
            if (l < planes16) vals[b * planes16 + l] = v;
        }
    }
    if (l < nb) a.words[row + l] = word;
}

// Lane `k` of each group of four lanes, broadcast to the group.
template <int K>
__device__ __forceinline__ float quad_lane(float v)
{
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), K * 0x55, 0xf, 0xf, true));
}

// sdf3d_normal (sdf3d_normal.wgsl:4-9) of the vertex at p, by the four lanes of a group, one per
// tap (v1=(1,-1,-1), v2=(-1,-1,1), v3=(-1,1,-1), v4=(1,1,1) at p + v * eps, summed left to
// right, normalized), so the SDF is inlined once: o[3..5].
template <class F>
__device__ __forceinline__ void tap_normal(const F& sdf, float px, float py, float pz, float eps, uint32_t tap, float* o)
{
    const float ex = (tap == 0u || tap == 3u) ? eps : -eps;
    const float ey = tap >= 2u ? eps : -eps;
    const float ez = (tap == 1u || tap == 3u) ? eps : -eps;
    const float d = sdf(px + ex, py + ey, pz + ez);
    const float d1 = quad_lane<0>(d), d2 = quad_lane<1>(d), d3 = quad_lane<2>(d), d4 = quad_lane<3>(d);
    write_unit(o, ((d1 + (-d2)) + (-d3)) + d4, (((-d1) + (-d2)) + d3) + d4, (((-d1) + d2) + (-d3)) + d4);
}

// Normals of the vertices the slab has written, [counters[kDenseVtxPrev],
// counters[kDenseVtxTotal]) below vcap, their positions in place.  LIB: the library's
// normal of the SDF F, else F(px, py, pz, eps, o) writes o[3..5].
constexpr uint32_t kDenseVtxTotal = 0, kDenseVtxPrev = 1;  // Counter (internal.h)
template <bool LIB, class F>
__device__ __forceinline__ void vertex_normals(const F& f, float eps, float* vtx, const uint64_t* counters, uint64_t vcap)
{
    constexpr uint32_t kLanes = LIB ? 4u : 1u;
    const uint64_t beg = counters[kDenseVtxPrev], end = min(counters[kDenseVtxTotal], vcap);
    const uint32_t tap = LIB ? threadIdx.x & 3u : 0u;
    for (uint64_t v = beg + ((uint64_t)blockIdx.x * 256u + threadIdx.x) / kLanes; v < end; v += gridDim.x * (256u / kLanes)) {
        float* o = vtx + 6 * v;
        if constexpr (LIB) {
            float n[6];
            tap_normal(f, o[0], o[1], o[2], eps, tap, n);
            if (tap < 3u) o[3u + tap] = tap == 0u ? n[3] : tap == 1u ? n[4] : n[5];
        } else {
            f(o[0], o[1], o[2], eps, o);
        }
    }
}

}  // namespace s2m
