// device_interval.h - interval bounds of the SDF tape over a box of points, and exact
// per-box tape pruning.
//
// For a box of lattice points B (and anything within `pad` of it), an interval bounds the
// fp32 value the tape interpreter computes at any point of B.  Bounds follow the
// real-valued function (every library primitive is a distance, every operator is monotone
// in each operand) and are widened by kMargin x the magnitudes involved, 64 ulps, which
// covers the rounding of the few fp32 operations of each op and of the few fp32
// operations of its bound: each is within about 8 ulps of those magnitudes (differences
// of coordinates and centres are exact to half an ulp of the difference on both sides;
// square roots and reciprocals of bounds are the hardware's, 1 ulp).  kFloor covers
// squares that underflow.  tests/test_interval.py checks bounds and dropped operands against
// the evaluation with those roots and reciprocals moved by an ulp at random: over 120 M
// values none is out of bounds down to a margin of 8 ulps, the first at 4.  (In fp64 the bounds took twice the registers and LDS and a
// dozen instructions per square root or division; the walks are serial chains of them.)
//
// Pruning keeps the postfix tape's value identical, not approximately equal: an operator
// is replaced by one operand only when the interval bounds force the fp32 result to be
// exactly that operand on the whole box:
//   min(d1,d2), max(d1,d2): bounds of one operand entirely on one side of the other;
//   max(-d1,d2):            d2 >= -d1 everywhere  -> d2;
//   smooth union:  d2 >= d1 + k  -> h = 1, mix(d2,d1,1) - k*1*0 = d1;
//                  d2 <= d1 - k  -> h = 0, result d2;
//   smooth intersection: the mirror image; smooth subtraction: d1 + d2 >= k -> d2.
// (The replaced result can differ from the operand only in the sign of a zero, which no
// comparison `> 0`, subtraction or division downstream can observe.)
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/sdf2mesh.h"

namespace s2m {

constexpr float kMargin = 64.0f / 16777216.0f;  // 64 fp32 ulps, relative
constexpr float kUlps = 4.0f / 16777216.0f;     // of a comparison's own additions
constexpr float kFloor = 2e-19f;                // > the root of the largest denormal
constexpr float kHuge = 1e30f;

struct Iv {
    float lo, hi;
    bool known;
};

__device__ __forceinline__ Iv iv_unknown() { return {-kHuge, kHuge, false}; }

__device__ __forceinline__ Iv iv_make(float lo, float hi, float mag)
{
    const float m = kMargin * fabsf(mag) + kFloor;
    Iv r{lo - m, hi + m, true};
    if (!(r.lo > -kHuge && r.hi < kHuge)) return iv_unknown();  // also catches NaN
    return r;
}

// range of |q| for q in the box [lo, hi] (per component)
__device__ __forceinline__ void abs_range(float lo, float hi, float& near, float& far)
{
    near = lo > 0 ? lo : (hi < 0 ? -hi : 0.0f);
    far = fmaxf(fabsf(lo), fabsf(hi));
}

// distance range from the origin to the points of an n-D box
__device__ __forceinline__ void norm_range(const float* lo, const float* hi, int n, float& dmin,
                                           float& dmax)
{
    float s0 = 0, s1 = 0;
    for (int a = 0; a < n; ++a) {
        float nr, fr;
        abs_range(lo[a], hi[a], nr, fr);
        s0 += nr * nr;
        s1 += fr * fr;
    }
    dmin = __builtin_amdgcn_sqrtf(s0);
    dmax = __builtin_amdgcn_sqrtf(s1);
}

// Real-valued smooth operators (sdf_op.wgsl:7-23).
__device__ __forceinline__ float r_clamp01(float x) { return fminf(fmaxf(x, 0.0f), 1.0f); }
__device__ __forceinline__ float r_su(float d1, float d2, float k)
{
    const float h = r_clamp01(0.5f + 0.5f * (d2 - d1) * __builtin_amdgcn_rcpf(k));
    return d2 * (1 - h) + d1 * h - k * h * (1 - h);
}
__device__ __forceinline__ float r_si(float d1, float d2, float k)
{
    const float h = r_clamp01(0.5f - 0.5f * (d2 - d1) * __builtin_amdgcn_rcpf(k));
    return d2 * (1 - h) + d1 * h + k * h * (1 - h);
}
__device__ __forceinline__ float r_ss(float d1, float d2, float k)
{
    const float h = r_clamp01(0.5f - 0.5f * (d2 + d1) * __builtin_amdgcn_rcpf(k));
    return d2 * (1 - h) - d1 * h + k * h * (1 - h);
}

// Bounds of one primitive over the box [bl, bh].
__device__ __forceinline__ Iv iv_primitive(uint32_t code, const float* f, const float* bl,
                                           const float* bh)
{
    float lo[3], hi[3];
    if (code == S2M_OP_CAPSULE || code == S2M_OP_MANDELBULB) {
        for (int a = 0; a < 3; ++a) {
            lo[a] = bl[a];
            hi[a] = bh[a];
        }
    } else {  // translated primitives: q = p - c
        for (int a = 0; a < 3; ++a) {
            lo[a] = bl[a] - f[a];
            hi[a] = bh[a] - f[a];
        }
    }
    switch (code) {
    case S2M_OP_SPHERE: {  // length(q) - s
        float dmin, dmax;
        norm_range(lo, hi, 3, dmin, dmax);
        const float s = f[3];
        return iv_make(dmin - s, dmax - s, dmax + fabsf(s));
    }
    case S2M_OP_BOX: {  // monotone in each q_a = |p_a - c_a| - b_a/2
        float ql[3], qh[3], mag = 0;
        for (int a = 0; a < 3; ++a) {
            float nr, fr;
            abs_range(lo[a], hi[a], nr, fr);
            const float hb = 0.5f * f[3 + a];
            ql[a] = nr - hb;
            qh[a] = fr - hb;
            mag += fr + fabsf(hb);
        }
        auto g = [](const float* q) {
            const float x = fmaxf(q[0], 0.0f), y = fmaxf(q[1], 0.0f), z = fmaxf(q[2], 0.0f);
            return __builtin_amdgcn_sqrtf(x * x + y * y + z * z) + fminf(fmaxf(q[0], fmaxf(q[1], q[2])), 0.0f);
        };
        return iv_make(g(ql), g(qh), mag);
    }
    case S2M_OP_TORUS: {  // length(vec2(length(q.xz) - R, q.y)) - r
        const float xl[2] = {lo[0], lo[2]}, xh[2] = {hi[0], hi[2]};
        float rmin, rmax;
        norm_range(xl, xh, 2, rmin, rmax);
        const float ql[2] = {rmin - f[3], lo[1]}, qh[2] = {rmax - f[3], hi[1]};
        float dmin, dmax;
        norm_range(ql, qh, 2, dmin, dmax);
        const float r = f[4];
        return iv_make(dmin - r, dmax - r, rmax + fabsf(f[3]) + fabsf(lo[1]) + fabsf(hi[1]) +
                                               fabsf(r));
    }
    case S2M_OP_CYLINDER: {  // monotone in dx = length(q.xz) - r, dy = |q.y| - h
        const float xl[2] = {lo[0], lo[2]}, xh[2] = {hi[0], hi[2]};
        float rmin, rmax, ny, fy;
        norm_range(xl, xh, 2, rmin, rmax);
        abs_range(lo[1], hi[1], ny, fy);
        const float h = f[3], r = f[4];
        auto g = [](float dx, float dy) {
            const float px = fmaxf(dx, 0.0f), py = fmaxf(dy, 0.0f);
            return fminf(fmaxf(dx, dy), 0.0f) + __builtin_amdgcn_sqrtf(px * px + py * py);
        };
        return iv_make(g(rmin - r, ny - h), g(rmax - r, fy - h), rmax + fy + fabsf(h) + fabsf(r));
    }
    case S2M_OP_CAPSULE: {  // distance to segment ab, minus r
        const float a[3] = {f[0], f[1], f[2]}, b[3] = {f[3], f[4], f[5]};
        float half = 0, at = 0, ml[3], mh[3], al[3], ah[3], bl2[3], bh2[3];
        for (int i = 0; i < 3; ++i) {
            const float m = 0.5f * (a[i] + b[i]);
            at += fabsf(a[i]) + fabsf(b[i]);  // the midpoint is rounded at the scale of a and b
            half += (b[i] - a[i]) * (b[i] - a[i]);
            ml[i] = lo[i] - m;
            mh[i] = hi[i] - m;
            al[i] = lo[i] - a[i];
            ah[i] = hi[i] - a[i];
            bl2[i] = lo[i] - b[i];
            bh2[i] = hi[i] - b[i];
        }
        half = 0.5f * __builtin_amdgcn_sqrtf(half);
        float mmin, mmax, amin, amax, bmin, bmax;
        norm_range(ml, mh, 3, mmin, mmax);
        norm_range(al, ah, 3, amin, amax);
        norm_range(bl2, bh2, 3, bmin, bmax);
        const float r = f[6];
        return iv_make(fmaxf(mmin - half, 0.0f) - r, fminf(amax, bmax) - r, mmax + 2 * half + fabsf(r) + at);
    }
    default: return iv_unknown();  // Mandelbulb: iterated, may produce NaN
    }
}

enum Keep : int { kKeepBoth = 0, kKeepA = 1, kKeepB = 2 };

// Interval of op(A, B) and whether one operand can replace it exactly on the box.
__device__ __forceinline__ Iv iv_op(uint32_t code, Iv A, Iv B, float kf, int& keep)
{
    keep = kKeepBoth;
    if (!A.known || !B.known) return iv_unknown();
    const float k = kf;
    const float tiny = kUlps * (fabsf(A.lo) + fabsf(A.hi) + fabsf(B.lo) + fabsf(B.hi) + fabsf(k));
    switch (code) {
    case S2M_OP_UNION:
        if (B.lo >= A.hi + tiny) { keep = kKeepA; return A; }
        if (B.hi + tiny <= A.lo) { keep = kKeepB; return B; }
        return {fminf(A.lo, B.lo), fminf(A.hi, B.hi), true};
    case S2M_OP_INTERSECTION:
        if (B.hi + tiny <= A.lo) { keep = kKeepA; return A; }
        if (A.hi + tiny <= B.lo) { keep = kKeepB; return B; }
        return {fmaxf(A.lo, B.lo), fmaxf(A.hi, B.hi), true};
    case S2M_OP_SUBTRACTION:  // max(-A, B)
        if (B.lo >= -A.lo + tiny) { keep = kKeepB; return B; }
        return {fmaxf(-A.hi, B.lo), fmaxf(-A.lo, B.hi), true};
    default: break;
    }
    if (!(k > 0)) return iv_unknown();  // degenerate smoothing radius: no pruning
    const float mag = fmaxf(fabsf(A.lo), fabsf(A.hi)) + fmaxf(fabsf(B.lo), fabsf(B.hi)) + k;
    switch (code) {
    case S2M_OP_SMOOTH_UNION:
        if (B.lo >= A.hi + k + tiny) { keep = kKeepA; return A; }
        if (B.hi + k + tiny <= A.lo) { keep = kKeepB; return B; }
        return iv_make(r_su(A.lo, B.lo, k), r_su(A.hi, B.hi, k), mag);
    case S2M_OP_SMOOTH_INTERSECTION:
        if (B.lo >= A.hi + k + tiny) { keep = kKeepB; return B; }
        if (B.hi + k + tiny <= A.lo) { keep = kKeepA; return A; }
        return iv_make(r_si(A.lo, B.lo, k), r_si(A.hi, B.hi, k), mag);
    default:  // smooth subtraction: decreasing in A, increasing in B
        if (A.lo + B.lo >= k + tiny) { keep = kKeepB; return B; }
        return iv_make(r_ss(A.hi, B.lo, k), r_ss(A.lo, B.hi, k), mag);
    }
}

}  // namespace s2m
