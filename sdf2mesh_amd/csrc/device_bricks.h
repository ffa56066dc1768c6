// device_bricks.h - the dense path's bodies around a slab's sign words (device_dense.h): the
// vertex rule on the listed bricks and the emission of their vertices.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "device_dense.h"

namespace s2m {

// dualcontour.wgsl:72-131: crossings on the 12 edges in the reference's order (z-, y-, then
// x-edges), counted iff the sign changes and the crossing is not at the cell origin;
// the centroid if at least two count.  c in corner order 000,100,010,110,001,101,011,111.
__device__ __forceinline__ bool contour_cell(const float c[8], const float lo[3], const float hi[3], float pos[3])
{
    // (corner a, corner b, axis of t, fixed x, fixed y, fixed z)
    constexpr uint8_t E[12][6] = {{0, 4, 2, 0, 0, 0}, {2, 6, 2, 0, 1, 0}, {1, 5, 2, 1, 0, 0},
                                  {3, 7, 2, 1, 1, 0}, {0, 2, 1, 0, 0, 0}, {4, 6, 1, 0, 0, 1},
                                  {1, 3, 1, 1, 0, 0}, {5, 7, 1, 1, 0, 1}, {0, 1, 0, 0, 0, 0},
                                  {4, 5, 0, 0, 0, 1}, {2, 3, 0, 0, 1, 0}, {6, 7, 0, 0, 1, 1}};
    uint32_t pm = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k) pm |= (uint32_t)(c[k] > 0.0f) << k;
    if (pm == 0u || pm == 0xffu) return false;
    float ax = 0.0f, ay = 0.0f, az = 0.0f, cnt = 0.0f;
#pragma unroll
    for (int e = 0; e < 12; ++e) {
        const float v0 = c[E[e][0]], v1 = c[E[e][1]];
        const float t = (0.0f - v0) / (v1 - v0);
        float x = E[e][3], y = E[e][4], z = E[e][5];
        if (E[e][2] == 0) x = t;
        else if (E[e][2] == 1) y = t;
        else z = t;
        if ((v0 > 0.0f) == (v1 > 0.0f)) x = y = z = 0.0f;
        if (x > 0.0f || y > 0.0f || z > 0.0f) {
            ax = ax + x;
            ay = ay + y;
            az = az + z;
            cnt = cnt + 1.0f;
        }
    }
    if (cnt <= 1.0f) return false;
    pos[0] = canonical_nan(lo[0] + ((hi[0] - lo[0]) * ax) / cnt);
    pos[1] = canonical_nan(lo[1] + ((hi[1] - lo[1]) * ay) / cnt);
    pos[2] = canonical_nan(lo[2] + ((hi[2] - lo[2]) * az) / cnt);
    return true;
}

// contour_cell for a cell of a 5 x 5 x 5 block of values (val: its corner 000), over the
// edges that change sign only, with one copy of the division: fewer of them run.
// pm: the corners > 0.  Edge e goes from corner `a` (3 bits of kEdgeA) along axis 2 - e / 4.
__device__ __forceinline__ bool contour_block(const float* val, uint32_t pm, const float lo[3], const float hi[3],
                                              float pos[3])
{
    constexpr uint64_t kEdgeA = 0ull | 2ull << 3 | 1ull << 6 | 3ull << 9 | 0ull << 12 | 4ull << 15 | 1ull << 18 |
                                5ull << 21 | 0ull << 24 | 4ull << 27 | 2ull << 30 | 6ull << 33;
    uint32_t todo = 0;
#pragma unroll
    for (uint32_t e = 0; e < 12; ++e) {
        const uint32_t a = (uint32_t)(kEdgeA >> (3u * e)) & 7u, b = a + (4u >> (e >> 2));
        todo |= (((pm >> a) ^ (pm >> b)) & 1u) << e;
    }
    float ax = 0.0f, ay = 0.0f, az = 0.0f, cnt = 0.0f;
    while (todo) {
        const uint32_t e = (uint32_t)__builtin_ctz(todo), axis = 2u - (e >> 2);
        todo &= todo - 1u;
        const uint32_t a = (uint32_t)(kEdgeA >> (3u * e)) & 7u;
        const float* p = val + (a >> 2) * 25u + ((a >> 1) & 1u) * 5u + (a & 1u);
        const float v0 = p[0], v1 = p[axis == 0u ? 1 : axis == 1u ? 5 : 25];
        const float t = (0.0f - v0) / (v1 - v0);
        const float x = axis == 0u ? t : (float)(a & 1u), y = axis == 1u ? t : (float)((a >> 1) & 1u);
        const float z = axis == 2u ? t : (float)(a >> 2);
        if (x > 0.0f || y > 0.0f || z > 0.0f) {
            ax = ax + x;
            ay = ay + y;
            az = az + z;
            cnt = cnt + 1.0f;
        }
    }
    if (cnt <= 1.0f) return false;
    const float s[3] = {ax, ay, az};
    for (int k = 0; k < 3; ++k) pos[k] = canonical_nan(lo[k] + ((hi[k] - lo[k]) * s[k]) / cnt);
    return true;
}

// Sign bits of a cell (dualcontour.wgsl:57-69).
__device__ __forceinline__ uint32_t sign_bits(const float c[8])
{
    return (uint32_t)(c[1] > 0.0f) | ((uint32_t)(c[2] > 0.0f) << 1) | ((uint32_t)(c[4] > 0.0f) << 2) |
           ((uint32_t)(c[0] > 0.0f) << 3);
}

struct KeptValues {};  // in place of an SDF: its values are in `vals`

// The listed bricks, four at a time per block of 256 (one wave each).  The SDF at the
// corners of the cells with a sign change (at most 5 x 5 x 5 points per brick) goes into
// LDS: with KeptValues from `vals`, else evaluated, the four bricks' points listed together
// so that the evaluating waves are full; then one lane per cell, the vertex rule.  Vertices
// are staged (position, sign bits) at the record's base in cell order, the record's mask
// becomes the cells with a vertex and their bits are set in `actbits` (zero on entry).
template <class F>
__device__ __forceinline__ void contour_bricks(const F& sdf, const BrickArgs& a)
{
    constexpr bool kKept = __is_same(F, KeptValues);
    __shared__ float val[4 * 125];
    __shared__ uint16_t list[kKept ? 1 : 4 * 125];  // brick * 125 + point
    __shared__ uint32_t count[4], org[4][3];
    const uint32_t l = threadIdx.x & 63u, w = threadIdx.x >> 6, nrec = (uint32_t)*a.alloc;
    for (uint32_t r0 = blockIdx.x * 4u; r0 < nrec; r0 += gridDim.x * 4u) {  // block-uniform
        const bool mine = r0 + w < nrec;
        BrickRec* R = a.recs + (mine ? r0 + w : r0);
        const uint64_t mask = mine ? R->mask : 0ull;
        const uint32_t ix0 = R->bx * 4u, iy0 = R->by * 4u, iz0 = a.lz0 + R->bz * 4u;
        // points p = (z * 5 + y) * 5 + x used by a cell of the mask: of the cells x - 1, x (and
        // so on), as a 64-bit product of the three axes' pairs
        size_t brick = 0;  // the values of the lane's brick of the eight
        if constexpr (kKept) {
            const uint32_t d = l & 7u, bx = R->bx - a.bx0 + (d & 1u), by = R->by - a.by0 + ((d >> 1) & 1u);
            const uint32_t bz = R->bz + (d >> 2);
            if (l < 8u && bx < a.nbx && by < a.nby && bz < a.nbz) brick = brick_vals(a, bx, by, bz);
        }
        [[maybe_unused]] uint64_t need[2];
        [[maybe_unused]] uint32_t n = 0;
#pragma unroll
        for (uint32_t h = 0; h < 2; ++h) {
            const uint32_t p = h * 64u + l, pz = p / 25u, py = (p / 5u) % 5u, px = p % 5u;
            const uint32_t xm = (3u << px) >> 1 & 15u, ym = (3u << py) >> 1 & 15u, zm = (3u << pz) >> 1 & 15u;
            const uint32_t rows = ((ym & 1u) | (ym & 2u) << 3 | (ym & 4u) << 6 | (ym & 8u) << 9) * xm;
            const uint64_t cells = (zm & 1u ? (uint64_t)rows : 0ull) | (zm & 2u ? (uint64_t)rows << 16 : 0ull) |
                                   (zm & 4u ? (uint64_t)rows << 32 : 0ull) | (zm & 8u ? (uint64_t)rows << 48 : 0ull);
            const bool used = p < 125u && (mask & cells) != 0ull;
            if constexpr (kKept) {
                const uint32_t d = (px >> 2) | (py >> 2) << 1 | (pz >> 2) << 2;
                const size_t at = (size_t)__shfl((long long)brick, (int)(d & 7u), 64);
                if (used) val[w * 125u + p] = a.vals[at + (pz & 3u) * 16u + (py & 3u) * 4u + (px & 3u)];
            } else {
                need[h] = __ballot(used);
                n += (uint32_t)__popcll(need[h]);
            }
        }
        if constexpr (!kKept) {
            if (l == 0) {
                count[w] = n;
                org[w][0] = ix0;
                org[w][1] = iy0;
                org[w][2] = iz0;
            }
            __syncthreads();
            uint32_t at = 0, total = 0;
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k) {
                at += k < w ? count[k] : 0u;
                total += count[k];
            }
#pragma unroll
            for (uint32_t h = 0; h < 2; ++h) {
                if ((need[h] >> l) & 1ull)
                    list[at + (uint32_t)__popcll(need[h] & ((1ull << l) - 1ull))] = (uint16_t)(w * 125u + h * 64u + l);
                at += (uint32_t)__popcll(need[h]);
            }
            __syncthreads();
            for (uint32_t i = threadIdx.x; i < total; i += 256u) {
                const uint32_t q = list[i], b = q / 125u, p = q - b * 125u;
                val[q] = sdf(a.cx[org[b][0] + p % 5u], a.cy[org[b][1] + (p / 5u) % 5u], a.cz[org[b][2] + p / 25u]);
            }
        }
        __syncthreads();
        const uint32_t x = l & 3u, y = (l >> 2) & 3u, z = l >> 4;
        bool act = false;
        float pos[3] = {0.0f, 0.0f, 0.0f};
        uint32_t sg = 0;
        if ((mask >> l) & 1ull) {
            const float* c = val + w * 125u + (z * 5u + y) * 5u + x;
            uint32_t pm = 0;
#pragma unroll
            for (uint32_t k = 0; k < 8; ++k) pm |= (uint32_t)(c[(k >> 2) * 25u + ((k >> 1) & 1u) * 5u + (k & 1u)] > 0.0f) << k;
            const float lo[3] = {a.cx[ix0 + x], a.cy[iy0 + y], a.cz[iz0 + z]};
            const float hi[3] = {a.cx[ix0 + x + 1u], a.cy[iy0 + y + 1u], a.cz[iz0 + z + 1u]};
            act = contour_block(c, pm, lo, hi, pos);
            sg = ((pm >> 1) & 3u) | ((pm >> 2) & 4u) | ((pm & 1u) << 3);  // sign_bits
        }
        const uint64_t m = __ballot(act);
        if (act) {
            const uint64_t cell =
                ((uint64_t)(a.coz[iz0 + z] - a.z0) * a.ry + a.coy[iy0 + y]) * a.rx + a.cox[ix0 + x];
            atomicOr(&a.actbits[cell >> 6], 1ull << (cell & 63u));
            const uint64_t to = (uint64_t)a.stage0 + R->base + (uint32_t)__popcll(m & ((1ull << l) - 1ull));
            if (to < a.stage_cap) {
                float* s = a.stage + 3 * to;
                s[0] = pos[0];
                s[1] = pos[1];
                s[2] = pos[2];
                a.stage_sign[to] = (uint8_t)sg;
            }
        }
        if (mine && l == 0) R->mask = m;
        // the next round's writes to count, list and val follow barriers that every reader of
        // this round passes first: count is read before the second, list before the third,
        // val (own wave's bricks, written by all waves) after it, so one more is needed
        __syncthreads();
    }
}

// Ordered index of the vertex of slab cell `cell` (which has one).
__device__ __forceinline__ uint32_t vertex_rank(const BrickArgs& a, uint64_t cell)
{
    const unsigned long long word = a.actbits[cell >> 6];
    return a.cbase[cell >> 20] + a.boffset[cell >> 10] + a.wpre[cell >> 6] +
           (uint32_t)__popcll(word & ((1ull << (cell & 63u)) - 1ull));
}

// The staged vertices written at their ordered index with key, sign bits and normal (zeros
// without `normals` and with KeptValues as the SDF: vertex_normals follows), four bricks at a
// time per block of 256, their vertices listed together.  Four lanes per vertex, one per tap of
// the normal; three of them store the vertex as 8-byte pairs where vtx allows it.  One lane per
// vertex where no normal is taken here: the four bricks' vertices in one round.
template <class F>
__device__ __forceinline__ void emit_bricks(const F& sdf, const BrickArgs& a)
{
    __shared__ uint8_t list[256];  // brick << 6 | cell
    __shared__ uint32_t count[4], org[4][4];
    const uint32_t l = threadIdx.x & 63u, w = threadIdx.x >> 6, nrec = (uint32_t)*a.alloc;
    constexpr uint32_t kLanes = __is_same(F, KeptValues) ? 1u : 4u;
    const uint32_t tap = l & (kLanes - 1u);
    const bool pairs = ((size_t)a.vtx & 7u) == 0;  // a caller's buffer may be 4-byte aligned
    for (uint32_t r0 = blockIdx.x * 4u; r0 < nrec; r0 += gridDim.x * 4u) {  // block-uniform
        const bool mine = r0 + w < nrec;
        const BrickRec* R = a.recs + (mine ? r0 + w : r0);
        const uint64_t mask = mine ? R->mask : 0ull;
        if (l == 0) {
            count[w] = (uint32_t)__popcll(mask);
            org[w][0] = R->bx * 4u;
            org[w][1] = R->by * 4u;
            org[w][2] = a.lz0 + R->bz * 4u;
            org[w][3] = R->base;
        }
        __syncthreads();
        uint32_t first[4], total = 0;  // the bricks' first list entries
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) {
            first[k] = total;
            total += count[k];
        }
        const uint32_t at0 = w == 0 ? first[0] : w == 1 ? first[1] : w == 2 ? first[2] : first[3];
        if ((mask >> l) & 1ull) list[at0 + (uint32_t)__popcll(mask & ((1ull << l) - 1ull))] = (uint8_t)(w << 6 | l);
        __syncthreads();
        for (uint32_t e = threadIdx.x / kLanes; e < total; e += 256u / kLanes) {
            const uint32_t q = list[e], b = q >> 6, c = q & 63u;
            const uint32_t f = b == 0 ? first[0] : b == 1 ? first[1] : b == 2 ? first[2] : first[3];
            const uint32_t X = a.cox[org[b][0] + (c & 3u)], Y = a.coy[org[b][1] + ((c >> 2) & 3u)];
            const uint32_t Z = a.coz[org[b][2] + (c >> 4)];
            const uint32_t v = vertex_rank(a, ((uint64_t)(Z - a.z0) * a.ry + Y) * a.rx + X);
            const uint64_t at = (uint64_t)a.stage0 + org[b][3] + (e - f);
            if (v >= a.vcap) continue;  // the job is repeated with larger buffers
            if (at >= a.stage_cap) {    // likewise, but the quad pass reads this vertex's key: without sign
                                        // changes it forms no quads
                if (tap == 0u) {
                    a.keys[v] = (uint64_t)X | ((uint64_t)Y << 16) | ((uint64_t)Z << 32);
                    a.signs[v] = 0;
                }
                continue;
            }
            const float px = a.stage[3 * at], py = a.stage[3 * at + 1], pz = a.stage[3 * at + 2];
            float* o = a.vtx + 6 * (size_t)v;
            float nrm[6] = {px, py, pz, 0.0f, 0.0f, 0.0f};
            if constexpr (!__is_same(F, KeptValues))
                if (a.normals) tap_normal(sdf, px, py, pz, a.eps, tap, nrm);
            const uint32_t each = kLanes == 1u ? 3u : tap < 3u ? 1u : 0u;  // pairs of this lane
#pragma unroll
            for (uint32_t k = 0; k < (kLanes == 1u ? 3u : 1u); ++k) {
                const uint32_t i = kLanes == 1u ? k : tap;
                const float n0 = i == 0u ? nrm[0] : i == 1u ? nrm[2] : nrm[4];
                const float n1 = i == 0u ? nrm[1] : i == 1u ? nrm[3] : nrm[5];
                if (k < each && pairs) {
                    *reinterpret_cast<float2*>(o + 2 * i) = make_float2(n0, n1);
                } else if (k < each) {
                    o[2 * i] = n0;
                    o[2 * i + 1] = n1;
                }
            }
            if (tap == 0u) {
                a.keys[v] = (uint64_t)X | ((uint64_t)Y << 16) | ((uint64_t)Z << 32);
                a.signs[v] = a.stage_sign[at];
            }
        }
        __syncthreads();  // list, count and org are read
    }
}

}  // namespace s2m
