// kernels.hip - HIP kernels of the meshing path for gfx950 (wave64).
//
// The dense path meshes programs that interval bounds cannot prune (the Mandelbulb,
// compiled programs, S2M_DENSE_EVAL).  Per z-slab of cells the host launches, in stream
// order (bodies: device_dense.h, device_bricks.h; a compiled program's s2m_c_signs and
// s2m_c_normals are in its own module):
//   k_signs            sign of the SDF at every corner-lattice point, one bit each  (VALU bound)
//   k_find_bricks      the 4x4x4 bricks whose cells change sign
//   k_contour          their cells' corner values (kept by the sign pass, or taken where the signs
//                      were decided early), the vertex rule, staged vertices, one activity bit
//                      per cell
//   k_ranks            vertices before each word of 64 cells, block of 1024 cells and chunk
//   k_emit             staged vertices at their ordered index (after early signs with their 4-tap
//                      normals)
//   k_normals          4-tap normals
//   k_quads<0>, k_tri_offsets, k_quads<1>   triangles per 256 vertices, their offsets, triangles
//   k_slab_end         between slabs: the other slab's bits cleared
// (with several slabs the signs are evaluated one slab ahead on a second stream; per-cell
// corner dumps have k_cells<0/1> in place of the brick kernels).  A cell's vertex index is
// never stored: it is its chunk's first vertex plus the vertices before it in the chunk.  Cells are
// numbered in (z, y, x) order inside the slab, the reference's output order (VertexList
// order, mesh.rs:280-321).
#include <algorithm>
#include <mutex>

#include "device_bricks.h"
#include "device_dense.h"
#include "device_scan.h"
#include "device_sdf.h"
#include "internal.h"

namespace s2m {

__device__ __forceinline__ uint32_t fdiv(uint32_t n, FastDiv f)
{
    const uint64_t t = (uint64_t)__umulhi(n, f.m) + n;
    return (uint32_t)(t >> f.l);
}

__device__ __forceinline__ uint32_t lane_id() { return threadIdx.x & 63u; }

// Exclusive prefix of v over the 256 threads of the block (4 waves); *total = sum.
// Contains two __syncthreads: every thread of the block must call it.
__device__ __forceinline__ uint32_t block_exclusive_256(uint32_t v, uint32_t* lds, uint32_t* total)
{
    const uint32_t lane = lane_id(), w = threadIdx.x >> 6;
    uint32_t inc = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t t = __shfl_up(inc, d, 64);
        if (lane >= (uint32_t)d) inc += t;
    }
    if (lane == 63) lds[w] = inc;
    __syncthreads();
    uint32_t woff = 0, tot = 0;
#pragma unroll
    for (uint32_t k = 0; k < kBlock / 64; ++k) {
        const uint32_t s = lds[k];
        woff += (k < w) ? s : 0u;
        tot += s;
    }
    __syncthreads();
    *total = tot;
    return woff + inc - v;
}

// ---------------------------------------------------------------------------------
// SDFs of the tape programs, for the dense bodies (device_dense.h).
// ---------------------------------------------------------------------------------
// (The kernels take the tape as a __restrict__ argument and the call is inlined, so that the
// wave-uniform ops are read through the scalar cache beside the kernels' stores.)
struct TapeSdf {
    const s2m_op* ops;
    uint32_t n;
    __device__ __forceinline__ float operator()(float x, float y, float z) const { return tape_eval(ops, n, x, y, z); }
};

// A tape that is one power-8 Mandelbulb op: the estimator called directly with its operands
// (wave-uniform loads), as tape_eval calls it, so the values are the interpreter's bit for
// bit without its dispatch and the other forms' registers.
struct MandelSdf {
    float offset, bailout, t2;
    uint32_t iters;
    bool swap;
    __device__ explicit MandelSdf(const s2m_op* op)
        : offset(op->f[2]), bailout(op->f[1]), t2(op->f[3]), iters(op->iarg & 0xffffu),
          swap((op->iarg & S2M_MANDEL_SWAP_YZ) != 0)
    {
    }
    __device__ float operator()(float x, float y, float z) const
    {
        return mandelbulb8<false>(x, swap ? z : y, swap ? y : z, offset, iters, t2, bailout, 0.0f);
    }
};

// Its sign, with the early decisions of mandelbulb8<true> (their preconditions hold:
// mandel_sign_ok), and of whole bricks by the two decisions of the first step on the box:
// inside the inner ball everywhere, or past the bailout (or predicted past it) everywhere.
struct MandelSign : MandelSdf {
    float gain;
    static constexpr bool kBricks = true;
    static constexpr bool kValue = false;
    __device__ explicit MandelSign(const s2m_op* op) : MandelSdf(op), gain(mandel_gain(op->f[1])) {}
    __device__ float operator()(float x, float y, float z) const
    {
        return mandelbulb8<true>(x, swap ? z : y, swap ? y : z, offset, iters, t2, bailout, gain);
    }
    __device__ int brick(float x0, float x1, float y0, float y1, float z0, float z1) const
    {
        const float xn = fmaxf(fmaxf(x0, -x1), 0.0f), xf = fmaxf(fabsf(x0), fabsf(x1));
        const float yn = fmaxf(fmaxf(y0, -y1), 0.0f), yf = fmaxf(fabsf(y0), fabsf(y1));
        const float zn = fmaxf(fmaxf(z0, -z1), 0.0f), zf = fmaxf(fabsf(z0), fabsf(z1));
        const float far2 = 1.0001f * (xf * xf + yf * yf + zf * zf);
        if (!(far2 < 1e30f)) return -1;
        if (far2 <= kMandelInner) return 0;
        const float near2 = 0.9999f * (xn * xn + yn * yn + zn * zn), n4 = near2 * near2;
        const float xy2 = xn * xn + (swap ? zn * zn : yn * yn);  // of the swizzled point
        const float far = 1.0001f * __builtin_amdgcn_sqrtf(far2), r = fminf(far, 1.0001f * bailout);
        const float r2 = r * r, r7 = r2 * r2 * r2 * r;
        if (n4 * n4 > 1.02f * (bailout + far) && xy2 >= 2.0f * kMandelAxis &&
            1.001f * (8.0f * r7 + 1.0f) * offset <= gain)
            return 1;
        return -1;
    }
};

// Lattice evaluation (s2m_eval_lattice): one thread per lattice point, each wave a
// 4 x 4 x 4 block.  Held to 64 VGPRs (8 waves per SIMD; a 12-byte spill): 3 % faster on
// a 64-primitive CSG program.
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(8, 8))) void k_eval_lattice(
    const s2m_op* __restrict__ ops, uint32_t nops, const float* __restrict__ cx, const float* __restrict__ cy,
    const float* __restrict__ cz, uint32_t nx, uint32_t ny, uint32_t lz0, uint32_t nzl, uint32_t pitch,
    float* __restrict__ lat)
{
    eval_lattice_point(TapeSdf{ops, nops}, cx, cy, cz, nx, ny, lz0, nzl, pitch, lat);
}

// MANDEL = 1: the tape is one power-8 Mandelbulb op (k_signs<2>: its sign may be decided
// early as well).
template <int MANDEL>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(8, 8))) void k_signs(BrickArgs a,
                                                                                         const s2m_op* __restrict__ ops,
                                                                                         uint32_t nops)
{
    if constexpr (MANDEL == 2) sign_words(MandelSign(ops), a);
    else if constexpr (MANDEL == 1) sign_words(PointSign<MandelSdf>{MandelSdf(ops)}, a);
    else sign_words(PointSign<TapeSdf>{TapeSdf{ops, nops}}, a);
}

// KEPT: from the values the sign pass has kept (normals from k_normals or s2m_c_normals), else
// with the power-8 Mandelbulb op `op`, whose signs were decided early.
template <bool KEPT>
__global__ __launch_bounds__(256) void k_contour(BrickArgs a, const s2m_op* __restrict__ op)
{
    if constexpr (KEPT) contour_bricks(KeptValues{}, a);
    else contour_bricks(MandelSdf(op), a);
}

template <bool KEPT>
__global__ __launch_bounds__(256) void k_emit(BrickArgs a, const s2m_op* __restrict__ op)
{
    if constexpr (KEPT) emit_bricks(KeptValues{}, a);
    else emit_bricks(MandelSdf(op), a);
}

// Normals of a tape's vertices, four full lanes each: a tap costs a whole program, where k_emit's
// rounds over the vertices of four bricks leave a third of the lanes idle (252 us for 136 in
// CSG-64 at 256^3).
template <bool MANDEL>
__global__ __launch_bounds__(256) void k_normals(const s2m_op* __restrict__ ops, uint32_t nops, float eps, float* vtx,
                                                 const uint64_t* counters, uint64_t vcap)
{
    if constexpr (MANDEL) vertex_normals<true>(MandelSdf(ops), eps, vtx, counters, vcap);
    else vertex_normals<true>(TapeSdf{ops, nops}, eps, vtx, counters, vcap);
}

// ---------------------------------------------------------------------------------
// k_find_bricks: kFindBricks bricks per thread, kBlock apart.  A brick's 64 cells' corner
// signs differ where the OR of the 8 shifted words (the brick's and its 7 neighbours'
// towards +x, +y, +z) is set and the AND is not: axis by axis, OR and AND of the word and
// its shift.  Cells between two coordinates a rounding apart, past the grid or in another
// slab are masked off by the axes' cell tables.  Bricks with a cell left are appended to
// the list, their cells reserving staging space: one 64-bit counter (records low, staged
// vertices high), one update per block of 1024 bricks (a returning update of the one
// address takes about 25 ns, one after the other: one per wave took 69 us for 157 K
// bricks of which 2 500 waves listed some).  Reads 8 words per brick, mostly from cache.
// ---------------------------------------------------------------------------------
constexpr uint32_t kFindBricks = 4;

__device__ __forceinline__ uint64_t mixed_cells(const BrickArgs& a, uint32_t i, uint32_t& bx, uint32_t& by, uint32_t& bz)
{
    const uint32_t row = i / a.ownx;
    bx = i - row * a.ownx;
    bz = row / a.owny;
    by = row - bz * a.owny;
    const uint32_t dx = bx + 1 < a.nbx ? 1u : 0u;  // past the end: cells that are masked off
    const size_t dy = by + 1 < a.nby ? a.nbx : 0u, dz = bz + 1 < a.nbz ? (size_t)a.nbx * a.nby : 0u;
    const uint64_t* w = a.words + ((size_t)bz * a.nby + by) * a.nbx + bx;
    uint64_t o[4], n4[4];  // OR / AND along x of the rows (y, z), (y + 1, z), (y, z + 1), (y + 1, z + 1)
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const uint64_t* r = w + (k & 1 ? dy : 0) + (k & 2 ? dz : 0);
        const uint64_t u = r[0], v = r[dx];
        const uint64_t s = ((u >> 1) & 0x7777777777777777ull) | ((v & 0x1111111111111111ull) << 3);
        o[k] = u | s;
        n4[k] = u & s;
    }
    auto shy = [](uint64_t u, uint64_t v) {
        return ((u >> 4) & 0x0fff0fff0fff0fffull) | ((v & 0x000f000f000f000full) << 12);
    };
    const uint64_t o0 = o[0] | shy(o[0], o[1]), o1 = o[2] | shy(o[2], o[3]);
    const uint64_t n0 = n4[0] & shy(n4[0], n4[1]), n1 = n4[2] & shy(n4[2], n4[3]);
    const uint64_t mask = (o0 | (o0 >> 16) | (o1 << 48)) & ~(n0 & ((n0 >> 16) | (n1 << 48)));
    if (!mask) return 0ull;
    uint32_t vx = 0, vy = 0, vz = 0;  // the axes' cells
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) {
        const uint32_t ix = (a.bx0 + bx) * 4u + k, iy = (a.by0 + by) * 4u + k, iz = bz * 4u + k;
        if (ix < a.nx && a.cox[ix] != kNoCell) vx |= 1u << k;
        if (iy < a.ny && a.coy[iy] != kNoCell) vy |= 1u << (4u * k);
        if (iz + 1u < a.nzl) {
            const uint32_t z = a.coz[a.lz0 + iz];
            if (z >= a.z0 && z < a.z1) vz |= 1u << k;
        }
    }
    const uint64_t rows = vx * vy;
    return mask & ((vz & 1u ? rows : 0ull) | (vz & 2u ? rows << 16 : 0ull) | (vz & 4u ? rows << 32 : 0ull) |
                   (vz & 8u ? rows << 48 : 0ull));
}

__global__ __launch_bounds__(256) void k_find_bricks(BrickArgs a)
{
    __shared__ uint32_t wrecs[kBlock / 64], wcells[kBlock / 64];
    __shared__ uint64_t base;
    const uint32_t n = a.ownx * a.owny * a.nbz;
    uint64_t mask[kFindBricks];
    BrickRec rec[kFindBricks];
    uint32_t recs = 0, cells = 0;  // of this thread
#pragma unroll
    for (uint32_t k = 0; k < kFindBricks; ++k) {
        const uint32_t i = (blockIdx.x * kFindBricks + k) * kBlock + threadIdx.x;
        uint32_t bx = 0, by = 0, bz = 0;
        mask[k] = i < n ? mixed_cells(a, i, bx, by, bz) : 0ull;
        rec[k] = BrickRec{mask[k], 0u, (uint16_t)(a.bx0 + bx), (uint16_t)(a.by0 + by), (uint16_t)bz, 0};
        recs += mask[k] != 0ull ? 1u : 0u;
        cells += (uint32_t)__popcll(mask[k]);
    }
    const uint32_t ir = wave_scan(recs), ic = wave_scan(cells);
    const uint32_t w = threadIdx.x >> 6;
    if (lane_id() == 63u) {
        wrecs[w] = ir;
        wcells[w] = ic;
    }
    __syncthreads();
    uint32_t br = 0, bc = 0, tr = 0, tc = 0;
#pragma unroll
    for (uint32_t k = 0; k < kBlock / 64; ++k) {
        br += k < w ? wrecs[k] : 0u;
        bc += k < w ? wcells[k] : 0u;
        tr += wrecs[k];
        tc += wcells[k];
    }
    if (tr == 0) return;  // block-uniform
    if (threadIdx.x == 0) base = atomicAdd((unsigned long long*)a.alloc, (unsigned long long)tr | ((unsigned long long)tc << 32));
    __syncthreads();
    uint32_t at = (uint32_t)base + br + ir - recs, to = (uint32_t)(base >> 32) + bc + ic - cells;
#pragma unroll
    for (uint32_t k = 0; k < kFindBricks; ++k) {
        if (!mask[k]) continue;
        rec[k].base = to;
        a.recs[at++] = rec[k];
        to += (uint32_t)__popcll(mask[k]);
    }
}

__device__ __forceinline__ void cell_coords(const SlabArgs& a, uint32_t i, uint32_t& x, uint32_t& y,
                                            uint32_t& zl)
{
    const uint32_t row = fdiv(i, a.div_rx);  // y + ry * zl
    x = i - row * a.rx;
    zl = fdiv(i, a.div_rxy);
    y = row - zl * a.ry;
}

// ---------------------------------------------------------------------------------
// Cell passes over per-cell corner dumps (s2m_contour_cells).  EMIT = 0: every cell's
// vertex rule, each cell's activity bit (one ballot word per 64 cells).  EMIT = 1: the
// block's cells with a vertex, listed in LDS in order, are contoured again on full waves
// (the same rule on the same corners gives the same vertex) and their vertices written.
// ---------------------------------------------------------------------------------
__device__ __forceinline__ bool cell_vertex(const SlabArgs& a, const float* __restrict__ corners, uint32_t i,
                                            uint32_t x, uint32_t y, uint32_t zl, float (&c)[8], float (&pos)[3])
{
    const float* src = corners + 8 * (size_t)i;
#pragma unroll
    for (int k = 0; k < 8; ++k) c[k] = src[k];
    const uint32_t zg = a.z0 + zl;
    const float lo[3] = {a.cx[a.lox[x]], a.cy[a.loy[y]], a.cz[a.loz[zg]]};
    const float hi[3] = {a.cx[a.hix[x]], a.cy[a.hiy[y]], a.cz[a.hiz[zg]]};
    return contour_cell(c, lo, hi, pos);
}

template <int EMIT>
__global__ __launch_bounds__(256) void k_cells(SlabArgs a, MeshBufs b, const float* __restrict__ corners)
{
    const uint32_t base = blockIdx.x * kCellsPerBlock;
    if constexpr (!EMIT) {
        for (uint32_t j = 0; j < kRounds; ++j) {
            const uint32_t i = base + j * kBlock + threadIdx.x;
            bool act = false;
            if (i < a.ncells) {
                uint32_t x, y, zl;
                float c[8], pos[3];
                cell_coords(a, i, x, y, zl);
                act = cell_vertex(a, corners, i, x, y, zl, c, pos);
            }
            const uint64_t w = __ballot(act);
            if (lane_id() == 0 && i < a.ncells) b.actbits[i >> 6] = w;
        }
    } else {
        __shared__ uint32_t list[kCellsPerBlock];  // the block's active cells, in vertex order
        const uint32_t first = b.bits.cbase[blockIdx.x >> 10] + b.bits.boffset[blockIdx.x];
        uint32_t before = 0;  // active cells of earlier rounds
        for (uint32_t j = 0; j < kRounds; ++j) {
            const uint32_t i0 = base + j * kBlock, i = i0 + threadIdx.x;
            const uint32_t wv = threadIdx.x >> 6, ln = lane_id();
            uint64_t wd[kBlock / 64];
#pragma unroll
            for (uint32_t k = 0; k < kBlock / 64; ++k) wd[k] = i0 + 64u * k < a.ncells ? b.actbits[(i0 >> 6) + k] : 0ull;
            uint32_t rank = before, total = 0;
#pragma unroll
            for (uint32_t k = 0; k < kBlock / 64; ++k) {
                const uint32_t pc = (uint32_t)__builtin_popcountll(wd[k]);
                total += pc;
                if (k < wv) rank += pc;
            }
            const uint64_t mine = wd[wv];
            rank += (uint32_t)__builtin_popcountll(mine & ((1ull << ln) - 1ull));
            if (i < a.ncells && ((mine >> ln) & 1ull)) list[rank] = i;
            before += total;
        }
        __syncthreads();  // the block's list is complete
        for (uint32_t q = threadIdx.x; q < before; q += kBlock) {
            const uint32_t i = list[q];
            const uint64_t v = (uint64_t)first + q;
            uint32_t x, y, zl;
            float c[8], pos[3];
            cell_coords(a, i, x, y, zl);
            cell_vertex(a, corners, i, x, y, zl, c, pos);
            if (v < b.vcap) {
                float* o = b.vtx + 6 * v;
                o[0] = pos[0];
                o[1] = pos[1];
                o[2] = pos[2];
                o[3] = 0.0f;
                o[4] = 0.0f;
                o[5] = 0.0f;
                b.keys[v] = (uint64_t)x | ((uint64_t)y << 16) | ((uint64_t)(a.z0 + zl) << 32);
                b.signs[v] = (uint8_t)sign_bits(c);
            }
        }
    }
}

// ---------------------------------------------------------------------------------
// k_ranks: from the slab's activity bits, the vertices before each word in its block of 16
// words, before each block in its chunk of 1024 blocks, and each chunk's first vertex.
// One workgroup of 1024 per chunk (a thread's 16 words, 1024 apart, in flight at once; 16
// lanes per block), so a slab of 32 M cells is 32 workgroups of 128 KB each.  A chunk adds
// its sum to the bases of the chunks after it and to the running total (set to the
// slab's first vertex by the kernel that begins the slab): one launch, with no workgroup
// waiting for others.  A count kernel and a two-launch scan took 14 us at any small size; a
// last workgroup scanning behind device-scope fences more than that.
// ---------------------------------------------------------------------------------
__global__ __launch_bounds__(1024) void k_ranks(const uint64_t* __restrict__ bits, uint32_t nwords,
                                                uint16_t* __restrict__ wpre, uint32_t* __restrict__ boffset,
                                                uint32_t* __restrict__ cbase, uint64_t* __restrict__ counters)
{
    __shared__ uint32_t count[1024], wsum[16];
    const uint32_t t = threadIdx.x, l = t & 15u, w0 = blockIdx.x * 16384u;
    uint64_t word[16];
#pragma unroll
    for (uint32_t k = 0; k < 16u; ++k) {
        const uint32_t i = w0 + k * 1024u + t;
        word[k] = i < nwords ? bits[i] : 0ull;
    }
#pragma unroll
    for (uint32_t k = 0; k < 16u; ++k) {
        const uint32_t i = w0 + k * 1024u + t, n = (uint32_t)__popcll(word[k]);
        const uint32_t upto = row_scan(n);
        if (i < nwords) wpre[i] = (uint16_t)(upto - n);
        if (l == 15u) count[k * 64u + (t >> 4)] = upto;
    }
    __syncthreads();
    const uint32_t mine = count[t], upto = wave_scan(mine);
    if (lane_id() == 63u) wsum[t >> 6] = upto;
    __syncthreads();
    uint32_t before = 0, all = 0;
#pragma unroll
    for (uint32_t k = 0; k < 16u; ++k) {
        before += k < (t >> 6) ? wsum[k] : 0u;
        all += wsum[k];
    }
    if (blockIdx.x * 1024u + t < (nwords + 15u) / 16u) boffset[blockIdx.x * 1024u + t] = before + upto - mine;
    if (all == 0u) return;
    if (t < gridDim.x && t > blockIdx.x) atomicAdd(&cbase[t], all);
    if (t == 0) atomicAdd((unsigned long long*)&counters[kVtxTotal], (unsigned long long)all);
}

// The slab's vertices that have been written, [kVtxPrev, kVtxTotal) below the capacity, in
// groups of kBlock.
__device__ __forceinline__ uint32_t vertex_groups(const uint64_t* counters, uint64_t vcap)
{
    const uint64_t beg = counters[kVtxPrev], end = min(counters[kVtxTotal], vcap);
    return end > beg ? (uint32_t)((end - beg + kBlock - 1u) / kBlock) : 0u;
}

// A slab's or pass's totals to mapped host memory (kSnapWords): past the device's caches, so
// that a polling host sees them while the kernels after this one run.
__device__ __forceinline__ void write_snapshot(uint64_t* snap, uint64_t nv, uint64_t nt, uint64_t slots, uint64_t staged)
{
    const uint64_t v[kSnapWords] = {nv, nt, slots, staged};
    for (uint32_t i = 0; i < kSnapWords; ++i)
        __hip_atomic_store(snap + i, v[i] | kSnapValid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// The groups' triangle counts (k_quads<0>) into their offsets, and the running total, by one
// workgroup: a slab's 600 K vertices are 2 400 groups, one round.  The staging use is folded into
// its maximum here, and after a job's last slab the counters (final then: k_quads<1> changes
// none) go to `back` (mapped host memory, else NULL), so that no k_slab_end follows it.
__global__ __launch_bounds__(1024) void k_tri_offsets(const uint32_t* __restrict__ tcount, uint32_t* __restrict__ toffset,
                                                      uint64_t* __restrict__ counters, uint64_t vcap,
                                                      uint64_t* snap, uint64_t* back)
{
    __shared__ uint32_t wsum[16];
    const uint32_t groups = vertex_groups(counters, vcap), t = threadIdx.x;
    const uint64_t prev = counters[kTriTotal];
    uint64_t run = prev;
    for (uint32_t g0 = 0; g0 < groups; g0 += 4096u) {
        uint32_t n[4], sum = 0;
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) {
            const uint32_t g = g0 + 4u * t + k;
            n[k] = g < groups ? tcount[g] : 0u;
            sum += n[k];
        }
        const uint32_t upto = wave_scan(sum);
        __syncthreads();  // the previous round's readers of wsum
        if (lane_id() == 63u) wsum[t >> 6] = upto;
        __syncthreads();
        uint32_t before = 0, all = 0;
#pragma unroll
        for (uint32_t k = 0; k < 16u; ++k) {
            before += k < (t >> 6) ? wsum[k] : 0u;
            all += wsum[k];
        }
        uint64_t at = run + before + upto - sum;
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) {
            const uint32_t g = g0 + 4u * t + k;
            if (g < groups) toffset[g] = (uint32_t)at;
            at += n[k];
        }
        run += all;
    }
    if (t == 0) {
        counters[kTriPrev] = prev;
        counters[kTriTotal] = run;
        const uint64_t used = counters[kBrickAlloc] >> 32;
        if (snap) write_snapshot(snap, counters[kVtxTotal], run, 0, used);
        if (used > counters[kStageMax]) counters[kStageMax] = used;
        if (back)
            for (uint32_t i = 0; i < kNumCounters; ++i) back[i] = counters[i];
    }
}

// ---------------------------------------------------------------------------------
// Quad pass (mesh.rs:267-324).  Per vertex of the slab, [kVtxPrev, kVtxTotal) in cell
// order: the x-, y- and z-edge quads of its cell from its key and sign bits, neighbour
// vertices from the activity bits of this slab and, for plane z0 - 1, of the one before.
// A quad with a missing vertex is skipped and counted (mesh.rs:270-278).  Blocks walk
// groups of kBlock vertices (their number is only known on the device).  EMIT = 0 counts
// the groups' triangles, EMIT = 1 writes them in order.  A vertex beyond the output
// capacity has no key: it forms no quads (the job repeats with a larger capacity).
// ---------------------------------------------------------------------------------
template <int EMIT>
__global__ __launch_bounds__(256) void k_quads(SlabArgs a, MeshBufs b, SlabBits prev)
{
    __shared__ uint32_t lds[kBlock / 64];
    const uint64_t vbeg = b.counters[kVtxPrev], vend = min(b.counters[kVtxTotal], b.vcap);
    const uint32_t groups = vertex_groups(b.counters, b.vcap);
    const uint64_t plane = (uint64_t)a.rx * a.ry;
    const bool lag = (a.flags & S2M_COMPAT_DROP_LAST_SLICE) != 0;
    uint32_t invalid = 0;
    for (uint32_t g = blockIdx.x; g < groups; g += gridDim.x) {  // block-uniform
        const uint64_t vv = vbeg + (uint64_t)g * kBlock + threadIdx.x;
        uint32_t q[3][4];
        uint32_t nq = 0;  // bit e set: quad e is valid
        if (vv < vend) {
            const uint32_t v = (uint32_t)vv;
            const uint64_t key = b.keys[v];
            const uint32_t x = (uint32_t)(key & 0xffffu), y = (uint32_t)((key >> 16) & 0xffffu);
            const uint32_t zg = (uint32_t)(key >> 32), zl = zg - a.z0;
            // the vertex of the cell at offset `off` of the cell plane (EMIT = 0: whether it
            // has one), in this plane or the one below
            auto at = [&](bool below, uint64_t off) -> uint32_t {
                const bool old = below && zl == 0;
                const SlabBits& t = old ? prev : b.bits;
                const uint64_t cell = old ? prev.last_plane + off : (uint64_t)(zl - (below ? 1u : 0u)) * plane + off;
                const unsigned long long word = t.words[cell >> 6];
                const uint32_t bit = (uint32_t)(cell & 63u);
                if (!((word >> bit) & 1ull)) return kNone;
                if (!EMIT) return 0u;
                return t.cbase[cell >> 20] + t.boffset[cell >> 10] + t.wpre[cell >> 6] + (uint32_t)__popcll(word & ((1ull << bit) - 1ull));
            };
            const uint32_t s = b.signs[v];
            const bool c0 = s & 1, c1 = (s >> 1) & 1, c2 = (s >> 2) & 1, c3 = (s >> 3) & 1;
            const uint64_t r0 = (uint64_t)y * a.rx, rm = r0 - a.rx;
            // x-edge: Quad(v(x,y-1,z-1), v(x,y,z-1), v(x,y,z), v(x,y-1,z)).swap(c.0)
            if (c0 != c3 && y > 0) {
                if (zg > 0) {
                    uint32_t t[4] = {at(true, rm + x), at(true, r0 + x), v, at(false, rm + x)};
                    if (c0) { q[0][0] = t[3]; q[0][1] = t[2]; q[0][2] = t[1]; q[0][3] = t[0]; }
                    else { q[0][0] = t[0]; q[0][1] = t[1]; q[0][2] = t[2]; q[0][3] = t[3]; }
                    if (t[0] != kNone && t[1] != kNone && t[3] != kNone) nq |= 1;
                    else ++invalid;
                } else if (lag) {
                    ++invalid;  // the lagged reference looks up label z-1 and misses
                }
            }
            // y-edge: Quad(v(x-1,y,z-1), v(x,y,z-1), v(x,y,z), v(x-1,y,z)).swap(!c.1)
            if (c1 != c3 && x > 0) {
                if (zg > 0) {
                    uint32_t t[4] = {at(true, r0 + x - 1), at(true, r0 + x), v, at(false, r0 + x - 1)};
                    if (!c1) { q[1][0] = t[3]; q[1][1] = t[2]; q[1][2] = t[1]; q[1][3] = t[0]; }
                    else { q[1][0] = t[0]; q[1][1] = t[1]; q[1][2] = t[2]; q[1][3] = t[3]; }
                    if (t[0] != kNone && t[1] != kNone && t[3] != kNone) nq |= 2;
                    else ++invalid;
                } else if (lag) {
                    ++invalid;
                }
            }
            // z-edge: Quad(v(x-1,y-1,z), v(x,y-1,z), v(x,y,z), v(x-1,y,z)).swap(c.2)
            if (c2 != c3 && x > 0 && y > 0) {
                uint32_t t[4] = {at(false, rm + x - 1), at(false, rm + x), v, at(false, r0 + x - 1)};
                if (c2) { q[2][0] = t[3]; q[2][1] = t[2]; q[2][2] = t[1]; q[2][3] = t[0]; }
                else { q[2][0] = t[0]; q[2][1] = t[1]; q[2][2] = t[2]; q[2][3] = t[3]; }
                if (t[0] != kNone && t[1] != kNone && t[3] != kNone) nq |= 4;
                else ++invalid;
            }
        }
        const uint32_t ntri = 2u * (uint32_t)__builtin_popcount(nq);
        uint32_t total;
        const uint32_t rank = block_exclusive_256(ntri, lds, &total);
        if (EMIT) {
            uint64_t t = (uint64_t)b.toffset[g] + rank;
#pragma unroll
            for (int e = 0; e < 3; ++e) {
                if (!(nq & (1u << e))) continue;
                // make_triangles: (q2, q1, q0), (q0, q3, q2)  (lib.rs:199-205)
                if (t + 1 < b.tcap) {
                    uint32_t* o = b.tri + 3 * t;
                    o[0] = q[e][2];
                    o[1] = q[e][1];
                    o[2] = q[e][0];
                    o[3] = q[e][0];
                    o[4] = q[e][3];
                    o[5] = q[e][2];
                }
                t += 2;
            }
        } else if (threadIdx.x == 0) {
            b.tcount[g] = total;
        }
    }
    if (!EMIT && invalid) atomicAdd((unsigned long long*)&b.counters[kInvalid], (unsigned long long)invalid);
}

// ---------------------------------------------------------------------------------
// Every float bit pattern x: sincosf(x) against sinf(x) and cosf(x), bitwise.  cnt[0] /
// cnt[2]: sine / cosine results that differ, cnt[1] / cnt[3]: those of them where both
// are NaN.  (The Mandelbulb's escape step takes sine and cosine with one sincosf.)
// ---------------------------------------------------------------------------------
// Each side in a function of its own that is never inlined: a sinf and a cosf of the
// same argument in one function may be merged into one sincos call by the compiler,
// and the check would then compare sincosf with itself.
__device__ __attribute__((noinline)) float check_sin(float x) { return sinf(x); }
__device__ __attribute__((noinline)) float check_cos(float x) { return cosf(x); }
__device__ __attribute__((noinline)) void check_sincos(float x, float* s, float* c) { sincosf(x, s, c); }

__global__ __launch_bounds__(256) void k_sincos_check(unsigned long long* __restrict__ cnt)
{
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < (1ull << 32);
         i += (uint64_t)gridDim.x * blockDim.x) {
        const float x = __uint_as_float((uint32_t)i);
        const float s1 = check_sin(x), c1 = check_cos(x);
        float s2, c2;
        check_sincos(x, &s2, &c2);
        if (__float_as_uint(s1) != __float_as_uint(s2)) atomicAdd(&cnt[(s1 != s1 && s2 != s2) ? 1 : 0], 1ull);
        if (__float_as_uint(c1) != __float_as_uint(c2)) atomicAdd(&cnt[(c1 != c1 && c2 != c2) ? 3 : 2], 1ull);
    }
}

// The Mandelbulb's bailout test r > b on r = sqrtf(r^2) taken as r^2 > t with
// t = bailout_threshold(b).  Bailouts b: 2^20 bit patterns spread over all 2^32
// (stride 4099: denormals, normals, infinities, NaNs, both signs) and 2.0; squared
// lengths x: the 65 floats around b * b and 0, the smallest denormal, 1, +inf and NaN,
// each x >= 0 or NaN as a sum of squares is.  cnt[0]: comparisons, cnt[1]: those where
// the two tests disagree.
// ---------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_bailout_check(unsigned long long* __restrict__ cnt)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i > (1u << 20)) return;
    const float b = i == (1u << 20) ? 2.0f : __uint_as_float(i * 4099u);
    const float t = bailout_threshold(b);
    const uint32_t u = __float_as_uint(b * b);
    uint32_t checked = 0, bad = 0;
    for (int d = -37; d <= 32; ++d) {
        float x;
        switch (d) {
        case -37: x = 0.0f; break;
        case -36: x = __uint_as_float(1u); break;
        case -35: x = 1.0f; break;
        case -34: x = __uint_as_float(0x7f800000u); break;
        case -33: x = __uint_as_float(0x7fc00000u); break;
        default: x = __uint_as_float(u + (uint32_t)d); break;
        }
        if (x != x ? false : (__float_as_uint(x) >> 31) != 0u) continue;  // negative: no sum of squares
        ++checked;
        bad += (sqrtf(x) > b) != (x > t);
    }
    atomicAdd(&cnt[0], (unsigned long long)checked);
    if (bad) atomicAdd(&cnt[1], (unsigned long long)bad);
}

// ---------------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------------
hipError_t launch_eval_lattice(hipStream_t s, const s2m_op* ops, uint32_t nops, const float* cx,
                               const float* cy, const float* cz, uint32_t nx, uint32_t ny,
                               uint32_t lz0, uint32_t nzl, uint32_t pitch, float* lat)
{
    if (nx == 0 || ny == 0 || nzl == 0) return hipSuccess;
    dim3 grid((nx + 15) / 16, (ny + 3) / 4, (nzl + 3) / 4);
    hipLaunchKernelGGL(k_eval_lattice, grid, dim3(256), 0, s, ops, nops, cx, cy, cz, nx, ny, lz0, nzl,
                       pitch, lat);
    return hipGetLastError();
}

// Whether a tape is one power-8 Mandelbulb op, and whether mandelbulb8<true>'s
// preconditions hold for it.
bool mandel_power8(const s2m_op* ops, uint32_t n)
{
    return n == 1 && ops[0].code == S2M_OP_MANDELBULB && ops[0].f[0] == 8.0f && !(ops[0].iarg & S2M_MANDEL_TRIG);
}
static bool mandel_sign_ok(const s2m_op& o)
{
    return o.f[1] >= 1.5f && o.f[1] <= 16.0f && o.f[2] >= 0.0f && o.f[2] <= 1000.0f && (o.iarg & 0xffffu) >= 1u;
}

// Whether a Mandelbulb's signs are decided early.  That saves part of every orbit, but the surface's
// corners and taps are evaluated afterwards, in waves that are not full and for orbits that take
// every iteration; else values are kept.  So it pays with many points to an iteration.  Early / kept,
// us, on the cube of edge 2.5: 8 iterations 128^3 90 / 85, 256^3 190 / 184, 640^3 1350 / 1450,
// 16 iterations 128^3 104 / 92, 256^3 250 / 229, 640^3 1710 / 1840, 60 iterations 128^3 180 / 134,
// 400^3 1228 / 1129, 640^3 3790 / 4090, 128 iterations 256^3 963 / 628.
bool sign_early(const s2m_op* ops, uint32_t n, uint64_t points)
{
    return mandel_power8(ops, n) && mandel_sign_ok(*ops) && points >= (uint64_t)(ops->iarg & 0xffffu) << 20;
}

dim3 sign_grid(const BrickArgs& a) { return dim3((a.nbx + a.run - 1u) / a.run, (a.nby + 3u) / 4u, a.nbz); }

// Bricks per wave of the sign kernel: runs of 16 share their coordinate loads, brick tests
// and store, but a slab gets at least four rounds of the device's 8192 waves, so that the
// last round (and runs whose bricks iterate longest) leaves little of it idle.  Measured
// over whole jobs, run 1 / 4 / 16: Mandelbulb 1024^3 in slabs of 680 K bricks 8.7 / 6.5 /
// 6.1 ms, 128^3 (43 K bricks) 136 / 134 / 151 us, the compiled estimator at 200^3 (157 K
// bricks) 1258 / 1249 / 1313 us.
// Long tapes take single bricks: their points cost so much that only the last round counts
// (CSG-64 at 256^3 2.14 -> 2.00 ms, without allocation at 512^3 50.0 -> 48.8; a 9-op tree at
// 256^3, 300 us, loses 15).
// Likewise the more iterations a Mandelbulb takes, the shorter its runs (60 iterations, exact corners:
// 256^3 1.68 ms with runs of 1, 2.14 of 16; 512^3 7.2, 6.3).
uint32_t sign_run(uint64_t bricks, const s2m_op* ops, uint32_t nops)
{
    if (nops >= 100u) return 1;
    const uint32_t iters = mandel_power8(ops, nops) ? ops->iarg & 0xffffu : 0u;
    uint32_t run = 16;
    while (run > 1u && bricks / run < 4u * 8192u * std::max(1u, iters / 8u)) run /= 2u;
    return run;
}

hipError_t launch_signs(hipStream_t s, const BrickArgs& a, const s2m_op* host_ops, const s2m_op* ops, uint32_t nops,
                        bool early)
{
    const dim3 grid = sign_grid(a);
    if (early) hipLaunchKernelGGL(k_signs<2>, grid, dim3(256), 0, s, a, ops, nops);
    else if (mandel_power8(host_ops, nops)) hipLaunchKernelGGL(k_signs<1>, grid, dim3(256), 0, s, a, ops, nops);
    else hipLaunchKernelGGL(k_signs<0>, grid, dim3(256), 0, s, a, ops, nops);
    return hipGetLastError();
}

hipError_t launch_contour(hipStream_t s, const BrickArgs& a, const s2m_op* op)
{
    if (op) hipLaunchKernelGGL(k_contour<false>, dim3(kBrickBlocks), dim3(256), 0, s, a, op);
    else hipLaunchKernelGGL(k_contour<true>, dim3(kBrickBlocks), dim3(256), 0, s, a, op);
    return hipGetLastError();
}

hipError_t launch_emit(hipStream_t s, const BrickArgs& a, const s2m_op* op)
{
    if (op) hipLaunchKernelGGL(k_emit<false>, dim3(kBrickBlocks), dim3(256), 0, s, a, op);
    else hipLaunchKernelGGL(k_emit<true>, dim3(kBrickBlocks), dim3(256), 0, s, a, op);
    return hipGetLastError();
}

hipError_t launch_normals(hipStream_t s, const s2m_op* host_ops, const s2m_op* ops, uint32_t nops, float eps,
                          const MeshBufs& b)
{
    const dim3 grid(kNormalBlocks);
    if (mandel_power8(host_ops, nops))
        hipLaunchKernelGGL(k_normals<true>, grid, dim3(256), 0, s, ops, nops, eps, b.vtx, b.counters, b.vcap);
    else
        hipLaunchKernelGGL(k_normals<false>, grid, dim3(256), 0, s, ops, nops, eps, b.vtx, b.counters, b.vcap);
    return hipGetLastError();
}

hipError_t launch_find_bricks(hipStream_t s, const BrickArgs& a)
{
    const uint64_t n = (uint64_t)a.ownx * a.owny * a.nbz;
    if (n > 0x7fffffffull) return hipErrorInvalidValue;
    const uint64_t per = kFindBricks * kBlock;
    hipLaunchKernelGGL(k_find_bricks, dim3((uint32_t)((n + per - 1u) / per)), dim3(kBlock), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_ranks(hipStream_t s, const MeshBufs& b, uint32_t ncells)
{
    const uint32_t nwords = (ncells + 63u) / 64u, chunks = (nwords + 16383u) / 16384u;
    if (chunks > kRankChunks || chunks == 0) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_ranks, dim3(chunks), dim3(1024), 0, s, b.actbits, nwords, const_cast<uint16_t*>(b.bits.wpre),
                       const_cast<uint32_t*>(b.bits.boffset), const_cast<uint32_t*>(b.bits.cbase), b.counters);
    return hipGetLastError();
}

hipError_t launch_cells_from_corners(hipStream_t s, const SlabArgs& a, const float* corners,
                                     const MeshBufs& b, int emit)
{
    const uint32_t nb = (a.ncells + kCellsPerBlock - 1) / kCellsPerBlock;
    if (nb == 0) return hipSuccess;
    if (emit) hipLaunchKernelGGL(k_cells<1>, dim3(nb), dim3(kBlock), 0, s, a, b, corners);
    else hipLaunchKernelGGL(k_cells<0>, dim3(nb), dim3(kBlock), 0, s, a, b, corners);
    return hipGetLastError();
}

hipError_t launch_sincos_check(hipStream_t s, uint64_t* cnt)
{
    hipLaunchKernelGGL(k_sincos_check, dim3(8192), dim3(256), 0, s, reinterpret_cast<unsigned long long*>(cnt));
    return hipGetLastError();
}

// One thread per op of a tape in device memory: a Mandelbulb op's f[3] (unused by the
// estimator's operands) gets bailout_threshold(f[1]), the r^2 bound of its power-8 step.
__global__ __launch_bounds__(256) void k_tape_prepare(s2m_op* __restrict__ ops, uint32_t n)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n && ops[i].code == S2M_OP_MANDELBULB) ops[i].f[3] = bailout_threshold(ops[i].f[1]);
}

hipError_t launch_tape_prepare(hipStream_t s, s2m_op* ops, uint32_t n)
{
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_tape_prepare, dim3((n + 255) / 256), dim3(256), 0, s, ops, n);
    return hipGetLastError();
}

hipError_t launch_bailout_check(hipStream_t s, uint64_t* cnt)
{
    hipLaunchKernelGGL(k_bailout_check, dim3(((1u << 20) + 256u) / 256u), dim3(256), 0, s,
                       reinterpret_cast<unsigned long long*>(cnt));
    return hipGetLastError();
}

// Before a job's first slab: its counters and the slab's activity bits cleared, and the
// axis tables (n16 16-byte words) copied from mapped host memory, where given: one kernel
// instead of a copy and memsets with gaps between them.
__global__ __launch_bounds__(256) void k_dense_begin(uint64_t* __restrict__ counters, uint32_t n,
                                                     uint64_t* __restrict__ words, uint32_t nwords,
                                                     const uint4* __restrict__ host_tables, uint4* __restrict__ tables,
                                                     uint32_t n16, uint32_t* __restrict__ cbase)
{
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x, stride = gridDim.x * blockDim.x;
    for (uint32_t i = t; i < n16; i += stride) tables[i] = host_tables[i];
    for (uint32_t i = t; i < n; i += stride) counters[i] = 0ull;
    if (t < kRankChunks) cbase[t] = 0u;
    for (uint32_t i = t; i < nwords; i += stride) words[i] = 0ull;
}

// After the quad pass of a slab that is not the last: the allocation counter (of parts:
// counters) reset, and the other activity words and chunk bases (the previous slab's, read for
// the last time by this slab's quads) set up for the next slab.
__global__ __launch_bounds__(256) void k_slab_end(uint64_t* __restrict__ counters, uint32_t ncounters,
                                                  uint64_t* __restrict__ words, uint32_t nwords,
                                                  uint32_t* __restrict__ cbase)
{
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    for (uint32_t i = kNumCounters + t; i < ncounters; i += gridDim.x * blockDim.x) counters[i] = 0ull;
    if (t < kRankChunks) cbase[t] = (uint32_t)counters[kVtxTotal];
    if (t == 0) {
        counters[kVtxPrev] = counters[kVtxTotal];
        counters[kBrickAlloc] = 0;
    }
    for (uint32_t i = t; i < nwords; i += gridDim.x * blockDim.x) words[i] = 0ull;
}

hipError_t launch_dense_begin(hipStream_t s, uint64_t* counters, uint32_t ncounters, uint64_t* words, uint32_t ncells,
                              const void* host_tables, void* tables, size_t bytes, uint32_t* cbase)
{
    const uint32_t n = (ncells + 63u) / 64u, n16 = (uint32_t)((bytes + 15u) / 16u);
    hipLaunchKernelGGL(k_dense_begin, dim3(std::max(1u, std::min((std::max(n, n16) + 255u) / 256u, 2048u))), dim3(256), 0,
                       s, counters, ncounters, words, n, static_cast<const uint4*>(host_tables),
                       static_cast<uint4*>(tables), n16, cbase);
    return hipGetLastError();
}

hipError_t launch_slab_end(hipStream_t s, uint64_t* counters, uint32_t ncounters, uint64_t* words, uint32_t ncells,
                           uint32_t* cbase)
{
    const uint32_t n = (ncells + 63u) / 64u;
    hipLaunchKernelGGL(k_slab_end, dim3(std::max(1u, std::min((n + 255u) / 256u, 2048u))), dim3(256), 0, s, counters,
                       ncounters, words, n, cbase);
    return hipGetLastError();
}

// Up to four arrays to page-locked host memory (16-byte words, then the last bytes): for
// small meshes one launch right after the job's last kernel in place of a DMA copy per
// array (each about 10 us beside its transfer).  Large ones go by DMA: a copying kernel
// reaches the same 55 GB/s but its queued stores hold up every other kernel's.
__global__ __launch_bounds__(256) void k_copy_out(CopyList c)
{
    const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x, step = (uint64_t)gridDim.x * blockDim.x;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const uint64_t n16 = c.bytes[k] >> 4, rest = c.bytes[k] & 15u;
        const uint4* s = static_cast<const uint4*>(c.src[k]);
        uint4* d = static_cast<uint4*>(c.dst[k]);
        for (uint64_t i = t; i < n16; i += step) d[i] = s[i];
        if (t < rest) reinterpret_cast<uint8_t*>(d + n16)[t] = reinterpret_cast<const uint8_t*>(s + n16)[t];
    }
}

hipError_t launch_copy_out(hipStream_t s, const CopyList& c)
{
    uint64_t most = 0;
    for (uint64_t b : c.bytes) most = std::max(most, b);
    if (most == 0) return hipSuccess;
    const uint32_t blocks = (uint32_t)std::min<uint64_t>((most / 16u + 255u) / 256u + 1u, 128u);
    hipLaunchKernelGGL(k_copy_out, dim3(blocks), dim3(256), 0, s, c);
    return hipGetLastError();
}

hipError_t launch_quads(hipStream_t s, const SlabArgs& a, const MeshBufs& b, const SlabBits& prev,
                        uint64_t* snap, uint64_t* back)
{
    if (a.ncells == 0) return hipSuccess;
    const uint32_t groups = (a.ncells + kBlock - 1u) / kBlock;  // if every cell had a vertex
    const dim3 grid(std::min(groups, 2048u));
    hipLaunchKernelGGL((k_quads<0>), grid, dim3(kBlock), 0, s, a, b, prev);
    hipLaunchKernelGGL(k_tri_offsets, dim3(1), dim3(1024), 0, s, b.tcount, b.toffset, b.counters, b.vcap, snap,
                       back);
    hipLaunchKernelGGL((k_quads<1>), grid, dim3(kBlock), 0, s, a, b, prev);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------
// Scratch of the no-allocation entry point (s2m_mesh_device_noalloc): one static device
// array per GPU that holds every working buffer of a dense job (coordinate tables, the
// slab's sign words, kept values, brick records and staged vertices, activity bits with
// their prefix tables, block counts and offsets, counters).  Host code never passes the array's name to a kernel or a copy (on the
// host it names a stand-in, not the device memory): it uses the address
// hipGetSymbolAddress returns for the device, taken once per device by noalloc_scratch.
// ---------------------------------------------------------------------------------
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

namespace {
std::mutex g_scratch_mu;
void* g_scratch_addr[kMaxDevices] = {};
hipError_t g_scratch_err[kMaxDevices] = {};
bool g_scratch_done[kMaxDevices] = {};
}  // namespace

hipError_t noalloc_scratch(int device, void** ptr)
{
    *ptr = nullptr;
    if (device < 0 || device >= (int)kMaxDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> g(g_scratch_mu);
    if (!g_scratch_done[device]) {
        int cur = -1;
        hipError_t e = hipGetDevice(&cur);
        if (e == hipSuccess && cur != device) e = hipErrorInvalidDevice;  // caller makes it current
        void* a = nullptr;
        if (e == hipSuccess) e = hipGetSymbolAddress(&a, HIP_SYMBOL(scratch));
        g_scratch_addr[device] = e == hipSuccess ? a : nullptr;
        g_scratch_err[device] = e;
        g_scratch_done[device] = true;
    }
    *ptr = g_scratch_addr[device];
    return g_scratch_err[device];
}

}  // namespace s2m
