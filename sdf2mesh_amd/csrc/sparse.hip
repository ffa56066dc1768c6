// sparse.hip - the tile-sparse meshing pipeline, for one job or a batch of jobs.
//
// Programs that interval pruning applies to (every library primitive and operator except
// the Mandelbulb, which is kept whole) are meshed tile by tile: cells are grouped in
// tiles of 8x8x8 and super-tiles of 4x4x4 tiles, and only tiles whose SDF can change sign
// are evaluated and contoured.  A pass covers the tiles of one slab of one job, or of
// every job of a batch (each job whole); tiles, super-tiles and row segments of the pass
// are numbered job after job.  In stream order:
//   k_sp_prune      exact interval pruning, one wave per super-tile: the job's program on
//                   the super-tile's padded box, then the super-tile's list on each of its
//                   tiles (one lane per tile); single-signed tiles are dropped, the others
//                   get a slot in a pool shared by all jobs (and a flag when their list is
//                   a left fold).  Also clears what the pass's later kernels count into.
//   k_sp_bricks     per slot, one lane per brick of 2x2x2 cells: interval bounds of a
//                   left fold on the brick (bricks that keep one sign are not evaluated),
//                   and the slot's record: header, live bricks, axis tables, box
//                   coordinates and the program in k_sp_tiles' LDS layout
//   k_sp_tiles      per slot (one block): the pruned program in LDS (left folds: from the
//                   record, read while the block contours the slot before), at the
//                   lattice points the tile's live bricks use (left folds) or at all
//                   points of its box (other programs; those too long to be staged in
//                   a large pass: a launch without operand stacks in LDS), into an LDS
//                   box; then the tile's cells: vertex and sign bits of each active cell,
//                   staged compactly, the slot's cell bits and each row segment's vertex
//                   count
//   k_sp_quadcount  per slot: valid quads of the staged cells (neighbour cells' bits),
//                   two triangles each, per row segment; invalid quads counted
//   k_sp_rowsum / k_sp_rowdown   offsets of the row segments in the reference's
//                   VertexList order (job after job, then z, y, tile x): per row, the
//                   segments of its active tiles; then a scan over rows, which also gives
//                   each job's first vertex and triangle index
//   k_sp_emit       per slot: the staged vertices at their ordered index with their
//                   4-tap normals (the tile's pruned program), then the triangles of
//                   their quads, vertex indices relative to the job's first vertex
//   k_sp_boundary   (multi-slab single job) cell -> vertex map of the slab's last plane
// The totals go to mapped host memory from k_sp_rowdown and k_sp_emit: a pass of folds is
// seven launches (of about 4.5 us each at any small size).
// The per-slot kernels are persistent (as many blocks as the device holds) and draw slots
// from a work queue.  A cell's vertex index is never stored: it is the first index of its row segment plus
// the number of cells with a vertex before it in the segment (the slot's cell bits).
// Loops over slots read their bound on the device: no host round trip inside a pass.
#include <algorithm>
#include <mutex>
#include <vector>

#include "device_bricks.h"
#include "device_interval.h"
#include "device_scan.h"
#include "device_sdf.h"
#include "device_staged.h"
#include "internal.h"

namespace s2m {

// threadIdx.x through an opaque copy: values derived from it are recomputed where they
// are used instead of being hoisted out of the kernels' slot loops and held in registers
// for the whole kernel (which costs occupancy).
__device__ __forceinline__ uint32_t thread_id()
{
    uint32_t t;
    asm volatile("v_mov_b32 %0, %1" : "=v"(t) : "v"((uint32_t)threadIdx.x));
    return t;
}

namespace {

__device__ __forceinline__ uint32_t lane() { return thread_id() & 63u; }

// Slots of the pass.  k_sp_rowdown moves the count from kSlotsUsed (zero when k_sp_prune
// starts) to kSlotsNow, where k_sp_emit reads it.
__device__ __forceinline__ uint32_t active_slots(const SpPass& P, uint32_t counter = kSlotsUsed)
{
    const uint64_t n = P.counters[counter];
    return (uint32_t)(n < P.slot_cap ? n : P.slot_cap);
}

// Work queues of a persistent launch: block b draws turns from the counter of its group g = b
// mod G, G = min(kQueueGroups, blocks), so blocks that draw cheap tiles take more of them.
// One counter per group, each on its own 128-byte line: updates of one address are serialised
// by the memory system (some 25 ns each), so a single counter for all blocks would throttle
// them.  A block's first turn is its own, without a draw.
// Neighbouring slots are mostly neighbouring tiles: runs of kTurnRun of them go to one XCD (the
// hardware deals blocks to XCDs in turn), so rows and output lines they share stay in one L2.
struct Turns {
    uint32_t* queue;
    uint32_t G, g, own, mine;  // own: blocks of the group

    __device__ Turns(const SpPass& P, uint32_t q, uint32_t block, uint32_t blocks)
    {
        G = min(kQueueGroups, blocks);
        g = block % G;
        own = (blocks - g + G - 1u) / G;
        queue = P.queues + (q * kQueueGroups + g) * 32u;
        mine = block / G;
    }
    __device__ __forceinline__ uint32_t first() const { return turn(mine); }
    // One lane's draw; turn(own + draw()) increases with every draw of the group.
    __device__ __forceinline__ uint32_t draw() const { return atomicAdd(queue, 1u); }
    __device__ __forceinline__ uint32_t drawn(uint32_t d) const { return turn(own + d); }
    // Turn j of group g: every index once.
    __device__ __forceinline__ uint32_t turn(uint32_t j) const
    {
        if (G != kQueueGroups) return j * G + g;
        const uint32_t m = j * (kQueueGroups / 8u) + (g >> 3);
        return ((m / kTurnRun) * 8u + (g & 7u)) * kTurnRun + m % kTurnRun;
    }
    static constexpr uint32_t kTurnRun = 16;
};

// Launches that run both kinds of slots (kBothKinds): the first blocks take the slots that are
// no folds, a share by their number and cost (a tile of them costs some two of a fold: every
// point of its box is evaluated).
constexpr uint32_t kGeneralCost = 2;
__device__ __forceinline__ uint32_t general_blocks(uint32_t general, uint32_t slots)
{
    if (general == 0) return 0;
    const uint64_t w = (uint64_t)kGeneralCost * general;
    const uint32_t n = (uint32_t)(gridDim.x * w / (w + (slots - min(slots, general))));
    return min(max(n, 1u), gridDim.x - 1u);
}

// Per-slot row data: array k (kRowVtx, kRowTri: counts; kRowVtxOff, kRowTriOff: first
// vertex / triangle of the row segment within its row) of slot `slot`, row r = (z % 8) * 8
// + y % 8 of the tile.
enum RowArray : uint32_t { kRowVtx = 0, kRowTri = 1, kRowVtxOff = 2, kRowTriOff = 3 };
__device__ __forceinline__ uint32_t* slot_row(const SpPass& P, uint32_t k, uint32_t slot)
{
    return P.slot_rows + ((size_t)k * P.slot_cap + slot) * 64u;
}

// Row (zl, y) of job J in the pass's row numbering (rows job after job, zl then y).
__device__ __forceinline__ size_t row_index(const SpJob& J, uint32_t zl, uint32_t y)
{
    return J.row_base + (size_t)zl * J.ry + y;
}

// Tile coordinates (tx, ty, tile layer within the pass) of pass tile `tile` of job J.
__device__ __forceinline__ void tile_xyz(const SpJob& J, uint64_t tile, uint32_t& tx, uint32_t& ty,
                                         uint32_t& tzl)
{
    const uint32_t t = (uint32_t)(tile - J.tile_base);
    tx = t % J.ntx;
    ty = (t / J.ntx) % J.nty;
    tzl = t / (J.ntx * J.nty);
}

// The slot of tile (tx, ty, tile layer tzl of the pass) of job J, -1 without one.
__device__ __forceinline__ int32_t slot_at(const SpPass& P, const SpJob& J, uint32_t tx, uint32_t ty, uint32_t tzl)
{
    static_assert(kSuper == 4, "64 tiles per super-tile");
    const SuperSlots S = P.super_act[J.super_base + ((uint64_t)(tzl >> 2) * J.nsy + (ty >> 2)) * J.nsx + (tx >> 2)];
    const uint32_t bit = ((tzl & 3u) * 4u + (ty & 3u)) * 4u + (tx & 3u);
    if (!((S.act >> bit) & 1ull)) return -1;
    return (int32_t)(S.first + (uint32_t)__builtin_popcountll(S.act & ((1ull << bit) - 1ull)));
}

// The pruned op indices of a slot.
__device__ __forceinline__ uint16_t* slot_list(const SpPass& P, uint32_t slot, uint64_t tile)
{
    return P.lists + (size_t)(P.lists_by_tile ? tile : slot) * P.list_stride;
}

// Existence bits of row r (= z % 8 * 8 + y % 8) of a tile with a slot: bit x % 8.
__device__ __forceinline__ uint32_t slot_row_bits(const SpPass& P, int32_t slot, uint32_t r)
{
    return (P.cellbits[(size_t)slot * 16u + (r >> 2)] >> ((r & 3u) * 8u)) & 0xffu;
}

// Cells (8 * tx - 1 + i, y, z), i = 0..8, of job J (z is the job's plane index, y and z
// may be -1; cells outside the grid have no vertex): bit i of the result is set iff the
// cell has a vertex.  INDEX: idx[i] = its pass-level vertex index, kNone if none (the
// first vertex of the row segment plus the cell's rank in it).  Plane z0 - 1 comes from
// the previous slab's boundary map.
// ns: the slots of the tile (tx, ty, tz) and of its look-back neighbours, ns[(dz * 2 + dy) * 2
// + dx] for tile (tx - dx, ty - dy, tz - dz) (k_sp_bricks), -1 without one.
template <bool INDEX>
__device__ uint32_t nb_row(const SpPass& P, const SpJob& J, uint32_t tx, uint32_t ty, uint32_t tz,
                           const int32_t (&ns)[8], int y, int z, uint32_t* idx)
{
    uint32_t bits = 0;
    if (INDEX)
        for (int i = 0; i < 9; ++i) idx[i] = kNone;
    if (y < 0 || z < 0 || (uint32_t)y >= J.ry || (uint32_t)z >= J.z0 + J.nz) return 0;
    if ((uint32_t)z < J.z0) {
        for (int i = 0; i < 9; ++i) {
            const int x = (int)(tx * 8u) + i - 1;
            if (x < 0 || (uint32_t)x >= J.rx) continue;
            const uint32_t v = J.boundary[(size_t)y * J.rx + (uint32_t)x];
            if (v != kNone) bits |= 1u << i;
            if (INDEX) idx[i] = v;
        }
        return bits;
    }
    const uint32_t zl = (uint32_t)z - J.z0;
    const uint32_t nsel = ((tz - ((uint32_t)z >> 3)) * 2u + (ty - ((uint32_t)y >> 3))) * 2u;
    const uint32_t r = ((uint32_t)z & 7u) * 8u + ((uint32_t)y & 7u);
    // the tile column's own cells and the cell before it; every load without a branch (slot 0
    // for a tile without one), so that they are in flight together
    const int32_t s0 = ns[nsel], s1 = ns[nsel + 1u];
    const int32_t a0 = max(s0, 0), a1 = max(s1, 0);
    uint32_t b0 = slot_row_bits(P, a0, r), b1 = slot_row_bits(P, a1, r);
    uint32_t f0 = 0, f1 = 0;
    if (INDEX) {
        const uint32_t row = P.row_off[row_index(J, zl, (uint32_t)y)];
        f0 = slot_row(P, kRowVtxOff, (uint32_t)a0)[r] + row;
        f1 = slot_row(P, kRowVtxOff, (uint32_t)a1)[r] + row;
    }
    b0 = s0 < 0 ? 0u : b0;
    b1 = s1 < 0 ? 0u : b1;
    bits = b0 << 1 | b1 >> 7;
    if (INDEX) {
        if (b1 & 0x80u) idx[0] = f1 + (uint32_t)__builtin_popcount(b1 & 0x7fu);
        for (uint32_t i = 0; i < 8; ++i)
            if ((b0 >> i) & 1u) idx[i + 1] = f0 + (uint32_t)__builtin_popcount(b0 & ((1u << i) - 1u));
    }
    return bits;
}

// Pass-level vertex index of cell (x, y, z) of job J (z is the job's plane index), kNone
// if it has no vertex.  Plane z0 - 1 comes from the previous slab's boundary map.
__device__ __forceinline__ uint32_t vertex_at(const SpPass& P, const SpJob& J, uint32_t x, uint32_t y,
                                              uint32_t z)
{
    if (z < J.z0) return J.boundary[(size_t)y * J.rx + x];
    const int32_t slot = slot_at(P, J, x >> 3, y >> 3, (z >> 3) - J.tz0);
    if (slot < 0) return kNone;
    const uint32_t b8 = slot_row_bits(P, slot, (z & 7u) * 8u + (y & 7u)), i = x & 7u;
    if (!((b8 >> i) & 1u)) return kNone;
    return slot_row(P, kRowVtxOff, (uint32_t)slot)[(z & 7u) * 8u + (y & 7u)] + P.row_off[row_index(J, z - J.z0, y)] +
           (uint32_t)__builtin_popcount(b8 & ((1u << i) - 1u));
}

// Exact pruning of postfix programs on boxes (device_interval.h).  The kept op indices
// are written in order; the interval of the result is `top` when the walk ends.  The top
// of the interval stack is kept in registers, deeper entries in LDS columns (entry d of
// lane l at [d * 64 + l]).
struct PruneStack {
    float* lo;         // [depth][64]
    float* hi;         // [depth][64]
    uint32_t* sum;     // [depth][64] PruneWalk::top_sum of the entry
    uint16_t* start;   // [depth][64]
    uint16_t* single;  // [depth][64] op index of a one-primitive subtree, else kComposite

    // LDS bytes of a stack of `depth` entries per lane, and its layout from `base`.
    static constexpr size_t bytes(uint32_t depth)
    {
        return (size_t)depth * 64u * (2 * sizeof(float) + sizeof(uint32_t) + 2 * sizeof(uint16_t));
    }
    __device__ static PruneStack at(float* base, uint32_t depth)
    {
        uint32_t* s32 = reinterpret_cast<uint32_t*>(base + 128u * depth);
        uint16_t* s16 = reinterpret_cast<uint16_t*>(s32 + 64u * depth);
        return PruneStack{base, base + 64u * depth, s32, s16, s16 + 64u * depth};
    }
};

constexpr uint32_t kComposite = 0xffffu;
constexpr uint32_t kFoldBit = 0x80000000u;  // PruneWalk sums: the subtree's list is a left fold

// A tile's list while it is walked, in LDS: lane ln's entry k.  (A walk reads entries back when
// it drops or turns a subtree; from global memory each such step waits for the memory.)
struct LdsList {
    uint16_t* p;
    uint32_t ln;
    __device__ __forceinline__ uint16_t& operator[](uint32_t k) const { return p[k * 64u + ln]; }
};

// kTurn: an operator between a primitive and a longer fold is written as a fold too, the
// fold first, then the primitive, then the operator marked kSwapped (union and
// intersection need no mark): any tree whose operators each keep a primitive operand
// becomes a left fold, which the tile kernels run without an operand stack.
template <bool kTurn>
struct PruneWalk {
    Iv top = iv_unknown();
    uint32_t top_start = 0, depth = 0, len = 0;  // depth: entries below `top`
    uint32_t top_single = kComposite;  // op index when `top` is one primitive
    // flops of the kept ops of the top subtree (op_flops), | kFoldBit when its list is a left
    // fold of library primitives (a primitive other than the Mandelbulb, or a left fold,
    // such a primitive and an operator): the tile's flops and left-fold flag without reading
    // its list back
    uint32_t top_sum = 0;

    // The primitive with op index i, interval v (q: its position in the program; sum: its
    // flops | kFoldBit unless it is a Mandelbulb).
    template <class List>
    __device__ __forceinline__ void prim(uint32_t q, uint32_t i, const Iv& v, const List& out, const PruneStack& S,
                                         uint32_t ln, uint32_t sum = 0)
    {
        if (q != 0) {  // push the previous top
            S.lo[depth * 64u + ln] = top.lo;
            S.hi[depth * 64u + ln] = top.hi;
            S.sum[depth * 64u + ln] = top_sum;
            S.start[depth * 64u + ln] = (uint16_t)top_start;
            S.single[depth * 64u + ln] = (uint16_t)top_single;
            ++depth;
        }
        top = v;
        top_start = len;
        top_single = i;
        top_sum = sum;
        out[len++] = (uint16_t)i;
    }

    // Operator i (code, smoothing radius k, flops fl) on the two topmost values.
    template <class List>
    __device__ __forceinline__ void op(uint32_t i, uint32_t code, float k, const List& out, const PruneStack& S,
                                       uint32_t ln, uint32_t fl = 0)
    {
        const Iv B = top;
        const uint32_t sB = top_start;
        --depth;
        const float alo = S.lo[depth * 64u + ln], ahi = S.hi[depth * 64u + ln];
        const Iv A{alo, ahi, alo > -kHuge};  // iv_make / iv_unknown: known iff lo > -kHuge
        const uint32_t sA = S.start[depth * 64u + ln], singleA = S.single[depth * 64u + ln];
        const uint32_t sumA = S.sum[depth * 64u + ln];
        int keep;
        const Iv r = iv_op(code, A, B, k, keep);
        if (keep == kKeepBoth) {
            bool fold = (sumA & kFoldBit) && top_single != kComposite && (top_sum & kFoldBit);
            uint32_t mark = 0;
            if (kTurn && !fold && (sumA & kFoldBit) && singleA != kComposite && (top_sum & kFoldBit)) {
                for (uint32_t j = sB; j < len; ++j) out[j - 1u] = out[j];  // A is the one entry before B
                out[len - 1u] = (uint16_t)singleA;
                mark = code == S2M_OP_UNION || code == S2M_OP_INTERSECTION ? 0u : kSwapped;
                fold = true;
            }
            out[len++] = (uint16_t)(i | mark);
            top_sum = ((sumA & ~kFoldBit) + (top_sum & ~kFoldBit) + fl) | (fold ? kFoldBit : 0u);
            top = r;
            top_single = kComposite;
        } else if (keep == kKeepA) {
            len = sB;  // drop B's subtree and the operator
            top = A;
            top_single = singleA;
            top_sum = sumA;
        } else {       // drop A's subtree and the operator
            if (top_single != kComposite) {  // B is one primitive: no read-back of the list
                out[sA] = (uint16_t)top_single;
                len = sA + 1;
            } else {
                const uint32_t nb = len - sB;
                for (uint32_t j = 0; j < nb; ++j) out[sA + j] = out[sB + j];
                len = sA + nb;
            }
            top = B;
        }
        top_start = sA;
    }

    __device__ __forceinline__ bool one_sign() const { return top.known && (top.lo > 0.0f || top.hi < 0.0f); }
};

// PruneWalk for a left fold (P0 P1 op1 P2 op2 ..., at most kStageOps ops): the same decisions and
// sums with the accumulated value and the latest primitive in registers instead of the LDS
// stack (every operator's left operand is the accumulated value), and the kept primitives
// (each with the operator behind it) as a bit mask in place of a list, bit (q + 1) / 2 for the
// primitive at position q; the list is written once the tile has a slot.
struct FoldMask {
    Iv top = iv_unknown();
    uint64_t kept = 0;
    uint32_t top_sum = 0;
    Iv b = iv_unknown();
    uint32_t b_sum = 0;

    __device__ __forceinline__ void prim(uint32_t q, const Iv& v, uint32_t sum)
    {
        static_assert(kStageOps <= 128, "one bit per primitive");
        if (q == 0) {
            top = v;
            top_sum = sum;
            kept = 1ull;
        } else {
            b = v;
            b_sum = sum;
        }
    }

    // The operator at position q >= 2.
    __device__ __forceinline__ void op(uint32_t q, uint32_t code, float k, uint32_t fl)
    {
        int keep;
        const Iv r = iv_op(code, top, b, k, keep);
        const uint64_t bit = 1ull << (q >> 1);
        if (keep == kKeepBoth) {
            kept |= bit;
            const bool fold = (top_sum & kFoldBit) && (b_sum & kFoldBit);
            top_sum = ((top_sum & ~kFoldBit) + (b_sum & ~kFoldBit) + fl) | (fold ? kFoldBit : 0u);
            top = r;
        } else if (keep != kKeepA) {  // the list is the primitive
            kept = bit;
            top = b;
            top_sum = b_sum;
        }
    }

    __device__ __forceinline__ uint32_t len() const { return 2u * (uint32_t)__builtin_popcountll(kept) - 1u; }
    __device__ __forceinline__ bool one_sign() const { return top.known && (top.lo > 0.0f || top.hi < 0.0f); }
};

__device__ __forceinline__ uint32_t job_of(const SpPass& P, uint64_t index, bool super)
{
    uint32_t lo = 0, hi = P.njobs - 1;  // last job whose first tile (super-tile) <= index
    while (lo < hi) {
        const uint32_t mid = (lo + hi + 1) / 2;
        if ((super ? P.jobs[mid].super_base : P.jobs[mid].tile_base) <= index) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

}  // namespace

// Padded box of the tiles [t0, t1] (per axis, t1 inclusive; z: tile layers of the job).  The
// pad is 1.25 times what the taps and roundings of a vertex need (J.pad), which covers the
// rounding of the box itself: a quarter of 1e-6 (1 + max |coordinate|) is four half ulps.
__device__ __forceinline__ void tiles_box(const SpJob& J, const uint32_t t0[3], const uint32_t t1[3], float bl[3],
                                          float bh[3])
{
    const float pad = 1.25f * (float)J.pad;
    const float* e[3] = {J.ext, J.ext + 2 * J.ntx, J.ext + 2 * J.ntx + 2 * J.nty};
    const uint32_t n[3] = {J.ntx, J.nty, J.ntz};
    for (int a = 0; a < 3; ++a) {  // (an axis may run from its maximum to its minimum)
        bl[a] = fminf(e[a][t0[a]], e[a][t1[a]]) - pad;
        bh[a] = fmaxf(e[a][n[a] + t0[a]], e[a][n[a] + t1[a]]) + pad;
    }
}

// Tiles of super-tile s of job J: first and last tile per axis (z: tile layer of the job).
__device__ __forceinline__ void super_tiles(const SpJob& J, uint64_t s, uint32_t t0[3], uint32_t t1[3])
{
    const uint32_t t = (uint32_t)(s - J.super_base);
    const uint32_t sx = t % J.nsx, sy = (t / J.nsx) % J.nsy, szl = t / (J.nsx * J.nsy);
    const uint32_t layers = (J.nz + kTile - 1) / kTile;  // tile layers of this pass
    t0[0] = sx * kSuper;
    t1[0] = min(t0[0] + kSuper, J.ntx) - 1;
    t0[1] = sy * kSuper;
    t1[1] = min(t0[1] + kSuper, J.nty) - 1;
    t0[2] = J.tz0 + szl * kSuper;
    t1[2] = J.tz0 + min(szl * kSuper + kSuper, layers) - 1;
}

// ---------------------------------------------------------------------------------
// k_sp_prune, one wave per super-tile (one launch: three or four of these steps as kernels
// of their own cost more in launches and list traffic than in work):
//  1. the super-tile's list: the job's program exactly pruned on its padded box, or
//     kSingleSign when the SDF keeps one sign there.  Left folds of unions: prune_fold, a
//     lane per op.  Other programs: a lane per primitive for its interval on the box
//     (prim_intervals), then a lane per op up and down the tree (prune_levels); of more than
//     kStageOps ops: every lane walks the program in order (walk_super).
//  2. lane l = its tile (l % 4, l / 4 % 4, l / 16): the list pruned on the tile's padded box
//     (every lane walks the same list: wave-uniform op dispatch).  Tiles that keep one sign
//     are dropped, the others get a slot in the pool shared by all jobs (and a flag when
//     their list is a left fold).
// Dynamic LDS: the prune stack (P.prune_depth entries per lane), then P.walk_ops list entries
// per lane for the tiles' walks of programs that are no left folds.  Lists and intervals of
// programs of at most kStageOps ops live in LDS, of longer ones in lists, super_lists and
// super_iv.
// ---------------------------------------------------------------------------------

// prune_fold: the super-tile list of a program that is a left fold of unions and smooth
// unions (P0 P1 op1 P2 op2 ..., op in {UNION, SMOOTH_UNION with k > 0}), without a
// sequential walk: lane q evaluates op q's interval, and primitive P_m (m >= 1) is dropped
// with its operator when
//     lo(P_m) >= U_{m-1} + k_m + slack,   U_{m-1} = min over j < m of hi(P_j),
// a prefix minimum over the lanes.  The accumulated value after m - 1 steps never exceeds
// min_j p_j by more than the rounding of its fp32 operations (smooth union <= min of its
// operands), which the slack bounds: kMargin (64 ulps) x the magnitude of every step so
// far, each bounded by |p_j| + k_j + max_i |p_i| + sum_i k_i / 4 (|acc| never exceeds the
// last two terms); so p_m >= acc + k_m everywhere on the box, h = 1 and
// the operator returns acc bit for bit (union: p_m >= acc returns acc).  Dropping never
// changes acc, so later bounds stay valid.  The super-tile keeps one sign when
// min_j hi(P_j) + slack < 0 (acc < 0), or when min over the kept P_j of lo(P_j) - the kept
// smooth radii / 4 - slack > 0 (smooth union >= min of its operands - k / 4).
__device__ __forceinline__ uint32_t prune_fold(const SpJob& J, const float* bl, const float* bh, uint32_t ln,
                                               uint16_t* out)
{
    const s2m_op* ops = J.ops;
    const uint32_t nops = J.nops;
    float carry_u = kHuge;    // min hi(P_j) over the primitives so far
    float carry_mag = 0.0f;    // sum of |P_j| + k_j over the primitives so far
    float carry_max = 0.0f;    // max of |P_j| + k_j so far
    float carry_ka = 0.0f;     // sum of k_j / 4 so far
    float carry_cnt = 0.0f;    // primitives so far
    float carry_lo = kHuge;   // min lo(P_j) over the kept primitives
    float carry_k4 = 0.0f;     // sum of the kept smooth radii / 4
    uint32_t nkept = 0;
    bool prev_kept = true;     // was the last primitive of the previous chunk kept?
    for (uint32_t c0 = 0; c0 < nops; c0 += 64u) {
        const uint32_t q = c0 + ln;
        const bool valid = q < nops;
        const bool prim = valid && (q == 0 || (q & 1u));  // a left fold: P0, then P_m at odd q
        // the operator after primitive q (q >= 1) and its smoothing radius
        float kk = 0.0f;
        if (prim && q >= 1 && ops[q + 1].code == S2M_OP_SMOOTH_UNION) kk = ops[q + 1].f[0];
        Iv B = iv_unknown();
        if (prim) B = iv_primitive(ops[q].code, ops[q].f, bl, bh);
        const float mag = prim ? fmaxf(fabsf(B.lo), fabsf(B.hi)) + kk : 0.0f;
        // prefix scans over the lanes (inclusive): min hi, sum and max of the magnitudes,
        // sum of k / 4, count of primitives
        const float u_in = wave_min(prim ? B.hi : kHuge, kHuge);
        float m_in = wave_sum(mag), x_in = wave_max(mag, 0.0f), ka_in = wave_sum(0.25f * kk);
        float c_in = (float)__builtin_popcountll(__ballot(prim) & ((2ull << ln) - 1ull));
        float u_ex = lane_below(u_in, kHuge);
        u_ex = fminf(u_ex, carry_u);
        m_in += carry_mag;
        x_in = fmaxf(x_in, carry_max);
        ka_in += carry_ka;
        c_in += carry_cnt;
        const float slack = kMargin * (m_in + c_in * (x_in + ka_in));
        const float tiny = kUlps * (fabsf(u_ex) + fabsf(B.lo) + fabsf(B.hi) + kk);
        const bool drop = prim && q >= 1 && B.known && u_ex < kHuge && B.lo >= u_ex + kk + tiny + slack;
        // an operator (even q >= 2) is kept with its primitive q - 1
        const uint64_t pk = __ballot(prim && !drop);
        const bool prev_prim_kept = ln == 0 ? prev_kept : ((pk >> (ln - 1)) & 1ull) != 0;
        const bool kept = valid && (prim ? !drop : prev_prim_kept);
        const uint64_t km = __ballot(kept);
        if (kept) out[nkept + (uint32_t)__builtin_popcountll(km & ((1ull << ln) - 1ull))] = (uint16_t)q;
        nkept += (uint32_t)__builtin_popcountll(km);
        // one-sign bounds over the kept primitives
        carry_lo = fminf(carry_lo, last_lane(wave_min((prim && !drop) ? B.lo : kHuge, kHuge)));
        carry_k4 += last_lane(wave_sum((prim && !drop) ? 0.25f * kk : 0.0f));
        carry_u = fminf(carry_u, last_lane(u_in));
        carry_mag = last_lane(m_in);
        carry_max = last_lane(x_in);
        carry_ka = last_lane(ka_in);
        carry_cnt = last_lane(c_in);
        // the chunk's last primitive: at the highest odd q of the chunk (q = c0 + 63 when
        // the chunk is full; 64 is even, so lane 63 is odd)
        const uint32_t last = min(nops - c0, 64u) - 1u;
        const uint32_t lastp = (c0 + last) & 1u ? last : (last ? last - 1u : 0u);
        prev_kept = ((pk >> lastp) & 1ull) != 0;
    }
    const float slack = kMargin * (carry_mag + carry_cnt * (carry_max + carry_ka));
    const bool one_sign = (carry_u + slack < 0.0f) || (carry_lo > -kHuge && carry_lo - carry_k4 - slack > 0.0f);
    return one_sign ? kSingleSign : nkept;
}

// The intervals of the job's primitives on the box, a lane per op.
__device__ __forceinline__ void prim_intervals(const SpJob& J, const float* bl, const float* bh, uint32_t ln, float2* iv)
{
    for (uint32_t q = ln; q < J.nops; q += 64u) {
        const s2m_op& o = J.ops[q];
        const uint32_t code = o.code;
        if (code >= S2M_OP_UNION) continue;
        const Iv v = iv_primitive(code, o.f, bl, bh);
        iv[q] = make_float2(v.lo, v.hi);
    }
}

// The super-tile's list of a program of at most kStageOps ops from its primitives' intervals: a
// lane per op, level by level up the tree (an op when its operands are done), then down it for
// the ops no operator above has dropped.  A walk in the program's order takes some 700 cycles
// per op; a tree of 39 ops has six to eight levels.  `alive`: a word per op.
__device__ __forceinline__ uint32_t prune_levels(const SpJob& J, float2* iv, uint32_t* alive, uint32_t ln, uint16_t* out)
{
    static_assert(kStageOps <= 128, "two ops per lane");
    const uint32_t n = J.nops, levels = J.levels;
    const uint32_t* tree = J.op_flops + n;
    uint32_t code[2] = {0, 0}, place[2] = {0, 0};
    float k[2] = {0.0f, 0.0f};
    int keep[2] = {kKeepBoth, kKeepBoth};
#pragma unroll
    for (uint32_t s = 0; s < 2; ++s) {
        const uint32_t q = ln + 64u * s;
        if (q >= n) continue;
        code[s] = J.ops[q].code;
        k[s] = J.ops[q].f[0];
        place[s] = tree[q];
        alive[q] = q + 1u == n ? 1u : 0u;
    }
    __syncthreads();  // the intervals are visible
    for (uint32_t h = 1; h <= levels; ++h) {
#pragma unroll
        for (uint32_t s = 0; s < 2; ++s) {
            if (place[s] >> 16 != h) continue;
            const uint32_t q = ln + 64u * s;
            const float2 a = iv[place[s] & 0xffffu], b = iv[q - 1u];  // known iff lo > -kHuge
            const Iv r = iv_op(code[s], Iv{a.x, a.y, a.x > -kHuge}, Iv{b.x, b.y, b.x > -kHuge}, k[s], keep[s]);
            iv[q] = make_float2(r.lo, r.hi);
        }
        __syncthreads();
    }
    for (uint32_t h = levels; h >= 1; --h) {
#pragma unroll
        for (uint32_t s = 0; s < 2; ++s) {
            const uint32_t q = ln + 64u * s;
            if (place[s] >> 16 != h || !alive[q]) continue;
            alive[place[s] & 0xffffu] = keep[s] != kKeepB;
            alive[q - 1u] = keep[s] != kKeepA;
        }
        __syncthreads();
    }
    uint32_t len = 0;
#pragma unroll
    for (uint32_t s = 0; s < 2; ++s) {
        const uint32_t q = ln + 64u * s;
        const bool in = q < n && alive[q] && keep[s] == kKeepBoth;
        const uint64_t w = __ballot(in);
        if (in) out[len + (uint32_t)__builtin_popcountll(w & ((1ull << ln) - 1ull))] = (uint16_t)q;
        len += (uint32_t)__builtin_popcountll(w);
    }
    const float2 top = iv[n - 1u];
    return top.x > -kHuge && (top.x > 0.0f || top.y < 0.0f) ? kSingleSign : len;
}

// A longer program walked in order on those intervals; every lane takes the same steps and
// writes the same list.
__device__ __forceinline__ uint32_t walk_super(const SpJob& J, const float2* iv, const PruneStack& S, uint32_t ln,
                                               uint16_t* out)
{
    PruneWalk<false> w;  // the tiles' walks take its list in the program's order
    for (uint32_t q = 0; q < J.nops; ++q) {
        const uint32_t code = __builtin_amdgcn_readfirstlane(J.ops[q].code);
        if (code < S2M_OP_UNION) {
            const float2 v = iv[q];
            w.prim(q, q, Iv{v.x, v.y, v.x > -kHuge}, out, S, ln);  // known iff lo > -kHuge
        } else {
            w.op(q, code, J.ops[q].f[0], out, S, ln);
        }
    }
    return w.one_sign() ? kSingleSign : w.len;
}

// What the pass's later kernels count into, cleared (by all blocks): the job rows and
// counters of a job's first pass (for a later pass the totals so far become its first
// indices), work queues with the statistics beside them, chunk sums, and before a
// multi-pass job the boundary plane (no vertex carried yet).  kSlotsUsed, kGenUsed and
// kStageUsed, which this kernel and the tile kernels count, are zero already (k_sp_rowdown).
__device__ __forceinline__ void clear_pass(const SpPass& P)
{
    const uint32_t t = blockIdx.x * 64u + (thread_id() & 63u), step = gridDim.x * 64u;
    for (uint32_t i = t; i < P.nclear; i += step)
        if (i != kSlotsUsed && i != kStageUsed && i != kGenUsed) P.counters[i] = 0;
    if (P.nclear == 0 && t == 0) {
        P.counters[kVtxPrev] = P.counters[kVtxTotal];
        P.counters[kTriPrev] = P.counters[kTriTotal];
    }
    constexpr uint32_t kLines = kQueues * kQueueGroups;
    for (uint32_t i = t; i < kLines; i += step) P.queues[i * 32u] = 0;
    if (P.nclear)  // the statistics are the whole job's
        for (uint32_t i = t; i < 3u * kQueueGroups; i += step)
            reinterpret_cast<uint64_t*>(P.queues)[(i % kQueueGroups) * 16u + 1u + i / kQueueGroups] = 0;
    for (uint32_t i = t; i < P.nbsum; i += step) P.bsum[i * kChunkSumStride] = 0;
    for (uint32_t i = t; i < P.nbnd; i += step) P.jobs[0].boundary[i] = kNone;
}

__global__ __launch_bounds__(64) void k_sp_prune(SpPass P)
{
    extern __shared__ float prune_lds[];
    __shared__ StagedTape T;          // the super-tile's list (at most kStageOps ops)
    __shared__ uint16_t idx[kStageOps];  // op index of each staged op
    __shared__ uint32_t sums[kStageOps];  // its flops | kFoldBit for primitives other than the Mandelbulb
    static_assert(sizeof T.f >= kStageOps * sizeof(float2), "intervals share the staged operands' space");
    clear_pass(P);
    const uint32_t D = P.prune_depth, ln = thread_id() & 63u;
    const PruneStack S = PruneStack::at(prune_lds, D);
    const uint64_t s = blockIdx.x;
    const uint32_t jid = __builtin_amdgcn_readfirstlane(job_of(P, s, true));
    const SpJob& J = P.jobs[jid];
    const bool small = J.nops <= kStageOps;
    uint16_t* in = small ? idx : P.super_lists + s * P.list_stride;
    uint32_t t0[3], t1[3];
    super_tiles(J, s, t0, t1);
    uint32_t sl;
    {
        float bl[3], bh[3];
        tiles_box(J, t0, t1, bl, bh);
        if (J.union_fold) {
            sl = prune_fold(J, bl, bh, ln, in);
        } else {
            float2* iv = small ? reinterpret_cast<float2*>(T.f) : P.super_iv + s * P.list_stride;
            prim_intervals(J, bl, bh, ln, iv);
            if (small) {
                sl = prune_levels(J, iv, sums, ln, in);
            } else {
                __syncthreads();  // visible to all lanes
                sl = walk_super(J, iv, S, ln, in);
            }
        }
        sl = __builtin_amdgcn_readfirstlane(sl);
    }
    __syncthreads();  // the list is visible
    const uint32_t tx = t0[0] + (ln & 3u), ty = t0[1] + ((ln >> 2) & 3u), tz = t0[2] + (ln >> 4);
    const bool valid = tx <= t1[0] && ty <= t1[1] && tz <= t1[2];
    const uint64_t tile = J.tile_base + ((uint64_t)(tz - J.tz0) * J.nty + ty) * J.ntx + tx;
    const s2m_op* ops = J.ops;
    const bool staged = sl != kSingleSign && sl <= kStageOps;
    auto op_sum = [&](uint32_t i) {
        const uint32_t c = ops[i].code;
        return J.op_flops[i] | (c < S2M_OP_UNION && c != S2M_OP_MANDELBULB ? kFoldBit : 0u);
    };
    if (staged) {
        stage_tape(T, ops, in, sl);
        for (uint32_t k = ln; k < sl; k += 64u) {
            const uint32_t i = in[k];
            if (!small) idx[k] = (uint16_t)i;
            sums[k] = op_sum(i);
        }
    }
    __syncthreads();
    bool surface = false;
    uint32_t lens = 0, flops = 0;
    uint64_t kept = 0;  // the tile's list of a staged fold (FoldMask)
    const LdsList list{reinterpret_cast<uint16_t*>(reinterpret_cast<char*>(prune_lds) + PruneStack::bytes(D)), ln};
    const bool in_lds = !J.left_fold && J.nops <= P.walk_ops;
    if (valid && sl != kSingleSign) {
        const uint32_t tt[3] = {tx, ty, tz};
        float bl[3], bh[3];
        tiles_box(J, tt, tt, bl, bh);
        auto done = [&](bool one_sign, uint32_t len, uint32_t sum) {
            // the pruned program is one subtree: its flops and whether it is a left fold
            surface = !one_sign;
            lens = len | (surface && (sum & kFoldBit) && len <= kStageOps ? kLinearFlag : 0u);
            flops = sum & ~kFoldBit;
        };
        auto walk = [&](auto& w, auto L) {
            if (staged) {  // every lane walks the same list: wave-uniform dispatch
                for (uint32_t q = 0; q < sl; ++q) {
                    const uint32_t code = uniform_code(T, q), i = idx[q], sum = sums[q];
                    if (code < S2M_OP_UNION) w.prim(q, i, iv_primitive(code, T.f[q], bl, bh), L, S, ln, sum);
                    else w.op(i, code, T.f[q][0], L, S, ln, sum);
                }
            } else {
                for (uint32_t q = 0; q < sl; ++q) {
                    const uint32_t i = __builtin_amdgcn_readfirstlane(in[q]);
                    const uint32_t code = ops[i].code, sum = op_sum(i);
                    if (code < S2M_OP_UNION) w.prim(q, i, iv_primitive(code, ops[i].f, bl, bh), L, S, ln, sum);
                    else w.op(i, code, ops[i].f[0], L, S, ln, sum);
                }
            }
            done(w.one_sign(), w.len, w.top_sum);
        };
        if (J.left_fold) {  // the super-tile's list is a left fold too, and staged
            FoldMask w;
            for (uint32_t q = 0; q < sl; ++q) {
                const uint32_t code = uniform_code(T, q), sum = sums[q];
                if (code < S2M_OP_UNION) w.prim(q, iv_primitive(code, T.f[q], bl, bh), sum);
                else w.op(q, code, T.f[q][0], sum);
            }
            done(w.one_sign(), w.len(), w.top_sum);
            kept = w.kept;
        } else if (in_lds) {
            PruneWalk<true> w;
            walk(w, list);
        } else {
            PruneWalk<true> w;
            walk(w, P.lists + (size_t)tile * P.list_stride);
        }
    }
    // slots for the surviving tiles: one counter update per wave.  (Some 25 ns each, but fewer of
    // them cost more than they gain: 92 us at CSG-64 1024^3, 98 with four super-tiles per block
    // and update, the block waiting for its slowest wave, 107 with two per wave in turn.)
    const uint64_t m = __ballot(surface);
    uint64_t wbase = 0;
    if (ln == 0 && m) wbase = atomicAdd((unsigned long long*)&P.counters[kSlotsUsed], (unsigned long long)__builtin_popcountll(m));
    wbase = __shfl(wbase, 0, 64);
    int32_t slot = -1;
    if (surface) {
        const uint64_t sidx = wbase + (uint64_t)__builtin_popcountll(m & ((1ull << ln) - 1ull));
        if (sidx < P.slot_cap) {
            slot = (int32_t)sidx;
            P.slot_info[sidx] = make_uint4((uint32_t)tile, jid, lens, flops);
            uint16_t* L = slot_list(P, (uint32_t)sidx, tile);
            uint32_t k = 0;
            for (; kept; kept &= kept - 1ull) {
                const uint32_t q = 2u * (uint32_t)__builtin_ctzll(kept);
                if (k) {  // the primitive at q - 1 and its operator
                    L[k] = idx[q - 1u];
                    L[k + 1] = idx[q];
                    k += 2;
                } else {
                    L[k++] = idx[q ? q - 1u : 0u];
                }
            }
            if (in_lds)
                for (uint32_t q = 0; q < (lens & ~kLinearFlag); ++q) L[q] = list[q];
        }
    }
    // the slots that are no folds, listed for the kernels that run them
    const uint64_t g = __ballot(slot >= 0 && !(lens & kLinearFlag));
    if (g) {
        uint64_t gbase = 0;
        if (ln == 0) gbase = atomicAdd((unsigned long long*)&P.counters[kGenUsed], (unsigned long long)__builtin_popcountll(g));
        gbase = __shfl(gbase, 0, 64);
        if ((g >> ln) & 1ull) P.gen_slots[gbase + (uint64_t)__builtin_popcountll(g & ((1ull << ln) - 1ull))] = (uint32_t)slot;
    }
    const uint64_t act = __ballot(slot >= 0);  // bit l: tile l of the super-tile has a slot
    if (ln == 0) P.super_act[s] = SuperSlots{act, (uint32_t)wbase, 0u};
}

// Per-axis corner tables of a tile's 8 cells: box-relative lattice index and coordinate
// of each cell's lo / hi corner.
struct TileAxes {
    uint8_t lo[3][8], hi[3][8];  // box indices (< 16)
    float clo[3][8], chi[3][8];
};

// Entry e (< 24) of A: axis e / 8, cell e % 8.  Cells past the end of the grid repeat the
// last cell's entries (their cells are never contoured).
__device__ __forceinline__ void load_tile_axes(TileAxes& A, const SpJob& J, uint32_t tx, uint32_t ty,
                                               uint32_t tz, uint32_t e)
{
    const uint32_t ax = e >> 3, c = e & 7u;
    const uint32_t t = ax == 0 ? tx : ax == 1 ? ty : tz;
    const uint32_t r = ax == 0 ? J.rx : ax == 1 ? J.ry : J.z0 + J.nz;  // cells on the axis
    const uint32_t* lo = ax == 0 ? J.lox : ax == 1 ? J.loy : J.loz;
    const uint32_t* hi = ax == 0 ? J.hix : ax == 1 ? J.hiy : J.hiz;
    const float* co = ax == 0 ? J.cx : ax == 1 ? J.cy : J.cz;
    const uint32_t org = J.ibox[2 * (ax == 0 ? 0 : ax == 1 ? J.ntx : J.ntx + J.nty) + t];
    const uint32_t g = t * 8u + c;   // cell index along the axis (z: of the job)
    const uint32_t gi = g < r ? g : r - 1;
    A.lo[ax][c] = lo[gi] - org;
    A.hi[ax][c] = hi[gi] - org;
    A.clo[ax][c] = co[lo[gi]];
    A.chi[ax][c] = co[hi[gi]];
}

// Per slot, written by k_sp_bricks: what k_sp_tiles<1> stages for the slot, in its LDS
// layout, so that one read of the record (made while the block contours the slot before)
// replaces the dependent loads of header, job, pruned list, ops, axis tables and
// coordinates.  Header and live bricks are written for every slot, the rest for slots
// whose program is a left fold.
struct alignas(16) TileRec {
    SlotHdr H;
    uint64_t live;              // bricks (2x2x2 cells) that may hold an active cell
    uint16_t xb[4];             // per x-brick: the box x indices its cells use (bit mask)
    TileAxes A;
    uint8_t bm[2][16];          // per box y (z) index: the y (z) bricks whose cells use it
    float pc[3][16];            // lattice coordinates of the box per axis
    StagedFold T;               // the pruned program (the used rows are read)
};
static_assert(sizeof(TileRec) == kTileRecBytes, "record size shared with the host");
constexpr uint32_t kRecVec = kTileRecBytes / 16;   // 16-byte words per record
constexpr uint32_t kRecPre = 64;                    // words read ahead: header .. codes, ops 0..22
constexpr uint32_t kRecRowsAt = (uint32_t)offsetof(TileRec, T) + (uint32_t)offsetof(StagedFold, f);
static_assert(kRecRowsAt + 32u * 12u <= 16u * kRecPre, "ops 0..22 are read ahead");
struct TileGen {  // k_sp_tiles<0>: the same parts, staged per slot
    StagedTape T;
    TileAxes A;
    float pc[3][16];
    uint32_t mandel;  // the program holds a Mandelbulb
};
struct TileLong {  // k_sp_tiles<3>
    TileAxes A;
    float pc[3][16];
};

// ---------------------------------------------------------------------------------
// n / d for n < 2^16 and d <= 256, r = recip(d): (n + 0.5) / d is at least 1 / (2 d) from an
// integer, and its error (three roundings of one ulp) below (n + 1) / d * 2^-21.
__device__ __forceinline__ float recip(uint32_t d) { return __builtin_amdgcn_rcpf((float)d); }
__device__ __forceinline__ uint32_t div_by(uint32_t n, float r) { return (uint32_t)(((float)n + 0.5f) * r); }

// ---------------------------------------------------------------------------------
// Bricks: the 4x4x4 blocks of 2x2x2 cells of a tile, brick (bx, by, bz) = bit
// (bz * 4 + by) * 4 + bx of its record's `live`.  Per slot (one 64-lane block
// iteration, lane = brick): interval bounds of the tile's program on the brick's lattice
// points; a brick whose values provably keep one sign holds no active cell, so its cells
// are not contoured and its points are not evaluated.  Left-fold programs only (other
// programs keep every brick).
// ---------------------------------------------------------------------------------
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(5, 8))) void k_sp_bricks(SpPass P)
{
    __shared__ StagedFold T;
    __shared__ TileAxes A;
    const uint32_t nslots = active_slots(P);
    // The slots' tile, job and list length are read two slots ahead with per-lane loads,
    // which barriers do not wait for.
    const uint32_t z = thread_id() & 0u;  // a per-lane zero: vector loads
    const uint32_t G = gridDim.x;
    uint4 i1 = make_uint4(0u, 0u, 0u, 0u), i2 = i1;
    if (blockIdx.x < nslots) i1 = P.slot_info[blockIdx.x + z];
    if (blockIdx.x + G < nslots) i2 = P.slot_info[blockIdx.x + G + z];
    for (uint32_t slot = blockIdx.x; slot < nslots; slot += G) {
        const uint32_t b = thread_id();
        const uint64_t tile = __builtin_amdgcn_readfirstlane(i1.x);
        const uint32_t lens = __builtin_amdgcn_readfirstlane(i1.z);
        const uint32_t n = lens & ~kLinearFlag;
        const uint32_t jid = __builtin_amdgcn_readfirstlane(i1.y);
        i1 = i2;
        if (slot + 2u * G < nslots) i2 = P.slot_info[slot + 2u * G + z];
        const SpJob& J = P.jobs[jid];
        uint32_t tx, ty, tzl;
        tile_xyz(J, tile, tx, ty, tzl);
        TileRec& RG = *reinterpret_cast<TileRec*>(P.slot_rec + (size_t)slot * kRecVec);
        if (b < 48) {  // the slot's header (lane a < 3: axis a's box origin and size) and coordinates
            const uint32_t a = b >> 4, i = b & 15u, t = a == 0 ? tx : a == 1 ? ty : J.tz0 + tzl;
            const uint32_t nt = a == 0 ? J.ntx : a == 1 ? J.nty : J.ntz;
            const uint32_t* ib = J.ibox + 2 * (a == 0 ? 0 : a == 1 ? J.ntx : J.ntx + J.nty);
            const uint32_t o = ib[t], e = ib[nt + t];
            const bool linear = (lens & kLinearFlag) && n <= kStageOps;
            if (linear && i <= e - o) RG.pc[a][i] = (a == 0 ? J.cx : a == 1 ? J.cy : J.cz)[o + i];
            if (i == 0) {
                const uint32_t box = o | ((e - o + 1) << 24);
                P.slot_hdr[slot].box[a] = box;
                RG.H.box[a] = box;
            }
            if (b == 0) {
                SlotHdr H;
                H.tile = (uint32_t)tile;
                H.job = jid;
                H.lens = lens;
                H.txy = tx | (ty << 16);
                H.tzl = tzl;
                for (SlotHdr* d : {&P.slot_hdr[slot], &RG.H}) {
                    d->tile = H.tile;
                    d->job = H.job;
                    d->lens = H.lens;
                    d->txy = H.txy;
                    d->tzl = H.tzl;
                }
            }
        }
        if (b >= 48 && b < 56) {  // the slot's look-back neighbours (nb_row): (tx - dx, ty - dy, tzl - dz)
            const uint32_t i = b - 48u, dx = i & 1u, dy = (i >> 1) & 1u, dz = i >> 2;
            int32_t ns = -1;
            if (tx >= dx && ty >= dy && tzl >= dz)
                ns = slot_at(P, J, tx - dx, ty - dy, tzl - dz);
            P.slot_nb[(size_t)slot * 8u + i] = ns;
        }
        if (!(lens & kLinearFlag) || n > kStageOps) {  // every brick is kept
            if (b == 0) RG.live = ~0ull;
            continue;
        }
        __syncthreads();  // the previous slot's readers of T and A are done
        stage_tape(T, J.ops, slot_list(P, slot, tile), n);
        if (b < 24) load_tile_axes(A, J, tx, ty, J.tz0 + tzl, b);
        __syncthreads();
        {  // the record's axes and program (codes and the rows in use)
            const uint32_t words = (uint32_t)(offsetof(StagedFold, f) + 32u * ((n + 1u) >> 1)) / 4u;
            for (uint32_t k = b; k < words; k += 64u)
                reinterpret_cast<uint32_t*>(&RG.T)[k] = reinterpret_cast<const uint32_t*>(&T)[k];
            for (uint32_t k = b; k < (uint32_t)sizeof(TileAxes) / 4u; k += 64u)
                reinterpret_cast<uint32_t*>(&RG.A)[k] = reinterpret_cast<const uint32_t*>(&A)[k];
            if (b < 4) {
                const uint32_t c = 2u * b;
                RG.xb[b] = (uint16_t)((1u << A.lo[0][c]) | (1u << A.hi[0][c]) | (1u << A.lo[0][c + 1]) |
                                      (1u << A.hi[0][c + 1]));
            } else if (b >= 32) {  // lane 32 + 16 (a - 1) + i: axis a (y, z), box index i
                const uint32_t a = 1u + ((b - 32u) >> 4), i = b & 15u;
                uint32_t m = 0;
                for (uint32_t c = 0; c < 8u; ++c)
                    if (A.lo[a][c] == i || A.hi[a][c] == i) m |= 1u << (c >> 1);
                RG.bm[a - 1u][i] = (uint8_t)m;
            }
        }
        // brick b: cells c, c + 1 per axis, from the first cell's lo corner to the second's hi
        // corner (which lies below it on an axis that runs from its maximum to its minimum)
        const uint32_t c[3] = {(b & 3u) * 2u, ((b >> 2) & 3u) * 2u, (b >> 4) * 2u};
        float bl[3], bh[3];
        for (int a = 0; a < 3; ++a) {
            const float lo = A.clo[a][c[a]], hi = A.chi[a][c[a] + 1];
            bl[a] = fminf(lo, hi);
            bh[a] = fmaxf(lo, hi);
        }
        Iv acc = iv_primitive(uniform_code(T, 0), T.f_at(0), bl, bh);
        for (uint32_t k = 1; k + 1 < n; k += 2) {
            const Iv d = iv_primitive(uniform_code(T, k), T.f_at(k), bl, bh);
            int keep;
            const uint32_t code = uniform_code(T, k + 1);
            if (code & kSwapCode) acc = iv_op(code & ~kSwapCode, d, acc, T.f_at(k + 1)[0], keep);
            else acc = iv_op(code, acc, d, T.f_at(k + 1)[0], keep);
        }
        const bool may_cross = !(acc.known && (acc.lo > 0.0f || acc.hi < 0.0f));
        const uint64_t m = __ballot(may_cross);
        if (b == 0) RG.live = m;
    }
}

// ---------------------------------------------------------------------------------
// The cells of one tile (all threads of the block; the tile's box values in LDS), in
// three steps: the cells whose 8 corners change sign are listed (cells of bricks outside
// `live` are skipped: their corner values keep one sign and were not evaluated); each
// listed cell gets its vertex (dualcontour.wgsl:72-131) and sign bits (:57-69); the
// cells with a vertex are staged compactly for k_sp_emit, their bits go to the slot's
// `cellbits` and each row segment's count to the slot's kRowVtx row.  Contains barriers.
// ---------------------------------------------------------------------------------
// Staged cells are allocated in chunks of kStageChunk per block: the block's own, then one
// counter update per chunk (with the first ones counted too, the blocks of a launch wait for
// each other's update of one address: up to 15 us of a launch of 1792).  A slot needs room for
// 8 entries per live brick (its cells) when its tile starts, so that its cells are contiguous,
// and takes what it has used; a chunk with less room left is abandoned.  Hence at most (staged
// cells) + (room needed by the slots that open a chunk) + blocks x kStageChunk are used; the
// host grows the buffer from the device count if that exceeds it.
constexpr uint32_t kStageChunk = kStageChunkHost;
// Threads of a k_sp_tiles block (one tile at a time).  128 would share a tile's fixed work
// among fewer waves, but then half of the waves fit (the box of the worst tile, 16^3 points,
// and the rest take 21 KB of LDS: seven blocks per compute unit either way): 318 against 300 us
// at CSG-64 1024^3, 201 against 153 at 512^3 (before the first chunks were the blocks' own).
constexpr uint32_t kTileThreads = 256;
static_assert(kRecVec - kRecPre <= kTileThreads, "one thread per record word past the read-ahead");
constexpr int kGeneralPoints = 4;       // (k_sp_tiles<0>: a box of up to 1024 points in one round,
constexpr uint32_t kWideDepth = 8;      // their operand stacks within 32 KB of LDS; deeper ones
                                        // take one point at a time)

struct ContourLds {  // block-shared state of contour_tile (and `cand`, 512 entries: the cells
                     // with a sign change among their corners)
    uint32_t rows[64];   // row czl * 8 + cyl: bit cxl = the cell has a vertex
    uint32_t ncand, nact;
    uint32_t base, left, slot_base;  // staging chunk of the block
};

// Reset for the next tile (thread_id() < 64; a barrier must follow before contour_tile).
__device__ __forceinline__ void contour_reset(ContourLds& L)
{
    if (thread_id() < 64) L.rows[thread_id()] = 0;
    if (thread_id() == 0) L.ncand = L.nact = 0;
}

// Thread 0: staging space for the slot's cells with a vertex, at most `cells` (8 per live
// brick), from the block's chunk; published by the barriers before contour_tile, which takes
// what the slot has used from the chunk.
__device__ __forceinline__ void contour_reserve(const SpPass& P, ContourLds& L, uint32_t cells)
{
    if (L.left < cells) {
        L.base = 2u * P.tile_blocks * kStageChunk +
                 (uint32_t)atomicAdd((unsigned long long*)&P.counters[kStageUsed], (unsigned long long)kStageChunk);
        L.left = kStageChunk;
    }
    L.slot_base = L.base + (kStageChunk - L.left);
}

__device__ __forceinline__ void tile_corners(const float* box, const TileAxes& A, uint32_t bx, uint32_t by,
                                             uint32_t c, float cv[8])
{
    const uint32_t cxl = c & 7u, cyl = (c >> 3) & 7u, czl = c >> 6;
    const uint32_t xi[2] = {A.lo[0][cxl], A.hi[0][cxl]};
    const uint32_t yi[2] = {A.lo[1][cyl], A.hi[1][cyl]};
    const uint32_t zi[2] = {A.lo[2][czl], A.hi[2][czl]};
#pragma unroll
    for (int k = 0; k < 8; ++k) cv[k] = box[(zi[(k >> 2) & 1] * by + yi[(k >> 1) & 1]) * bx + xi[k & 1]];
}

// The job's extents as wave-uniform values, read once per tile: the job table sits in
// global memory that the kernel also writes, so the compiler re-reads fields of a
// reference to it inside every loop.
struct TileGrid {
    uint32_t rx, ry, nz;  // cells per axis of the job's grid (nz: of this pass)
    uint32_t bx, by;      // box strides
};

__device__ __forceinline__ TileGrid tile_grid(const SpJob& J)
{
    TileGrid G;
    G.rx = __builtin_amdgcn_readfirstlane(J.rx);
    G.ry = __builtin_amdgcn_readfirstlane(J.ry);
    G.nz = __builtin_amdgcn_readfirstlane(J.nz);
    G.bx = __builtin_amdgcn_readfirstlane(J.bx);
    G.by = __builtin_amdgcn_readfirstlane(J.by);
    return G;
}

__device__ __forceinline__ void contour_tile(const SpPass& P, const TileGrid& G, uint32_t slot, uint32_t tx,
                                             uint32_t ty, uint32_t tzl, const float* box, const TileAxes& A,
                                             uint32_t nlive, const uint8_t* lb, uint16_t* cand, ContourLds& L)
{
    // 1. cells with a sign change: the 8 cells of each live brick (lb: the live bricks,
    // nlive of them), one per thread
    const uint32_t wave = __builtin_amdgcn_readfirstlane(thread_id() >> 6) * 64u;
    for (uint32_t k0 = wave; k0 < nlive * 8u; k0 += kTileThreads) {
        const uint32_t k = k0 + lane();
        uint32_t c = 0;
        bool cand_c = false;
        if (k < nlive * 8u) {
            const uint32_t b = lb[k >> 3], j = k & 7u;  // brick (x fastest), cell within it
            const uint32_t cxl = (b & 3u) * 2u + (j & 1u), cyl = ((b >> 2) & 3u) * 2u + ((j >> 1) & 1u);
            const uint32_t czl = (b >> 4) * 2u + (j >> 2);
            c = (czl * 8u + cyl) * 8u + cxl;
            if (tx * 8u + cxl < G.rx && ty * 8u + cyl < G.ry && tzl * 8u + czl < G.nz) {
                float cv[8];
                tile_corners(box, A, G.bx, G.by, c, cv);
                uint32_t pm = 0;
#pragma unroll
                for (int i = 0; i < 8; ++i) pm |= (uint32_t)(cv[i] > 0.0f) << i;
                cand_c = pm != 0u && pm != 0xffu;
            }
        }
        const uint64_t w = __ballot(cand_c);
        const uint32_t lead = (uint32_t)__builtin_ctzll(w | (1ull << 63));
        uint32_t wbase = 0;
        if (w && lane() == lead) wbase = atomicAdd(&L.ncand, (uint32_t)__builtin_popcountll(w));
        wbase = (uint32_t)__builtin_amdgcn_readlane((int)wbase, (int)lead);
        if (cand_c) cand[wbase + (uint32_t)__builtin_popcountll(w & ((1ull << lane()) - 1ull))] = (uint16_t)c;
    }
    __syncthreads();
    // 2. vertex and sign bits of each listed cell, staged at the space reserved by
    // contour_reserve
    const uint32_t ncand = L.ncand, stage_base = L.slot_base;
    for (uint32_t k0 = wave; k0 < ncand; k0 += kTileThreads) {
        const uint32_t k = k0 + lane();
        bool act = false;
        float pos[3];
        uint32_t c = 0, sg = 0;
        if (k < ncand) {
            c = cand[k];
            const uint32_t cxl = c & 7u, cyl = (c >> 3) & 7u, czl = c >> 6;
            float cv[8];
            tile_corners(box, A, G.bx, G.by, c, cv);
            const float lo[3] = {A.clo[0][cxl], A.clo[1][cyl], A.clo[2][czl]};
            const float hi[3] = {A.chi[0][cxl], A.chi[1][cyl], A.chi[2][czl]};
            act = contour_cell(cv, lo, hi, pos);
            // cell_sign_changes (dualcontour.wgsl:57-69)
            sg = (uint32_t)(cv[1] > 0.0f) | ((uint32_t)(cv[2] > 0.0f) << 1) | ((uint32_t)(cv[4] > 0.0f) << 2) |
                 ((uint32_t)(cv[0] > 0.0f) << 3);
        }
        const uint64_t w = __ballot(act);
        if (!w) continue;
        const uint32_t lead = (uint32_t)__builtin_ctzll(w);
        uint32_t wbase = 0;
        if (lane() == lead) wbase = atomicAdd(&L.nact, (uint32_t)__builtin_popcountll(w));
        wbase = (uint32_t)__builtin_amdgcn_readlane((int)wbase, (int)lead);
        if (act) {
            atomicOr(&L.rows[c >> 3], 1u << (c & 7u));
            const uint64_t at = (uint64_t)stage_base + wbase + (uint32_t)__builtin_popcountll(w & ((1ull << lane()) - 1ull));
            if (at < P.stage_cap) P.stage[at] = make_float4(pos[0], pos[1], pos[2], __uint_as_float(c | (sg << 12)));
        }
    }
    __syncthreads();
    // 3. row segment counts and the slot's cell bits
    if (thread_id() == 0) {
        P.slot_stage[2 * slot] = stage_base;
        P.slot_stage[2 * slot + 1] = L.nact;
        L.left -= L.nact;
    }
    if (thread_id() < 64) {
        const uint32_t row = thread_id();
        slot_row(P, kRowVtx, slot)[row] = (uint32_t)__builtin_popcount(L.rows[row]);  // 0 outside the grid
        if (row < 16)
            P.cellbits[(size_t)slot * 16u + row] = L.rows[4 * row] | (L.rows[4 * row + 1] << 8) |
                                                   (L.rows[4 * row + 2] << 16) | (L.rows[4 * row + 3] << 24);
    }
}

constexpr uint32_t kList = 1024;   // needed points held before they are evaluated
constexpr uint32_t kBoxAxis = 16;  // most lattice indices of a tile box per axis
static_assert(kList >= 8 * 8 * 8, "the point list doubles as the contour's candidate cells");
static_assert(kTileThreads >= kBoxAxis * kBoxAxis, "one box row per thread");

// Kinds of slots a launch runs: those that are no folds, folds, or both, each by a share of the
// blocks.  Two launches leave most of the device idle while a small pass's few slots of the
// one kind run, each some 15 to 30 us of latency; in one launch the folds are held to the
// registers of the other kind (four waves per SIMD instead of seven), which costs more than it
// saves from some 130 k tiles on.  Three trees, one launch against two, us: 160^3 182 / 222,
// 256^3 168 / 195, 352^3 249 / 273, 384^3 279 / 287, 448^3 297 / 298, 640^3 478 / 441.
// Slots whose program is too long to be staged have a launch of their own from some 2 k tiles on,
// without the operand stacks in LDS (32 KB and more beside the box: three blocks per compute
// unit instead of seven), and no other kinds share a launch then.  One launch for all against one
// for each, us: a 599-op fold at 64^3 3120 / 3360, 128^3 2800 / 2720, 256^3 2810 / 2150, 512^3
// 13,700 / 5600; a 511-op tree 3830 / 3900, 4700 / 4300, 3980 / 3920, 33,400 / 22,100.
enum Kind : int { kGeneralKind = 0, kFoldKind = 1, kBothKinds = 2, kLongKind = 3 };
constexpr uint64_t kBothTiles = 128u << 10, kBothTilesLong = 2u << 10;

// k_sp_tiles: per slot (persistent, slots drawn from a work queue), the tile's pruned
// program, staged in
// LDS, at the lattice points of its closed box that the tile's cells need (all points for
// programs that are not left folds), into an LDS box; then the tile's cells are contoured
// from it (contour_tile).  KIND (below) selects the slots: left folds (the others are skipped),
// the others (gen_slots) whose program is staged, or those whose program is longer and read
// from memory.
// Bound by instruction issue (three quarters of the issue slots at CSG-64 1024^3: 69.5 k slots,
// 258 points and 57 vertices each): of 277 us there, 60 evaluate, 42 place vertices, 28 look for
// sign changes, the rest is the fixed work of a tile.  355 us with the points dealt to all
// lanes, half of them twice, and a 64-bit division per row; 300 with every block's first
// staging chunk counted (512^3: 166, 151, now 136).
template <int KIND>
__device__ __forceinline__ void tiles_body(const SpPass& P, uint32_t block, uint32_t blocks)
{
    constexpr bool LINEAR = KIND == kFoldKind, LONG = KIND == kLongKind;
    extern __shared__ float box[];  // P.box_stride floats; kGeneralKind: then the operand stacks
                                    // (P.prune_depth entries per thread and point)
    // left folds: the slot's record (k_sp_bricks); other programs: staged here
    __shared__ std::conditional_t<LINEAR, TileRec, std::conditional_t<LONG, TileLong, TileGen>> R;
    // points to evaluate; then the contour's candidate cells (contour_tile's `cand`)
    __shared__ uint16_t list[LINEAR ? kList : 8 * 8 * 8];
    __shared__ uint32_t nlist;
    __shared__ ContourLds L;
    __shared__ uint32_t sh_slot, sh_next;
    __shared__ uint8_t lb[64];  // the live bricks of the slot (contour_tile)
    // other programs: indices into the list of the slots that are no folds
    const uint32_t nslots = active_slots(P, LINEAR ? kSlotsUsed : kGenUsed);
    constexpr uint32_t kQueue = LINEAR ? 0u : LONG ? 4u : 1u;
    if (thread_id() == 0) {  // the block's first staging chunk; published by the first slot's barriers
        L.base = (block + (LINEAR ? 0u : P.tile_blocks)) * kStageChunk;
        L.left = LONG ? 0u : kStageChunk;  // (long programs' first chunks are counted)
    }
    uint64_t tiles_done = 0, points_done = 0, flops_done = 0;  // thread 0: this block's share
    const Turns Q(P, kQueue, block, blocks);
    uint32_t next = Q.first();  // thread 0's counts
    // Left folds: threads < kRecPre hold the first kRecPre x 16 bytes of the next slot's
    // record, read while the current slot is contoured and stored to R at the loop's top.
    uint4 pre = make_uint4(0u, 0u, 0u, 0u);
    auto prefetch = [&]() {  // all threads; `next` published in sh_next before a barrier
        const uint32_t s = sh_next;
        if (thread_id() < kRecPre && s < nslots) pre = P.slot_rec[(size_t)s * kRecVec + thread_id()];
    };
    if constexpr (LINEAR) {
        if (thread_id() == 0) nlist = 0;
        if (thread_id() == 0) sh_next = next;
        __syncthreads();
        prefetch();
    }
    for (;;) {
        __syncthreads();  // the previous slot's readers of sh_slot, R, list, box, L are done
        if (thread_id() == 0) sh_slot = next;
        if (LINEAR && thread_id() < kRecPre) reinterpret_cast<uint4*>(&R)[thread_id()] = pre;
        __syncthreads();
        if (sh_slot >= nslots) break;
        const uint32_t slot = LINEAR ? sh_slot : P.gen_slots[sh_slot];
        if (thread_id() == 0) next = Q.drawn(Q.draw());  // prefetched
        const SlotHdr& H = [&]() -> const SlotHdr& {
            if constexpr (LINEAR) return R.H;
            else return P.slot_hdr[__builtin_amdgcn_readfirstlane(slot)];
        }();
        const uint32_t lens = __builtin_amdgcn_readfirstlane(H.lens);
        auto skip = [&]() {  // to the next slot (left folds: its record is read first)
            if (LINEAR) {
                if (thread_id() == 0) sh_next = next;
                __syncthreads();
                prefetch();
            }
        };
        if (((lens & kLinearFlag) != 0) != LINEAR || (!LINEAR && P.long_apart && (lens > kStageOps) != LONG)) {  // same for the block
            skip();
            continue;
        }
        const uint64_t tile = __builtin_amdgcn_readfirstlane(H.tile);
        // thread 0's flop count for the block statistics, read now so that the load has
        // landed when the tile ends
        const uint32_t tile_flops = thread_id() == 0 ? P.slot_info[slot].w : 0u;
        const uint32_t n = lens & ~kLinearFlag;
        const SpJob& J = P.jobs[__builtin_amdgcn_readfirstlane(H.job)];
        const uint32_t txy = __builtin_amdgcn_readfirstlane(H.txy);
        const uint32_t tx = txy & 0xffffu, ty = txy >> 16, tzl = __builtin_amdgcn_readfirstlane(H.tzl);
        const uint32_t bxh = __builtin_amdgcn_readfirstlane(H.box[0]), byh = __builtin_amdgcn_readfirstlane(H.box[1]);
        const uint32_t bzh = __builtin_amdgcn_readfirstlane(H.box[2]);
        const uint32_t nx = bxh >> 24, ny = byh >> 24, nz = bzh >> 24;
        const TileGrid G = tile_grid(J);
        const uint32_t bx = G.bx, by = G.by;
        const uint16_t* Lst = slot_list(P, slot, tile);
        uint64_t lv = ~0ull;
        uint32_t evaluated = 0;
        contour_reset(L);
        if constexpr (LINEAR) {
            lv = R.live;
            if (lv == 0) {  // no brick can hold an active cell: empty rows, no cell bits
                if (thread_id() < 64) slot_row(P, kRowVtx, slot)[thread_id()] = 0;
                if (thread_id() < 16) P.cellbits[(size_t)slot * 16u + thread_id()] = 0;
                if (thread_id() == 0) {
                    P.slot_stage[2 * slot] = 0;
                    P.slot_stage[2 * slot + 1] = 0;
                    tiles_done += 1;
                }
                skip();
                continue;
            }
            // the rest of a long program's record (rows past the prefetched part): loaded
            // now, stored to R once the point list is built (nothing before reads it)
            const uint32_t need = (kRecRowsAt + 32u * ((n + 1u) >> 1) + 15u) >> 4;
            const uint32_t kr = kRecPre + thread_id();
            uint4 rest = make_uint4(0u, 0u, 0u, 0u);
            if (kr < need) rest = P.slot_rec[(size_t)slot * kRecVec + kr];
            // The points that some live brick uses.  Per box row (iz, iy): the x-bricks of the
            // live bricks whose cells use it (rm), hence the row's needed x positions (the
            // union of those x-bricks' positions, xb).  One row per thread; each wave reserves
            // its rows' points in `list` with one atomic; entries are iz << 10 | iy << 5 | ix.
            // The list is evaluated window by window (one window unless more than kList points).
            if (thread_id() == 0) contour_reserve(P, L, 8u * (uint32_t)__builtin_popcountll(lv));
            const uint32_t nrow = ny * nz;
            const float rny = recip(ny);
            uint32_t M = 0, code = 0, off = 0, cnt = 0;
            if ((thread_id() & ~63u) < nrow) {  // the wave has rows
                const uint32_t q = thread_id();
                if (q < nrow) {
                    const uint32_t iz = div_by(q, rny), iy = q - iz * ny;
                    // rm = OR over the z-bricks bz and y-bricks by that use the row of the live
                    // bits of x-bricks (bz, by, 0..3): the used z layers of lv ORed (16 bits,
                    // by * 4 + bx), then the used y rows of that
                    const uint32_t mz = R.bm[1][iz], my = R.bm[0][iy];
                    uint32_t layers = 0, rm = 0;
#pragma unroll
                    for (uint32_t bz = 0; bz < 4; ++bz)
                        if ((mz >> bz) & 1u) layers |= (uint32_t)(lv >> (16u * bz)) & 0xffffu;
#pragma unroll
                    for (uint32_t by = 0; by < 4; ++by)
                        if ((my >> by) & 1u) rm |= (layers >> (4u * by)) & 0xfu;
                    M = ((rm & 1u) ? R.xb[0] : 0u) | ((rm & 2u) ? R.xb[1] : 0u) | ((rm & 4u) ? R.xb[2] : 0u) |
                           ((rm & 8u) ? R.xb[3] : 0u);
                    code = (iz << 10) | (iy << 5);
                }
                // the exclusive prefix sum of cnt (<= 16, 5 bits) over the wave's lanes, bit by
                // bit: lanes below with the bit set (mbcnt over its ballot) times its weight
                cnt = (uint32_t)__builtin_popcount(M);
                uint32_t below = 0, wtotal = 0;
#pragma unroll
                for (uint32_t b = 0; b < 5; ++b) {
                    const uint64_t m = __ballot((int)((cnt >> b) & 1u));
                    below += __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u)) << b;
                    wtotal += (uint32_t)__builtin_popcountll(m) << b;
                }
                uint32_t wbase = 0;
                if (lane() == 0 && wtotal) wbase = atomicAdd(&nlist, wtotal);
                off = (uint32_t)__builtin_amdgcn_readlane((int)wbase, 0) + below;
            }
            if (kr < need) reinterpret_cast<uint4*>(&R)[kr] = rest;
            // window 0 is filled at once (every wave has its offsets); the total is read
            // after the barrier that completes it
            uint32_t total = 0;
            for (uint32_t w0 = 0;; w0 += kList) {
                if (w0) __syncthreads();  // the previous window's readers of the list are done
                if (off < w0 + kList && off + cnt > w0) {
                    // the row's k-th needed x position at off + k, over the box's x positions
                    // (a loop that is the same for every lane)
                    const uint32_t at0 = off - w0;  // wraps below w0: skipped by the bound test
                    for (uint32_t b = 0; b < nx; ++b) {
                        const uint32_t at = at0 + (uint32_t)__builtin_popcount(M & ((1u << b) - 1u));
                        if (((M >> b) & 1u) && at < kList) list[at] = (uint16_t)(code | b);
                    }
                }
                __syncthreads();
                if (w0 == 0) total = nlist;  // reset for the next slot after the box is complete
                const uint32_t m = min(kList, total - w0);
                // a wave takes 128 points in a row, two per lane sharing each op's decode, or the
                // last 64 or fewer one per lane: whole waves have nothing left, instead of
                // every lane half of its points
                auto points = [&](auto np, uint32_t i0) {
                    constexpr int NP = decltype(np)::value;
                    float x[NP], y[NP], z[NP], v[NP];
                    uint32_t at[NP];
#pragma unroll
                    for (int p = 0; p < NP; ++p) {
                        const uint32_t e = list[min(i0 + p * 64u + lane(), m - 1u)];
                        const uint32_t ix = e & 31u, iy = (e >> 5) & 31u, iz = e >> 10;
                        x[p] = R.pc[0][ix];
                        y[p] = R.pc[1][iy];
                        z[p] = R.pc[2][iz];
                        at[p] = (iz * by + iy) * bx + ix;
                    }
                    run_linear<NP>(R.T, n, x, y, z, v);
#pragma unroll
                    for (int p = 0; p < NP; ++p)
                        if (i0 + p * 64u + lane() < m) box[at[p]] = v[p];
                };
                for (uint32_t i0 = __builtin_amdgcn_readfirstlane(thread_id() >> 6) * 128u; i0 < m; i0 += 2u * kTileThreads) {
                    if (m - i0 > 64u) points(std::integral_constant<int, 2>{}, i0);
                    else points(std::integral_constant<int, 1>{}, i0);
                }
                if (w0 + kList >= total) break;
            }
            evaluated = total;
            if (thread_id() == 0) sh_next = next;
        } else {
            const uint32_t x0 = bxh & 0xffffffu, y0 = byh & 0xffffffu, z0 = bzh & 0xffffffu;
            const uint32_t nxy = nx * ny, npts = nxy * nz;
            const float rx = recip(nx), rxy = recip(nxy);
            if (thread_id() == 0) contour_reserve(P, L, 8u * 8u * 8u);
            const bool staged = !LONG && n <= kStageOps;
            if constexpr (!LONG)
                if (staged) stage_tape(R.T, J.ops, Lst, n);
            if (thread_id() < 24) load_tile_axes(R.A, J, tx, ty, J.tz0 + tzl, thread_id());
            if (thread_id() < 48) {
                const uint32_t a = thread_id() >> 4, i = thread_id() & 15u;
                const float* c = a == 0 ? J.cx + x0 : a == 1 ? J.cy + y0 : J.cz + z0;
                if (i < (a == 0 ? nx : a == 1 ? ny : nz)) R.pc[a][i] = c[i];
            }
            if constexpr (!LONG) {
                if (thread_id() == 0) R.mandel = 0;
                __syncthreads();
                for (uint32_t q = thread_id(); staged && q < n; q += kTileThreads)
                    if (R.T.code[q] == S2M_OP_MANDELBULB) R.mandel = 1;
            }
            __syncthreads();
            auto point = [&](uint32_t q, float& x, float& y, float& z) {  // its entry in the box
                const uint32_t iz = div_by(q, rxy), r = q - iz * nxy;
                const uint32_t iy = div_by(r, rx), ix = r - iy * nx;
                x = R.pc[0][ix];
                y = R.pc[1][iy];
                z = R.pc[2][iz];
                return (iz * by + iy) * bx + ix;
            };
            if (!staged) {
                for (uint32_t q = thread_id(); q < npts; q += kTileThreads) {
                    float x, y, z;
                    const uint32_t at = point(q, x, y, z);
                    box[at] = tape_eval_list(J.ops, Lst, n, x, y, z);
                }
            }
            if constexpr (!LONG) {
                float* stack = box + P.box_stride + thread_id();
                if (staged && !R.mandel && P.prune_depth <= kWideDepth) {
                    for (uint32_t q0 = thread_id(); q0 < npts; q0 += kGeneralPoints * kTileThreads) {
                        float x[kGeneralPoints], y[kGeneralPoints], z[kGeneralPoints], v[kGeneralPoints];
                        uint32_t at[kGeneralPoints];
#pragma unroll
                        for (int p = 0; p < kGeneralPoints; ++p) {
                            const uint32_t q = q0 + p * kTileThreads;
                            at[p] = point(q < npts ? q : q0, x[p], y[p], z[p]);
                        }
                        run_general<kGeneralPoints, false>(R.T, n, x, y, z, v, stack, kTileThreads);
#pragma unroll
                        for (int p = 0; p < kGeneralPoints; ++p)
                            if (q0 + p * kTileThreads < npts) box[at[p]] = v[p];
                    }
                } else if (staged) {
                    for (uint32_t q = thread_id(); q < npts; q += kTileThreads) {
                        float x[1], y[1], z[1], v[1];
                        const uint32_t at = point(q, x[0], y[0], z[0]);
                        run_general<1, true>(R.T, n, x, y, z, v, stack, kTileThreads);
                        box[at] = v[0];
                    }
                }
            }
            evaluated = npts;
        }
        if (thread_id() < 64 && ((lv >> thread_id()) & 1ull))  // the live bricks, in order
            lb[__builtin_popcountll(lv & ((1ull << thread_id()) - 1ull))] = (uint8_t)thread_id();
        __syncthreads();  // the box is complete
        if (LINEAR) {
            if (thread_id() == 0) nlist = 0;  // every thread has read the total
            prefetch();  // the next slot's record, while this one is contoured
        }
        contour_tile(P, G, slot, tx, ty, tzl, box, R.A, (uint32_t)__builtin_popcountll(lv), lb, list, L);
        if (thread_id() == 0) {
            tiles_done += 1;
            points_done += evaluated;
            flops_done += (uint64_t)evaluated * tile_flops;
        }
    }
    if (thread_id() == 0 && tiles_done) {  // the job's statistics, one set per queue group (k_sp_emit sums them)
        unsigned long long* st = reinterpret_cast<unsigned long long*>(P.queues) + (blockIdx.x % kQueueGroups) * 16u + 1u;
        atomicAdd(&st[0], (unsigned long long)tiles_done);
        atomicAdd(&st[1], (unsigned long long)points_done);
        atomicAdd(&st[2], (unsigned long long)flops_done);
    }
}

template <int KIND>
__global__ void k_sp_tiles(SpPass P);
template <>
__global__ __launch_bounds__(kTileThreads) __attribute__((amdgpu_waves_per_eu(6, 8))) void k_sp_tiles<kFoldKind>(SpPass P)
{
    tiles_body<kFoldKind>(P, blockIdx.x, gridDim.x);
}
template <>
__global__ __launch_bounds__(kTileThreads) void k_sp_tiles<kGeneralKind>(SpPass P)
{
    tiles_body<kGeneralKind>(P, blockIdx.x, gridDim.x);
}
template <>
__global__ __launch_bounds__(kTileThreads) void k_sp_tiles<kLongKind>(SpPass P)
{
    tiles_body<kLongKind>(P, blockIdx.x, gridDim.x);
}
template <>
__global__ __launch_bounds__(kTileThreads) void k_sp_tiles<kBothKinds>(SpPass P)
{
    const uint32_t general = general_blocks(active_slots(P, kGenUsed), active_slots(P, kSlotsUsed));
    if (blockIdx.x >= general) tiles_body<kFoldKind>(P, blockIdx.x - general, gridDim.x - general);
    else tiles_body<kGeneralKind>(P, blockIdx.x, general);
}

// ---------------------------------------------------------------------------------
// Quads of a cell with a vertex (mesh.rs:267-324) from its sign bits s and its look-back
// neighbours (exists(dx, dy, dz), dx, dy, dz in {-1, 0}; x, y, z: the cell in the job):
// the mask of valid quads (bit 0: x-edge, 1: y-edge, 2: z-edge).  `invalid` counts the
// quads with a missing vertex, and with the readback lag the z = 0 ones that the lagged
// reference looks up (label z - 1) and misses.
// ---------------------------------------------------------------------------------
template <typename E>
__device__ __forceinline__ uint32_t cell_quads(uint32_t s, uint32_t x, uint32_t y, uint32_t z, bool lag,
                                               const E& exists, uint32_t& invalid)
{
    const bool c0 = s & 1u, c1 = (s >> 1) & 1u, c2 = (s >> 2) & 1u, c3 = (s >> 3) & 1u;
    uint32_t nq = 0;
    if (c0 != c3 && y > 0) {  // x-edge: v(x,y-1,z-1), v(x,y,z-1), v, v(x,y-1,z)
        if (z > 0) {
            if (exists(0, -1, -1) && exists(0, 0, -1) && exists(0, -1, 0)) nq |= 1u;
            else ++invalid;
        } else if (lag) {
            ++invalid;
        }
    }
    if (c1 != c3 && x > 0) {  // y-edge: v(x-1,y,z-1), v(x,y,z-1), v, v(x-1,y,z)
        if (z > 0) {
            if (exists(-1, 0, -1) && exists(0, 0, -1) && exists(-1, 0, 0)) nq |= 2u;
            else ++invalid;
        } else if (lag) {
            ++invalid;
        }
    }
    if (c2 != c3 && x > 0 && y > 0) {  // z-edge: v(x-1,y-1,z), v(x,y-1,z), v, v(x-1,y,z)
        if (exists(-1, -1, 0) && exists(0, -1, 0) && exists(-1, 0, 0)) nq |= 4u;
        else ++invalid;
    }
    return nq;
}

// ---------------------------------------------------------------------------------
// k_sp_quadcount: per slot (one 64-lane block iteration), the valid quads of the tile's
// cells with a vertex (their staged entries), two triangles each, summed per row segment
// into the slot's kRowTri row; the invalid ones are added to the pass's and the job's
// counts.
// ---------------------------------------------------------------------------------
__global__ __launch_bounds__(64) void k_sp_quadcount(SpPass P, MeshBufs b)
{
    __shared__ uint32_t ex[81];    // row (k, j): bit i = cell (8tx-1+i, 8ty-1+j, 8tz-1+k) has a vertex
    __shared__ uint32_t rowt[64];  // triangles of each row segment of the tile
    const uint32_t nslots = active_slots(P);
    for (uint32_t slot = blockIdx.x; slot < nslots; slot += gridDim.x) {
        const SlotHdr& H = P.slot_hdr[slot];
        const SpJob& J = P.jobs[__builtin_amdgcn_readfirstlane(H.job)];
        const uint32_t base = __builtin_amdgcn_readfirstlane(P.slot_stage[2 * slot]);
        const uint32_t n = __builtin_amdgcn_readfirstlane(P.slot_stage[2 * slot + 1]);
        const bool lag = (J.flags & S2M_COMPAT_DROP_LAST_SLICE) != 0;
        const uint32_t txy = __builtin_amdgcn_readfirstlane(H.txy);
        const uint32_t tx = txy & 0xffffu, ty = txy >> 16, tzl = __builtin_amdgcn_readfirstlane(H.tzl);
        __syncthreads();  // the previous slot's readers of ex / rowt are done
        int32_t ns[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) ns[i] = P.slot_nb[(size_t)slot * 8u + i];
        for (uint32_t t = thread_id(); t < 81u; t += 64u)
            ex[t] = nb_row<false>(P, J, tx, ty, J.tz0 + tzl, ns, (int)(ty * 8u + t % 9u) - 1,
                                  (int)(J.z0 + tzl * 8u + t / 9u) - 1, nullptr);
        rowt[thread_id()] = 0;
        __syncthreads();
        uint32_t invalid = 0;
        for (uint32_t k = thread_id(); k < n; k += 64u) {
            if ((uint64_t)base + k >= P.stage_cap) break;
            const uint32_t meta = __float_as_uint(P.stage[(uint64_t)base + k].w);
            const uint32_t c = meta & 511u, sg = meta >> 12;
            const uint32_t cxl = c & 7u, cyl = (c >> 3) & 7u, czl = c >> 6;
            auto exists = [&](int dx, int dy, int dz) {
                return ((ex[(czl + 1 + dz) * 9 + (cyl + 1 + dy)] >> (cxl + 1 + dx)) & 1u) != 0;
            };
            const uint32_t nq = cell_quads(sg, tx * 8u + cxl, ty * 8u + cyl, J.z0 + tzl * 8u + czl, lag, exists,
                                           invalid);
            if (nq) atomicAdd(&rowt[c >> 3], 2u * (uint32_t)__builtin_popcount(nq));
        }
        __syncthreads();
        {
            const uint32_t row = thread_id();
            slot_row(P, kRowTri, slot)[row] = rowt[row];  // 0 outside the grid
        }
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) invalid += __shfl_xor(invalid, d, 64);
        if (thread_id() == 0 && invalid) {
            atomicAdd((unsigned long long*)&b.counters[kInvalid], (unsigned long long)invalid);
            atomicAdd((unsigned long long*)&P.job_out[(size_t)J.out_index * kJobOut + 2], (unsigned long long)invalid);
        }
    }
}

// ---------------------------------------------------------------------------------
// k_sp_emit: per slot (one 64-lane block iteration), the staged vertices at their ordered
// index (row-segment offset + rank) with key, sign bits and the 4-tap normal of the
// tile's pruned program (sdf3d_normal.wgsl:4-9, dualcontour.wgsl:171), then the
// triangles of their valid quads at the row segment's triangle offset plus the
// triangles of the cells before them in the segment (make_triangles, mesh.rs:250-265).
// Triangle vertex indices are relative to the job's first vertex.  LINEAR = 1 handles the
// slots whose program is a left fold, LINEAR = 0 the others (launched only when a program
// of the pass is not a left fold; its stack interpreter needs more registers).
//
// A slot is a chain of dependent loads (header, neighbours' rows, staged vertices, tape), four
// folds per vertex and scattered stores of rows a few vertices long: bound by latency and by
// instruction issue alike (half of the issue slots), the 228 MB of a CSG-64 1024^3 mesh take
// 50 us at copy speed.  So the loads of a slot are issued together (no branch between them),
// rows are stored 8 bytes at a time, and blocks draw slots: with slots dealt out in advance
// a block's share of vertices varies twofold and half of the waves idled at the end.
// 325 -> 243 us there (69 k slots, 4.0 M vertices), 233 since no load waits for stores.
// ---------------------------------------------------------------------------------
// The first fold block of k_sp_emit after a job's last pass: the statistics summed and
// counters[0 .. nback) to P.back (mapped host memory, NULL: not wanted).  Nothing in the
// kernel changes them.
__device__ __forceinline__ void report(const SpPass& P)
{
    const uint32_t ln = lane();
    if (!P.back) return;
    static_assert(kQueueGroups == 64, "one statistics line per lane");
    const uint64_t* st = reinterpret_cast<const uint64_t*>(P.queues) + ln * 16u + 1u;
    uint64_t sum[3] = {st[0], st[1], st[2]};
#pragma unroll
    for (int q = 0; q < 3; ++q)
        for (int d = 32; d >= 1; d >>= 1) sum[q] += __shfl_xor(sum[q], d, 64);
    for (uint32_t i = ln; i < P.nback; i += 64u)
        P.back[i] = i == kTilesActive ? sum[0] : i == kEvalPoints ? sum[1] : i == kEvalFlops ? sum[2] : P.counters[i];
}

struct EmitLds {
    uint32_t nb[729];     // vertex of cell (8tx-1+i, 8ty-1+j, 8tz-1+k) at nb[(k*9+j)*9+i]
    uint32_t tc[128];     // triangles of cell c in byte c % 4 of tc[c / 4]
    uint32_t trow[64];    // first triangle of row segment c >> 3
    uint16_t quads[512];  // staged cell k: cell | signs << 9 | valid quads << 13
};

template <int LINEAR>
__device__ __forceinline__ void emit_body(const SpPass& P, const MeshBufs& b, EmitLds& E, uint32_t block, uint32_t blocks)
{
    __shared__ StagedTape T;      // programs that are not left folds (left folds: read in place)
    __shared__ uint32_t mandel;   // such a program holds a Mandelbulb
    extern __shared__ float taps[];  // their operand stacks: P.prune_depth entries of 4 per lane
    uint32_t *const nb = E.nb, *const tc = E.tc, *const trow = E.trow;
    uint16_t* const quads = E.quads;
    if (LINEAR && block == 0) report(P);
    const uint32_t nslots = active_slots(P, LINEAR ? kSlotsNow : kGenNow);
    // the turns after the first are drawn one ahead
    const Turns Q(P, LINEAR ? 2u : 3u, block, blocks);
    uint32_t drawn = 0;
    for (uint32_t turn = Q.first(); turn < nslots; turn = Q.drawn((uint32_t)__builtin_amdgcn_readfirstlane(drawn))) {
        if (thread_id() == 0) drawn = Q.draw();
        const uint32_t slot = LINEAR ? turn : P.gen_slots[turn];
        const SlotHdr& H = P.slot_hdr[slot];
        const uint64_t tile = __builtin_amdgcn_readfirstlane(H.tile);
        const SpJob& J = P.jobs[__builtin_amdgcn_readfirstlane(H.job)];
        const uint32_t base = __builtin_amdgcn_readfirstlane(P.slot_stage[2 * slot]);
        const uint32_t n = __builtin_amdgcn_readfirstlane(P.slot_stage[2 * slot + 1]);
        const uint32_t txy = __builtin_amdgcn_readfirstlane(H.txy);
        const uint32_t tx = txy & 0xffffu, ty = txy >> 16, tzl = __builtin_amdgcn_readfirstlane(H.tzl);
        const bool normals = !(J.flags & S2M_NO_NORMALS);
        const bool lag = (J.flags & S2M_COMPAT_DROP_LAST_SLICE) != 0;
        const uint32_t vbase = (uint32_t)P.job_out[(size_t)J.out_index * kJobOut + 0];
        const uint16_t* Lst = slot_list(P, slot, tile);
        const uint32_t lens = __builtin_amdgcn_readfirstlane(H.lens);
        const uint32_t len = lens & ~kLinearFlag;
        const bool linear = (lens & kLinearFlag) != 0, staged = len <= kStageOps;
        if (linear != (LINEAR != 0)) continue;  // the other launch's slot
        __syncthreads();  // the previous slot's readers of T, nb, tc are done
        if (!LINEAR && normals && staged) {
            if (thread_id() == 0) mandel = 0;
            stage_tape(T, J.ops, Lst, len);
            __syncthreads();
            for (uint32_t q = thread_id(); q < len; q += 64u)
                if (T.code[q] == S2M_OP_MANDELBULB) mandel = 1;
        }
        // left folds: the program as staged in the slot's record, read in place
        const ScalarFold TS =
            ScalarFold::at(reinterpret_cast<const char*>(P.slot_rec + (size_t)slot * kRecVec) + offsetof(TileRec, T));
        int32_t ns[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) ns[i] = P.slot_nb[(size_t)slot * 8u + i];
        // the first round's vertex and the segments' triangle offsets, read beside the rows
        float4 e0 = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (thread_id() < n && (uint64_t)base + thread_id() < P.stage_cap) e0 = P.stage[(uint64_t)base + thread_id()];
        {
            const uint32_t r = thread_id(), zl = tzl * 8u + (r >> 3), y = ty * 8u + (r & 7u);
            uint32_t t = 0;
            if (zl < J.nz && y < J.ry)
                t = slot_row(P, kRowTriOff, slot)[r] + P.row_off[P.nrows + row_index(J, zl, y)];
            trow[r] = t;
        }
        for (uint32_t t = thread_id(); t < 81u; t += 64u)
            (void)nb_row<true>(P, J, tx, ty, J.tz0 + tzl, ns, (int)(ty * 8u + t % 9u) - 1,
                               (int)(J.z0 + tzl * 8u + t / 9u) - 1, nb + 9u * t);
        for (uint32_t w = thread_id(); w < 128u; w += 64u) tc[w] = 0;
        __syncthreads();
        // vertices, and each cell's triangle count.  A load waits for the stores before it, so
        // the next round's vertex is loaded before this round's stores and the triangle loop
        // loads nothing.
        for (uint32_t k = thread_id(); k < n; k += 64u) {
            if ((uint64_t)base + k >= P.stage_cap) break;
            const float4 e = e0;
            if (k + 64u < n && (uint64_t)base + k + 64u < P.stage_cap) e0 = P.stage[(uint64_t)base + k + 64u];
            const uint32_t meta = __float_as_uint(e.w);
            const uint32_t c = meta & 511u, sg = meta >> 12;
            const uint32_t cxl = c & 7u, cyl = (c >> 3) & 7u, czl = c >> 6;
            const uint32_t at = ((czl + 1) * 9u + (cyl + 1)) * 9u + (cxl + 1);
            auto exists = [&](int dx, int dy, int dz) { return nb[(int)at + (dz * 9 + dy) * 9 + dx] != kNone; };
            uint32_t invalid = 0;
            const uint32_t nq =
                cell_quads(sg, tx * 8u + cxl, ty * 8u + cyl, J.z0 + tzl * 8u + czl, lag, exists, invalid);
            if (nq) atomicOr(&tc[c >> 2], (2u * (uint32_t)__builtin_popcount(nq)) << ((c & 3u) * 8u));
            quads[k] = (uint16_t)(c | (sg << 9) | (nq << 13));
            const uint64_t vi = nb[at];
            if (vi >= b.vcap) continue;
            float2* o = reinterpret_cast<float2*>(b.vtx + 6 * vi);
            o[0] = make_float2(e.x, e.y);
            b.keys[vi] = (uint64_t)(tx * 8u + cxl) | ((uint64_t)(ty * 8u + cyl) << 16) |
                         ((uint64_t)(J.z0 + tzl * 8u + czl) << 32);
            b.signs[vi] = (uint8_t)sg;
            if (!normals) {
                o[1] = make_float2(e.z, 0.0f);
                o[2] = make_float2(0.0f, 0.0f);
                continue;
            }
            const float px = e.x, py = e.y, pz = e.z, eps = J.eps;
            // sdf3d_normal (sdf3d_normal.wgsl:4-9): taps p + v_i * eps, then normalize
            const float tx4[4] = {px + eps, px + (-eps), px + (-eps), px + eps};
            const float ty4[4] = {py + (-eps), py + (-eps), py + eps, py + eps};
            const float tz4[4] = {pz + (-eps), pz + eps, pz + (-eps), pz + eps};
            float d[4];
            if constexpr (LINEAR != 0) {
                run_linear<4>(TS, len, tx4, ty4, tz4, d);
            } else if (staged && !mandel) {
                run_general<4, false>(T, len, tx4, ty4, tz4, d, taps + thread_id(), 64u);
            } else {
                for (int t = 0; t < 4; ++t) {
                    const float x[1] = {tx4[t]}, y[1] = {ty4[t]}, z[1] = {tz4[t]};
                    float v[1];
                    if (staged) run_general<1, true>(T, len, x, y, z, v, taps + thread_id(), 64u);
                    else v[0] = tape_eval_list(J.ops, Lst, len, x[0], y[0], z[0]);
                    d[t] = v[0];
                }
            }
            const float d1 = d[0], d2 = d[1], d3 = d[2], d4 = d[3];
            const float gx = ((d1 + (-d2)) + (-d3)) + d4;
            const float gy = (((-d1) + (-d2)) + d3) + d4;
            const float gz = (((-d1) + d2) + (-d3)) + d4;
            const float ln = sqrtf((gx * gx + gy * gy) + gz * gz);
            o[1] = make_float2(e.z, canonical_nan(gx / ln));
            o[2] = make_float2(canonical_nan(gy / ln), canonical_nan(gz / ln));
        }
        __syncthreads();  // every cell's triangle count is in tc
        // triangles, in vertex order: each quad (q2, q1, q0), (q0, q3, q2)
        for (uint32_t k = thread_id(); k < n; k += 64u) {
            if ((uint64_t)base + k >= P.stage_cap) break;
            const uint32_t word = quads[k], c = word & 511u, sg = (word >> 9) & 15u, nq = word >> 13;
            if (!nq) continue;
            const uint32_t cxl = c & 7u, cyl = (c >> 3) & 7u, czl = c >> 6;
            const uint32_t at = ((czl + 1) * 9u + (cyl + 1)) * 9u + (cxl + 1);
            auto nbv = [&](int dx, int dy, int dz) { return nb[(int)at + (dz * 9 + dy) * 9 + dx]; };
            const uint64_t row2 = ((uint64_t)tc[(c >> 3) * 2u + 1] << 32) | tc[(c >> 3) * 2u];  // 8 counts
            uint64_t t = trow[c >> 3];
            for (uint32_t i = 0; i < cxl; ++i) t += (row2 >> (8u * i)) & 0xffu;
            const uint32_t v = nbv(0, 0, 0);
            const bool c0 = sg & 1u, c1 = (sg >> 1) & 1u, c2 = (sg >> 2) & 1u;
            for (int q = 0; q < 3; ++q) {
                if (!(nq & (1u << q))) continue;
                uint32_t f[4];
                bool rev;
                if (q == 0) {
                    f[0] = nbv(0, -1, -1), f[1] = nbv(0, 0, -1), f[3] = nbv(0, -1, 0), rev = c0;
                } else if (q == 1) {
                    f[0] = nbv(-1, 0, -1), f[1] = nbv(0, 0, -1), f[3] = nbv(-1, 0, 0), rev = !c1;
                } else {
                    f[0] = nbv(-1, -1, 0), f[1] = nbv(0, -1, 0), f[3] = nbv(-1, 0, 0), rev = c2;
                }
                f[2] = v;
                uint32_t qv[4];
                for (int i = 0; i < 4; ++i) qv[i] = (rev ? f[3 - i] : f[i]) - vbase;
                if (t + 1 < b.tcap) {
                    // t is even: triangles come in pairs
                    uint2* o = reinterpret_cast<uint2*>(b.tri + 3 * t);
                    o[0] = make_uint2(qv[2], qv[1]);
                    o[1] = make_uint2(qv[0], qv[0]);
                    o[2] = make_uint2(qv[3], qv[2]);
                }
                t += 2;
            }
        }
    }
}

template <int KIND>
__global__ __launch_bounds__(64) void k_sp_emit(SpPass P, MeshBufs b)
{
    __shared__ EmitLds E;
    if constexpr (KIND != kBothKinds) {
        emit_body<KIND>(P, b, E, blockIdx.x, gridDim.x);
    } else {
        const uint32_t general = general_blocks(active_slots(P, kGenNow), active_slots(P, kSlotsNow));
        if (blockIdx.x >= general) emit_body<1>(P, b, E, blockIdx.x - general, gridDim.x - general);
        else emit_body<0>(P, b, E, blockIdx.x, general);
    }
}

// ---------------------------------------------------------------------------------
// Offsets in the reference's VertexList order: job after job, then (z, y, tile x).
//  k_sp_rowsum    one wave per tile row (job, tile layer, ty), lane = row (z % 8, y % 8):
//                 the row segments of the tile row's active tiles (the super-tiles'
//                 activity words) in x order: each segment's offset within its row
//                 (the slot's kRowVtxOff / kRowTriOff rows) and the row's totals (row_sum)
//                 and each 4096-row chunk's sums (one atomic per wave and chunk)
//  k_sp_rowdown   exclusive scan of the rows' totals (row_off), block b adding the sums of
//                 the chunks before it
// A segment's first vertex (triangle) is row_off[row] + its offset within the row.
// ---------------------------------------------------------------------------------
constexpr uint32_t kScanPer = 16;                  // rows per thread
constexpr uint32_t kScanThreads = 256;
constexpr uint32_t kScanChunk = kScanThreads * kScanPer;
static_assert(kScanChunk == kRowChunk, "rows per chunk of the offset scan");

__global__ __launch_bounds__(64) void k_sp_rowsum(SpPass P)
{
    uint32_t* bsum = P.bsum;
    const uint64_t tr = blockIdx.x;
    uint32_t lo = 0, hi = P.njobs - 1;  // last job whose first tile row <= tr
    while (lo < hi) {
        const uint32_t mid = (lo + hi + 1) / 2;
        if (P.jobs[mid].trow_base <= tr) lo = mid;
        else hi = mid - 1;
    }
    const SpJob& J = P.jobs[__builtin_amdgcn_readfirstlane(lo)];
    const uint32_t local = (uint32_t)(tr - J.trow_base), ty = local % J.nty, tzl = local / J.nty;
    const uint32_t zl = tzl * 8u + (lane() >> 3), y = ty * 8u + (lane() & 7u);
    const bool row_ok = zl < J.nz && y < J.ry;
    const uint64_t srow = J.super_base + ((uint64_t)(tzl / kSuper) * J.nsy + ty / kSuper) * J.nsx;
    const uint32_t bit0 = ((tzl % kSuper) * kSuper + ty % kSuper) * kSuper;
    uint32_t sv = 0, st = 0;
    for (uint32_t sx0 = 0; sx0 < J.nsx; sx0 += 16u) {
        // active tiles 4 * sx0 .. 4 * sx0 + 63: lane l < 16 reads super-tile sx0 + l's word
        // and the slot of the first of its active tiles in this tile row
        uint64_t mine = 0;
        uint32_t first = 0;
        if (lane() < 16u && sx0 + lane() < J.nsx) {
            const SuperSlots S = P.super_act[srow + sx0 + lane()];
            mine = ((S.act >> bit0) & 0xfull) << (4u * lane());
            first = S.first + (uint32_t)__builtin_popcountll(S.act & ((1ull << bit0) - 1ull));
        }
#pragma unroll
        for (int d = 8; d >= 1; d >>= 1) mine |= __shfl_xor(mine, d, 64);
        const uint32_t m0 = __builtin_amdgcn_readfirstlane((uint32_t)mine);
        const uint32_t m1 = __builtin_amdgcn_readfirstlane((uint32_t)(mine >> 32));
        uint64_t m = (uint64_t)m1 << 32 | m0;
        const uint64_t all = m;
        // the active tiles' row counts (one 256-byte row of each slot), 8 tiles at a time
        while (m) {
            uint32_t slots[8], v[8], t[8];
            uint32_t nb = 0;
#pragma unroll
            for (uint32_t k = 0; k < 8u; ++k) {
                slots[k] = 0;
                if (m) {
                    const uint32_t t = (uint32_t)__builtin_ctzll(m), l = t >> 2;
                    m &= m - 1ull;
                    slots[k] = (uint32_t)__builtin_amdgcn_readlane((int)first, (int)l) +
                               (uint32_t)__builtin_popcountll((all >> (4u * l)) & ((1ull << (t & 3u)) - 1ull));
                    nb = k + 1;
                }
            }
#pragma unroll
            for (uint32_t k = 0; k < 8u; ++k) {
                v[k] = t[k] = 0;
                if (k < nb) {
                    v[k] = slot_row(P, kRowVtx, slots[k])[lane()];
                    t[k] = slot_row(P, kRowTri, slots[k])[lane()];
                }
            }
#pragma unroll
            for (uint32_t k = 0; k < 8u; ++k) {
                if (k < nb) {
                    slot_row(P, kRowVtxOff, slots[k])[lane()] = sv;
                    slot_row(P, kRowTriOff, slots[k])[lane()] = st;
                }
                sv += v[k];
                st += t[k];
            }
        }
    }
    const uint64_t row = row_ok ? row_index(J, zl, y) : 0;
    if (row_ok) {
        P.row_sum[row] = sv;
        P.row_sum[P.nrows + row] = st;
    }
    // the rows' totals into their chunks' sums (bsum: per chunk a vertex and a triangle sum,
    // kChunkSumStride words apart), one atomic per chunk the wave's rows fall in
    const uint32_t chunk = (uint32_t)(row / kScanChunk);
    uint64_t rem = __ballot(row_ok && (sv | st));
    while (rem) {
        const uint32_t c = __shfl(chunk, (int)__builtin_ctzll(rem), 64);
        const bool mine = ((rem >> lane()) & 1ull) && chunk == c;
        uint32_t v = mine ? sv : 0u, t = mine ? st : 0u;
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) {
            v += __shfl_xor(v, d, 64);
            t += __shfl_xor(t, d, 64);
        }
        if (lane() == (uint32_t)__builtin_ctzll(rem)) {
            if (v) atomicAdd(&bsum[(2u * c) * kChunkSumStride], v);
            if (t) atomicAdd(&bsum[(2u * c + 1u) * kChunkSumStride], t);
        }
        rem &= ~__ballot(mine);
    }
}

// Exclusive offsets of the rows, block b = rows b * kScanChunk ...: the pass's first index
// (kVtxPrev / kTriPrev) plus the chunk sums of the blocks before it (bsum) plus the
// block-local scan.  The last block writes the totals after the pass (kVtxTotal / kTriTotal).
// Wave w of a block takes rows w * 1024 ... of its chunk, 64 at a time (a thread with 16 rows
// in a row made every load and store of a wave touch 64 lines).  Bound by latency: all that
// does not depend on something else is read at the start.  10.2 -> 4.7 us at tree 256^3,
// 17.6 -> 6.2 at CSG-64 1024^3.
__global__ __launch_bounds__(kScanThreads) void k_sp_rowdown(SpPass P)
{
    constexpr uint32_t kWaves = kScanThreads / 64;
    const uint32_t* bsum = P.bsum;
    __shared__ uint32_t lds[2][kWaves];
    __shared__ uint32_t pre[2][kWaves];
    const uint32_t wave = thread_id() >> 6;
    const uint64_t base = (uint64_t)blockIdx.x * kScanChunk + wave * 64u * kScanPer + lane();
    const bool last = blockIdx.x + 1 == gridDim.x && thread_id() == 0;
    uint32_t v[kScanPer], t[kScanPer];
#pragma unroll
    for (uint32_t k = 0; k < kScanPer; ++k) {
        const uint64_t r = base + 64u * k;
        v[k] = r < P.nrows ? P.row_sum[r] : 0u;
        t[k] = r < P.nrows ? P.row_sum[P.nrows + r] : 0u;
    }
    const uint32_t vprev = (uint32_t)P.counters[kVtxPrev], tprev = (uint32_t)P.counters[kTriPrev];
    uint64_t slots = 0, stage = 0, general = 0, slots_max = 0, stage_max = 0;
    if (last) {
        slots = P.counters[kSlotsUsed];
        stage = P.counters[kStageUsed] + 2ull * P.tile_blocks * kStageChunk;
        general = P.counters[kGenUsed];
        slots_max = P.counters[kSlotsMax];
        stage_max = P.counters[kStageMax];
    }
    uint32_t cv = 0, ct = 0;  // the chunks before this block
    for (uint32_t c = thread_id(); c < blockIdx.x; c += kScanThreads) {
        cv += bsum[(2u * c) * kChunkSumStride];
        ct += bsum[(2u * c + 1u) * kChunkSumStride];
    }
    // exclusive offsets within the wave's rows, in place
    uint32_t sv = 0, st = 0;
#pragma unroll
    for (uint32_t k = 0; k < kScanPer; ++k) {
        const uint32_t iv = wave_scan(v[k]), it = wave_scan(t[k]);
        v[k] = sv + iv - v[k];
        t[k] = st + it - t[k];
        sv += (uint32_t)__builtin_amdgcn_readlane((int)iv, 63);
        st += (uint32_t)__builtin_amdgcn_readlane((int)it, 63);
    }
    if (blockIdx.x) {
        cv = wave_scan(cv);
        ct = wave_scan(ct);
    }
    if (lane() == 63) {
        lds[0][wave] = sv;
        lds[1][wave] = st;
        pre[0][wave] = cv;
        pre[1][wave] = ct;
    }
    __syncthreads();
    uint32_t rv = vprev, rt = tprev, bv = vprev, bt = tprev;
#pragma unroll
    for (uint32_t w = 0; w < kWaves; ++w) {
        rv += pre[0][w] + (w < wave ? lds[0][w] : 0u);
        rt += pre[1][w] + (w < wave ? lds[1][w] : 0u);
        bv += pre[0][w] + lds[0][w];
        bt += pre[1][w] + lds[1][w];
    }
    if (last) {  // after the pass
        // for the host, which allocates and queues the copies of the pass's mesh while
        // k_sp_emit writes it
        if (P.snap) {
            const uint64_t n[kSnapWords] = {bv, bt, slots, stage};
            for (uint32_t q = 0; q < kSnapWords; ++q)
                __hip_atomic_store(P.snap + q, n[q] | kSnapValid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
        P.counters[kVtxTotal] = bv;
        P.counters[kTriTotal] = bt;
        // the pass's slots and staging: kept, folded into their maxima, reset
        P.counters[kGenNow] = general;
        P.counters[kGenUsed] = 0;
        P.counters[kSlotsNow] = slots;
        P.counters[kSlotsUsed] = 0;
        P.counters[kStageUsed] = 0;
        if (slots > slots_max) P.counters[kSlotsMax] = slots;
        if (stage > stage_max) P.counters[kStageMax] = stage;
    }
#pragma unroll
    for (uint32_t k = 0; k < kScanPer; ++k) {
        const uint64_t r = base + 64u * k;
        if (r >= P.nrows) break;
        P.row_off[r] = rv + v[k];
        P.row_off[P.nrows + r] = rt + t[k];
    }
    // the first vertex and triangle index of every job whose first slab this pass holds and
    // whose first row is this block's: the exclusive offsets of that row
    __syncthreads();
    const uint64_t lo = (uint64_t)blockIdx.x * kScanChunk, hi = lo + kScanChunk;
    for (uint32_t j = thread_id(); j < P.njobs; j += kScanThreads) {
        const SpJob& J = P.jobs[j];
        if (J.z0 != 0 || (uint64_t)J.nz * J.ry == 0 || J.row_base < lo || J.row_base >= hi) continue;
        uint64_t* o = P.job_out + (size_t)J.out_index * kJobOut;
        o[0] = (uint64_t)P.row_off[J.row_base];
        o[1] = (uint64_t)P.row_off[P.nrows + J.row_base];
    }
}

// Cell -> vertex map of the slab's last plane, for the next slab (single job).
__global__ __launch_bounds__(256) void k_sp_boundary(SpPass P)
{
    const SpJob& J = P.jobs[0];
    const uint32_t i = blockIdx.x * blockDim.x + thread_id();
    if (i >= J.rx * J.ry) return;
    J.boundary[i] = vertex_at(P, J, i % J.rx, i / J.rx, J.z0 + J.nz - 1);
}

// Blocks of a persistent launch: as many as the device holds at once (at most `cap`),
// so no block starts only when others end.  The occupancy query is slow (tens of
// microseconds), so its answer is cached per (kernel, block size, LDS bytes).
template <typename K>
static uint32_t resident_blocks(K kernel, int threads, size_t smem, int cus, uint32_t cap)
{
    struct Entry {
        const void* f;
        int threads;
        size_t smem;
        int per_cu;
    };
    static std::mutex mu;
    static std::vector<Entry> cache;
    const void* f = reinterpret_cast<const void*>(kernel);
    int per_cu = 0;
    {
        std::lock_guard<std::mutex> lock(mu);
        for (const Entry& e : cache)
            if (e.f == f && e.threads == threads && e.smem == smem) per_cu = e.per_cu;
    }
    if (per_cu == 0) {
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, f, threads, smem) != hipSuccess || per_cu < 1)
            per_cu = 1;
        std::lock_guard<std::mutex> lock(mu);
        cache.push_back(Entry{f, threads, smem, per_cu});
    }
    return std::min<uint32_t>(cap, (uint32_t)cus * (uint32_t)per_cu);
}

hipError_t launch_sparse_pass(hipStream_t s, SpPass P, const MeshBufs& b, int cus,
                              uint32_t tile_blocks, bool general_tiles, int boundary_plane, hipEvent_t* marks)
{
    if (P.ntiles == 0) return hipSuccess;
    const uint64_t nsb64 = (P.nrows + kScanChunk - 1) / kScanChunk;
    if (nsb64 > kMaxScanBlocks) return hipErrorInvalidValue;
    const uint32_t nsb = (uint32_t)nsb64;
    const uint32_t big = 1u << 20;
    auto mark = [&](int i) {
        if (marks && marks[i]) (void)hipEventRecord(marks[i], s);
    };
    const size_t prune_smem = PruneStack::bytes(P.prune_depth) + (size_t)P.walk_ops * 64u * sizeof(uint16_t);
    if (P.nsuper > 0x7fffffffull) return hipErrorInvalidValue;
    mark(0);
    hipLaunchKernelGGL(k_sp_prune, dim3((uint32_t)P.nsuper), dim3(64), prune_smem, s, P);
    hipLaunchKernelGGL(k_sp_bricks, dim3(resident_blocks(k_sp_bricks, 64, 0, cus, big)), dim3(64), 0, s, P);
    mark(1);
    const size_t smem = (size_t)P.box_stride * sizeof(float);
    const size_t gsmem = smem + (size_t)P.prune_depth * (P.prune_depth <= kWideDepth ? kGeneralPoints : 1) *
                                    kTileThreads * sizeof(float);
    const size_t esmem = (size_t)P.prune_depth * 4u * 64u * sizeof(float);
    const bool both = general_tiles && P.ntiles <= (P.lists_by_tile ? kBothTilesLong : kBothTiles);
    P.long_apart = P.lists_by_tile && !both ? 1u : 0u;
    auto tiles = [&](auto kernel, size_t lds) {
        hipLaunchKernelGGL(kernel, dim3(resident_blocks(kernel, kTileThreads, lds, cus, tile_blocks)), dim3(kTileThreads),
                           lds, s, P);
    };
    auto emit = [&](auto kernel, size_t lds) {
        hipLaunchKernelGGL(kernel, dim3(resident_blocks(kernel, 64, lds, cus, big)), dim3(64), lds, s, P, b);
    };
    if (both) {
        tiles(k_sp_tiles<kBothKinds>, gsmem);
    } else {
        tiles(k_sp_tiles<kFoldKind>, smem);
        if (general_tiles) tiles(k_sp_tiles<kGeneralKind>, gsmem);
        if (P.long_apart) tiles(k_sp_tiles<kLongKind>, smem);
    }
    mark(2);
    hipLaunchKernelGGL(k_sp_quadcount, dim3(resident_blocks(k_sp_quadcount, 64, 0, cus, big)), dim3(64), 0, s,
                       P, b);
    mark(3);
    if (P.ntrows) hipLaunchKernelGGL(k_sp_rowsum, dim3((uint32_t)P.ntrows), dim3(64), 0, s, P);
    if (nsb) hipLaunchKernelGGL(k_sp_rowdown, dim3(nsb), dim3(kScanThreads), 0, s, P);
    mark(4);
    if (both) {
        emit(k_sp_emit<kBothKinds>, esmem);
    } else {
        emit(k_sp_emit<kFoldKind>, 0);
        if (general_tiles) emit(k_sp_emit<kGeneralKind>, esmem);
    }
    if (boundary_plane) {
        hipLaunchKernelGGL(k_sp_boundary, dim3((uint32_t)((P.boundary_cells + 255) / 256)), dim3(256), 0,
                           s, P);
    }
    mark(5);
    return hipGetLastError();
}

}  // namespace s2m
