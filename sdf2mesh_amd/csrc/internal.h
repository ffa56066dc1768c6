// internal.h - declarations shared by the host runtime (api.cpp) and the kernels
// (kernels.hip).  Not part of the C ABI.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <string>

#include "../../include/sdf2mesh.h"

namespace s2m {

constexpr uint32_t kBlock = 256;             // threads per block of the cell kernels
constexpr uint32_t kRounds = 4;              // cells per thread (strided by kBlock)
constexpr uint32_t kCellsPerBlock = kBlock * kRounds;
constexpr uint32_t kMaxScanBlocks = 65536;   // most block counts one dense slab (sparse pass) scans
constexpr uint32_t kRankChunks = kMaxScanBlocks / 1024;  // chunks of 1024 blocks of a dense slab
static_assert(kRankChunks <= 256, "one block's threads set up the chunk bases");
constexpr uint32_t kBrickBlocks = 2048;      // blocks of 4 waves of the per-brick kernels: 8 waves per
                                             // SIMD of 256 CUs
constexpr uint32_t kNormalBlocks = 4096;     // blocks of 64 vertices of the normal kernels
constexpr uint32_t kNone = 0xffffffffu;      // "no vertex" (u32::MAX, mesh.rs:330)

// Unsigned division by a runtime constant d >= 1 (round-up multiplier method):
// n / d == (umulhi(n, m) + n) >> l for every 32-bit n, evaluated in 64 bits.
struct FastDiv {
    uint32_t d, m, l;
};
FastDiv make_fastdiv(uint32_t d);

// A pass's (slab's) totals for the host, written before its mesh is complete: vertices and
// triangles so far, slots and staged cells in use, each with kSnapValid set (the host polls
// for it, so the words need no order among them).
constexpr uint32_t kSnapWords = 4;
constexpr uint64_t kSnapValid = 1ull << 63;

// Arrays copied by one kernel (k_copy_out); addresses are 16-byte aligned.
struct CopyList {
    const void* src[4];
    void* dst[4];
    uint64_t bytes[4];
};

// Device counters of one job (u64 each).
enum Counter : uint32_t {
    kVtxTotal = 0,   // vertices emitted so far (all slabs)
    kVtxPrev = 1,    // vertex total before the current slab
    kTriTotal = 2,   // triangles emitted so far
    kTriPrev = 3,
    kInvalid = 4,    // quads skipped for a missing vertex
    kTilesActive = 5,  // tiles whose cells were evaluated (tiled path)
    kEvalPoints = 6,   // lattice points evaluated (tiled path)
    kEvalFlops = 7,    // algorithmic flops executed by the pruned tapes (tiled path)
    kSlotsUsed = 8,    // active tiles of the current slab (sparse path)
    kSlotsMax = 9,     // largest kSlotsUsed of the job so far
    kStageUsed = 10,   // staged active cells of the current pass (sparse path)
    kBrickAlloc = 11,  // dense slab: listed bricks (low word), staged vertices (high word)
    kSlotsNow = 13,    // sparse pass: its slots, once they are final
    kStageMax = 12,    // largest kStageUsed of the job so far
    kGenUsed = 15,     // sparse pass: slots whose program is no fold, being counted and final
    kGenNow = 16,
    kNumCounters = 20
};

// Everything the cell kernels need to address one slab of cells [z0, z0+nz).
struct SlabArgs {
    const float* cx;       // per-axis coordinate tables
    const float* cy;
    const float* cz;
    const uint32_t* lox;   // per-axis cell -> coordinate index of the min / max corner
    const uint32_t* hix;
    const uint32_t* loy;
    const uint32_t* hiy;
    const uint32_t* loz;
    const uint32_t* hiz;
    uint32_t rx, ry;       // cells per row, rows per plane
    uint32_t z0;           // first cell plane of the slab
    uint32_t ncells;       // rx * ry * nz
    FastDiv div_rx;
    FastDiv div_rxy;
    uint32_t flags;        // S2M_* flags
};

// A slab's cells with a vertex and their vertices' indices: cell c's is cbase[c / 2^20] +
// boffset[c / 1024] + wpre[c / 64] + the bits before c in its word.
struct SlabBits {
    const unsigned long long* words;
    const uint16_t* wpre;
    const uint32_t* boffset;
    const uint32_t* cbase;
    uint64_t last_plane;   // first cell of the slab's last plane
};

constexpr uint32_t kTile = 8;  // cells per tile edge (sparse pipeline)
constexpr uint32_t kSuper = 4;  // tiles per super-tile edge (first pruning level)
// A pruned list's operator entry with this bit applies its operator with the operands
// swapped: the stack's top is its first (sparse.hip, PruneWalk).
constexpr uint32_t kSwapped = 0x8000u;
static_assert(S2M_MAX_TAPE <= kSwapped, "op indices leave the bit free");
constexpr uint32_t kStageOps = 128;  // longest program staged in LDS (device_staged.h)
constexpr uint32_t kSingleSign = 0xffffffffu;  // a super-tile's list length: the SDF keeps one sign there
constexpr uint32_t kStageChunkHost = 1024;  // staged-cell allocation chunk (sparse.hip)
constexpr uint32_t kTileBlocksPerCU = 8;    // most k_sp_tiles blocks per compute unit
constexpr uint32_t kTileRecBytes = 2720;    // per slot: k_sp_tiles' staged record (sparse.hip)
constexpr uint32_t kRowChunk = 4096;        // rows per chunk of the row offset scan (sparse.hip)
constexpr uint32_t kChunkSumStride = 32;    // words between chunk sums (one 128-byte line each)
constexpr uint32_t kQueues = 5;        // work queues of a pass (k_sp_tiles<1/0>, k_sp_emit<1/0>, k_sp_tiles<3>)
constexpr uint32_t kQueueGroups = 64;  // counters per queue, 32 u32 (128 bytes) apart
// Profiling marks of one sparse pass: prune (tiles, bricks) | eval+contour | quad count |
// scan | emission
constexpr int kSparseMarks = 6;

// Tile-sparse pipeline (sparse.hip).  One job of a pass: a slab of a single job, or a
// whole job of a batch.  Pointers are device addresses.
constexpr uint32_t kJobOut = 4;  // per job: first vertex, first triangle, invalid quads, spare

struct SpJob {
    uint32_t rx, ry;           // cells per row / rows per plane
    uint32_t nz, z0;           // cell planes of this pass
    uint32_t ntx, nty, ntz;    // tiles of the whole job per axis
    uint32_t tz0;              // tile layer of plane z0
    uint32_t nops, flags;
    uint32_t union_fold;       // the program is a left fold of unions / smooth unions (k > 0)
    uint32_t left_fold;        // the program is a left fold of library primitives (at most kStageOps ops)
    uint32_t bx, by;           // lattice box dims of the job's tiles (slot box indexing)
    uint32_t out_index;        // row of the pass's job_out table
    float eps;
    double pad;                // tile box padding (normal taps, rounding)
    uint64_t tile_base;        // first tile of the job in the pass's numbering
    uint64_t row_base;         // first row (zl, y) of the job
    uint64_t trow_base;        // first tile row (tile layer, ty) of the job
    uint64_t super_base;       // first super-tile of the job
    uint32_t nsx, nsy, nsz;    // super-tiles of the job in this pass per axis
    const s2m_op* ops;
    const float* cx;
    const float* cy;
    const float* cz;
    const uint32_t* lox;
    const uint32_t* hix;
    const uint32_t* loy;
    const uint32_t* hiy;
    const uint32_t* loz;
    const uint32_t* hiz;
    const float* ext;          // tile coordinate extents: xmin[ntx] xmax[ntx] ymin.. zmax[ntz]
    const uint32_t* ibox;      // tile lattice index boxes, same layout
    const uint32_t* op_flops;  // [nops], then for programs of at most kStageOps ops [nops] op q's place in the
                               // tree: left operand (the right one is q - 1) | level << 16, primitives 0
    uint32_t levels;           // of the root
    uint32_t* boundary;        // [ry][rx] vertex of cell plane z0 - 1 (multi-slab job)
};

// Per slot, written by k_sp_bricks for the kernels after it.
struct SlotHdr {
    uint32_t tile, job, lens;
    uint32_t txy;    // tile x | tile y << 16
    uint32_t tzl;    // tile layer within the pass
    uint32_t box[3]; // per axis: first lattice index of the tile's box | points << 24
};

// The slots of a super-tile's tiles: bit (z * 4 + y) * 4 + x of `act` says that the tile has one,
// and they are numbered from `first` in bit order.
struct SuperSlots {
    uint64_t act;
    uint32_t first, unused;
};

struct SpPass {
    const SpJob* jobs;
    uint32_t njobs;
    uint32_t list_stride;      // >= nops of every job
    uint32_t prune_depth;      // >= 1, >= the deepest operand stack of any job's program - 1
    uint32_t walk_ops;         // longest program of a job that is no left fold, if at most kStageOps
    uint64_t ntiles;           // tiles of the pass
    uint64_t nrows;            // rows (z, y) of the pass
    uint64_t ntrows;           // tile rows (tile layer, ty) of the pass
    uint64_t boundary_cells;   // rx * ry of jobs[0] when a boundary plane is written
    uint64_t nsuper;           // super-tiles of the pass
    float2* super_iv;         // [super-tile][list_stride] primitive intervals (lo, hi), and pruned op
    uint16_t* super_lists;     // indices, of programs too long for LDS (kStageOps; NULL if none is)
    SuperSlots* super_act;     // [super-tile]
    uint16_t* lists;           // [slot][list_stride] pruned op indices ([tile] with lists_by_tile: programs
                               // longer than kStageOps are listed before their tile has a slot)
    uint32_t lists_by_tile;
    uint32_t long_apart;       // k_sp_tiles<3> runs the slots whose program is not staged
    uint4* slot_info;          // [slot] tile, job, pruned length (| kLinearFlag), its flops per point
    uint32_t* gen_slots;       // the slots whose program is no fold (kGenUsed of them)
    uint32_t slot_cap;
    uint32_t box_stride;       // floats of a tile's lattice box (LDS)
    uint32_t* cellbits;        // [slot][16] bit c: cell c of the tile has a vertex (row r = c / 8
                               // in byte r % 4 of word r / 4)
    float4* stage;             // [stage_cap] active cells: position, cell | signs << 12
    uint64_t stage_cap;
    uint32_t tile_blocks;      // most blocks of a k_sp_tiles launch: the first 2 * tile_blocks staging chunks
                               // are theirs without being counted
    uint32_t* slot_stage;      // [slot][2] first staged cell, staged cells
    SlotHdr* slot_hdr;         // [slot]
    int32_t* slot_nb;          // [slot][8] slots of the tile (tx - dx, ty - dy, tz - dz) at (dz * 2 + dy) * 2 + dx
    uint4* slot_rec;           // [slot] kTileRecBytes: k_sp_tiles<1>'s staged record
    uint32_t* slot_rows;       // [4][slot_cap][64] per row of each slot's tile: vertices,
                               // triangles, first vertex / triangle within the row
    uint32_t* row_sum;         // [2][nrows] vertices, triangles per row
    uint32_t* row_off;         // [2][nrows] exclusive offsets: global vertex / triangle index
    uint64_t* counters;
    uint32_t* queues;          // [kQueues][kQueueGroups][32] work queue counters (word 0); beside those of
                               // queue 0, as u64 words 1..3: tiles, points, flops of the job so far
    uint32_t* bsum;            // the offset scan's chunk sums, kChunkSumStride words apart
    uint32_t nbsum;
    uint32_t nclear;           // a job's first pass: counters and job rows to clear, else 0
    uint32_t nbnd;             // before a multi-pass job: cells of the boundary plane to clear
    uint32_t nback;            // words of `back`
    uint64_t* back;            // mapped host memory for the counters and job rows after a job's last
                               // pass, else NULL
    uint64_t* snap;            // mapped host memory for the pass's totals (kSnapWords), or NULL
    uint64_t* job_out;         // [job][kJobOut]
};

struct MeshBufs {
    float* vtx;            // 6 floats per vertex
    uint64_t* keys;
    uint8_t* signs;
    uint32_t* tri;         // 3 per triangle
    uint64_t vcap, tcap;   // capacities (vertices, triangles)
    uint64_t* counters;    // Counter
    // dense slab
    uint64_t* actbits;     // bit c % 64 of word c / 64 = cell c has a vertex
    SlabBits bits;         // the same words with their prefix tables
    uint32_t* tcount;      // triangles per kBlock vertices, and their offsets
    uint32_t* toffset;
};

// ---- launchers (kernels.hip) ----
hipError_t launch_eval_lattice(hipStream_t s, const s2m_op* ops, uint32_t nops, const float* cx,
                               const float* cy, const float* cz, uint32_t nx, uint32_t ny,
                               uint32_t lz0, uint32_t nzl, uint32_t pitch, float* lat);
// The dense slab's kernels (kernels.hip, bodies in device_dense.h and device_bricks.h).  host_ops: the host copy
// of the tape (it selects the kernel); op: the Mandelbulb op whose signs were decided early
// (sign_early), NULL where the sign pass has kept the values.
struct BrickArgs;
bool mandel_power8(const s2m_op* ops, uint32_t n);  // the tape is one power-8 Mandelbulb op
bool sign_early(const s2m_op* ops, uint32_t n, uint64_t points);  // its signs are decided early (no values to keep)
dim3 sign_grid(const BrickArgs& a);                 // blocks of 256
uint32_t sign_run(uint64_t bricks, const s2m_op* ops, uint32_t nops);  // BrickArgs::run
hipError_t launch_signs(hipStream_t s, const BrickArgs& a, const s2m_op* host_ops, const s2m_op* ops, uint32_t nops,
                        bool early);
hipError_t launch_find_bricks(hipStream_t s, const BrickArgs& a);
hipError_t launch_contour(hipStream_t s, const BrickArgs& a, const s2m_op* op);
hipError_t launch_emit(hipStream_t s, const BrickArgs& a, const s2m_op* op);
hipError_t launch_normals(hipStream_t s, const s2m_op* host_ops, const s2m_op* ops, uint32_t nops, float eps,
                          const MeshBufs& b);
hipError_t launch_ranks(hipStream_t s, const MeshBufs& b, uint32_t ncells);
hipError_t launch_dense_begin(hipStream_t s, uint64_t* counters, uint32_t ncounters, uint64_t* words, uint32_t ncells,
                              const void* host_tables, void* tables, size_t bytes, uint32_t* cbase);
hipError_t launch_slab_end(hipStream_t s, uint64_t* counters, uint32_t ncounters, uint64_t* words, uint32_t ncells,
                           uint32_t* cbase);
hipError_t launch_copy_out(hipStream_t s, const CopyList& c);
hipError_t launch_quads(hipStream_t s, const SlabArgs& a, const MeshBufs& b, const SlabBits& prev, uint64_t* snap,
                        uint64_t* back);
// cnt[0..4) (zeroed by the caller): k_sincos_check's mismatch counts.
hipError_t launch_sincos_check(hipStream_t s, uint64_t* cnt);
// cnt[0..2) (zeroed by the caller): k_bailout_check's comparisons and disagreements.
hipError_t launch_bailout_check(hipStream_t s, uint64_t* cnt);
// A tape just copied to the device: every Mandelbulb op's f[3] set to the bailout
// threshold of its f[1] (sd_mandelbulb reads it there instead of computing it per point).
hipError_t launch_tape_prepare(hipStream_t s, s2m_op* ops, uint32_t n);
// cus: compute units of the device; tile_blocks: most blocks of a k_sp_tiles launch (each
// holds a staging chunk); general_tiles: some tile's pruned program may not be a left fold
// (false when every job's whole program is one: its pruned programs are then left folds).
hipError_t launch_sparse_pass(hipStream_t s, SpPass P, const MeshBufs& b, int cus,
                              uint32_t tile_blocks, bool general_tiles, int boundary_plane, hipEvent_t* marks);
// Contour corner values given per cell (test hook): cells of the slab read their 8
// corners from `corners` (8 floats per cell, cells in (z,y,x) order from plane z0).
hipError_t launch_cells_from_corners(hipStream_t s, const SlabArgs& a, const float* corners,
                                     const MeshBufs& b, int emit);

// ---- no-allocation scratch (kernels.hip) ----
constexpr size_t kNoAllocScratchBytes = (size_t)S2M_NOALLOC_SCRATCH_BYTES;
constexpr uint32_t kMaxDevices = 64;
// Device address of the scratch array on `device`, which must be the current device.
// Looked up once per device (hipGetSymbolAddress); later calls return the kept address
// and the first lookup's status.
hipError_t noalloc_scratch(int device, void** ptr);

// ---- host memory for results (hostmem.cpp) ----
// Host memory for a result array: page-locked and recycled when large, malloc otherwise.
// Returned to the pool (or freed) by host_release; any other pointer is passed to free().
void* host_alloc(size_t bytes);
// Whether the device can write the block host_alloc returned (page-locked).
bool host_is_pinned(const void* p);
// A page-locked block shared by `refs` results: each points somewhere inside it and is
// released with host_release; the block returns to the pool after the last release.
void* host_alloc_shared(size_t bytes, uint32_t refs);
void host_release(void* p);

// ---- autotuner table (tune.cpp) ----
// Shapes the meshing calls use instead of their rules (0 = no choice for that knob).
struct TuneChoice {
    uint32_t stream_passes = 0;  // z-passes of a single tile-sparse job streamed to host memory
    uint32_t dense_slab = 0;     // cell planes per slab of the dense path
    uint64_t batch_cells = 0;    // most cells per pass of a batch
};
// The calling thread's override while s2m_tune times a candidate, else the table's entry.
bool tune_lookup(const std::string& key, TuneChoice* out);
// The table's entry only, with the time it was chosen for.
bool tune_cached(const std::string& key, TuneChoice* out, double* ms);
void tune_store(const std::string& key, const TuneChoice& c, double ms);
void tune_override(const TuneChoice* c);  // NULL: back to the table
// Index of the chosen candidate: the first one, replaced by any later one faster by more
// than 2 % (so a choice depends only on the timings and their order).
uint32_t tune_pick(const double* ms, uint32_t n);

// ---- host helpers (api.cpp) for the server ----
// A program from a gfx950 code object holding the s2m_c_* kernels (frontend_emit.cpp).
int program_from_code_object(s2m_ctx* ctx, const void* code, size_t size, s2m_program** out);
s2m_program* program_view(int device, const s2m_op* host_ops, uint32_t n, const s2m_op* d_ops);
hipStream_t context_stream(s2m_ctx* ctx);
bool tape_valid(const s2m_op* ops, uint32_t n);
int job_geometry(const s2m_params* p, uint32_t res[3], uint32_t* nz_cells);
int set_error(int code, const char* msg);
// Whether a request of the program (or tape `ops`) meshes alone on the dense path, by the
// rule s2m_mesh_batch uses (compiled, S2M_DENSE_EVAL, or a Mandelbulb above 128^3).
bool dense_request(const s2m_program* prog, const s2m_op* ops, uint32_t n, const s2m_params* p);
// Estimated device bytes of a dense job (working buffers of its slabs + outputs).
uint64_t dense_request_bytes(const s2m_params* p);
int program_device(const s2m_program* prog);

}  // namespace s2m
