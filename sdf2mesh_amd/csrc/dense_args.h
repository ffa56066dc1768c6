// dense_args.h - arguments of the dense path's per-brick kernels (device_dense.h,
// device_bricks.h), shared by the host runtime, the library's kernels and the programs
// compiled at run time.
#pragma once
#ifndef __HIPCC_RTC__
#include <stdint.h>
#endif

namespace s2m {

// One slab's bricks, for the kernels of device_dense.h and device_bricks.h, or a part of them: bricks
// (bx0, by0) .. (bx0 + nbx, by0 + nby) of every layer, of which the first ownx and owny per axis
// are listed; what lies past those is the next parts', evaluated for the corners they share.
// Lattice cell (i, j, k) of the slab has its corners at lattice points i, i + 1 (and so on):
// a grid cell's two corner coordinates are neighbours in its axis table.  co*: grid cell
// of each lattice index, kNoCell where two corner coordinates a rounding apart lie
// between cells.
constexpr uint32_t kNoCell = 0xffffffffu;
struct BrickRec {          // a brick with a sign change among its cells' corners
    uint64_t mask;         // its cells (bit (z * 4 + y) * 4 + x): with a sign change, then with a vertex
    uint32_t base;         // first staged vertex
    uint16_t bx, by, bz, unused;
};
struct BrickArgs {
    const float* cx;       // coordinates of the corner lattice (whole axes)
    const float* cy;
    const float* cz;
    const uint32_t* cox;
    const uint32_t* coy;
    const uint32_t* coz;
    uint32_t nx, ny, nzl;  // lattice points of the slab per axis
    uint32_t lz0;          // lattice index of the slab's first plane
    uint32_t nbx, nby, nbz;
    uint32_t bx0, by0, ownx, owny;
    uint32_t run;          // bricks along x per wave of the sign kernel (a power of two, at most 16)
    uint32_t rx, ry;       // cells per row, rows per plane
    uint32_t z0, z1;       // cell planes of the slab
    uint64_t* words;       // [nbz][nby][nbx] sign words
    float* vals;           // the values (brick_vals), NULL for a sign pass that does not take them
    BrickRec* recs;
    uint64_t* alloc;       // records (low word) and staged vertices (high word) in use
    float* stage;          // 3 floats per staged vertex
    uint8_t* stage_sign;   // its sign bits
    uint32_t stage0;       // first staged vertex of the part
    uint32_t stage_cap;
    unsigned long long* actbits;  // bit c % 64 of word c / 64: cell c of the slab has a vertex
    const uint16_t* wpre;  // per word: vertices of the words before it in its block of 16
    const uint32_t* boffset;  // per block of 16 words (1024 cells): vertices before it in its chunk
    const uint32_t* cbase;    // per chunk of 1024 blocks: its first vertex
    float* vtx;            // 6 floats per vertex
    uint64_t* keys;
    uint8_t* signs;
    uint64_t vcap;
    float eps;
    uint32_t normals;      // 0: normals are written as zeros
};

}  // namespace s2m
