"""Interval bounds of the tile pruning (device_interval.h) against the fp32 evaluation
(device_sdf.h), both compiled for the host: at any point of a box the value a primitive or an
operator takes must lie within its bounds, and an operand that the bounds let stand for an
operator must be the operator's result bit for bit (zeros of either sign are one value).

The bounds are fp32 like the evaluation and use the hardware's square root and reciprocal,
which may be an ulp off: the host's stand-ins are moved by -1, 0 or 1 ulp at random.  Boxes
and shapes from 2^-40 to 2^40, boxes far off the shapes and the origin, thin and empty ones."""
import ctypes as C
import subprocess
import tempfile
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "sdf2mesh_amd" / "csrc"

STUB = """#pragma once
#include <math.h>
#include <stdint.h>
#include <stddef.h>
#include <string.h>
#define __device__
#define __forceinline__ inline
static inline uint32_t __float_as_uint(float f) { uint32_t u; memcpy(&u, &f, 4); return u; }
static inline float __uint_as_float(uint32_t u) { float f; memcpy(&f, &u, 4); return f; }
extern uint64_t rng_state;
static inline uint32_t rnd() { rng_state = rng_state * 6364136223846793005ull + 1442695040888963407ull; return (uint32_t)(rng_state >> 33); }
static inline float off_by_an_ulp(float v)
{
    if (!(fabsf(v) > 0.0f) || !(fabsf(v) < INFINITY)) return v;
    return __uint_as_float(__float_as_uint(v) + rnd() % 3u - 1u);
}
#define __builtin_amdgcn_sqrtf(x) off_by_an_ulp(sqrtf(x))
#define __builtin_amdgcn_rcpf(x) off_by_an_ulp(1.0f / (x))
#define __builtin_amdgcn_rsqf(x) (1.0f / sqrtf(x))
#define __builtin_amdgcn_logf(x) log2f(x)
"""

HARNESS = """
#include "hip/hip_runtime.h"
uint64_t rng_state;
#include "device_sdf.h"
#include "device_interval.h"
using namespace s2m;

static float uni(float a, float b) { return a + (b - a) * ((float)(rnd() & 0xffffffu) / 16777216.0f); }
static bool same(float a, float b) { return memcmp(&a, &b, 4) == 0 || (a == 0.0f && b == 0.0f); }

struct Prim { uint32_t code; float f[8]; };

static Prim shape(float s)  // of scale s around points of scale s
{
    Prim p;
    p.code = S2M_OP_SPHERE + rnd() % 5u;
    for (int i = 0; i < 8; ++i) p.f[i] = uni(-s, s);
    const int first = p.code == S2M_OP_CAPSULE ? 6 : 3;
    for (int i = first; i < 8; ++i) p.f[i] = uni(0.0f, s);
    const uint32_t u = rnd() % 16u;
    if (u == 0) for (int i = 0; i < 3; ++i) p.f[i] = 0.0f;             // at the origin
    if (u == 1) for (int i = 0; i < 3; ++i) p.f[i] *= 4096.0f;         // far off
    if (u == 2) for (int i = 3; i < 8; ++i) p.f[i] *= 1e-5f;           // thin, nearly a point
    if (u == 3 && p.code == S2M_OP_CAPSULE) for (int i = 0; i < 3; ++i) p.f[3 + i] = p.f[i] * (1.0f + 1e-6f);
    return p;
}

// Random folds of `ops` primitives over random boxes: checks[0] bounds, checks[1] operands that
// stand for an operator; returns the number of violations, the first one's numbers in `where`.
extern "C" long run(uint64_t seed, long folds, int points, int ops, long* checks, double* where)
{
    rng_state = seed * 0x9E3779B97F4A7C15ull + 1;
    long bad = 0;
    auto fail = [&](int kind, uint32_t code, float v, Iv b, float s) {
        if (bad++ == 0) { where[0] = kind; where[1] = code; where[2] = v; where[3] = b.lo; where[4] = b.hi; where[5] = s; }
    };
    for (long n = 0; n < folds; ++n) {
        const float s = ldexpf(uni(1.0f, 2.0f), (int)(rnd() % 80u) - 40);
        float bl[3], bh[3];
        const float size = s * ldexpf(1.0f, -(int)(rnd() % 12u)), off = rnd() % 8u ? s : 64.0f * s;
        for (int a = 0; a < 3; ++a) {
            bl[a] = uni(-off, off);
            bh[a] = rnd() % 16u ? bl[a] + uni(0.0f, size) : bl[a];
        }
        float pts[32][3], acc[32];
        for (int i = 0; i < points; ++i)
            for (int a = 0; a < 3; ++a) {
                const uint32_t u = rnd() % 4u;
                pts[i][a] = u == 0 ? bl[a] : u == 1 ? bh[a] : fminf(fmaxf(uni(bl[a], bh[a]), bl[a]), bh[a]);
            }
        Iv A = iv_unknown();
        for (int q = 0; q < ops; ++q) {
            Prim p = shape(s);
            if (rnd() % 3u == 0)  // near the box
                for (int a = 0; a < 3; ++a) p.f[a] = uni(bl[a] - size, bh[a] + size);
            const Iv P = iv_primitive(p.code, p.f, bl, bh);
            float v[32];
            for (int i = 0; i < points; ++i) {
                v[i] = eval_primitive(p.code, 0, p.f, pts[i][0], pts[i][1], pts[i][2]);
                ++checks[0];
                if (P.known && !(v[i] >= P.lo && v[i] <= P.hi)) fail(0, p.code, v[i], P, s);
            }
            if (q == 0) {
                A = P;
                for (int i = 0; i < points; ++i) acc[i] = v[i];
                continue;
            }
            const uint32_t code = S2M_OP_UNION + rnd() % 6u;
            const uint32_t u = rnd() % 8u;
            const float k = u == 0 ? 0.0f : u == 1 ? s * 1e-6f : uni(0.0f, s);
            const bool swap = rnd() & 1u;  // (folds with swapped operands)
            const Iv X = swap ? P : A, Y = swap ? A : P;
            int keep;
            const Iv R = iv_op(code, X, Y, k, keep);
            for (int i = 0; i < points; ++i) {
                const float x = swap ? v[i] : acc[i], y = swap ? acc[i] : v[i];
                const float r = apply_op(code, x, y, k);
                ++checks[0];
                if (R.known && !(r >= R.lo && r <= R.hi)) fail(1, code, r, R, s);
                if (keep != kKeepBoth) {
                    ++checks[1];
                    if (!same(r, keep == kKeepA ? x : y)) fail(2, code, r, R, s);
                }
                acc[i] = r;
            }
            A = R;
        }
    }
    return bad;
}
"""


@pytest.fixture(scope="module")
def harness():
    tmp = Path(tempfile.mkdtemp(prefix="s2m_iv_"))
    (tmp / "hip").mkdir()
    (tmp / "hip" / "hip_runtime.h").write_text(STUB)
    (tmp / "run.cpp").write_text(HARNESS)
    so = tmp / "run.so"
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-fno-fast-math", f"-I{tmp}", f"-I{CSRC}",
                    "-shared", "-fPIC", "-o", str(so), str(tmp / "run.cpp")], check=True)
    lib = C.CDLL(str(so))
    lib.run.restype = C.c_long
    lib.run.argtypes = [C.c_uint64, C.c_long, C.c_int, C.c_int, C.POINTER(C.c_long), C.POINTER(C.c_double)]
    return lib.run


@pytest.mark.parametrize("ops", [1, 2, 6, 40])
def test_bounds_hold_and_dropped_operands_do_not_count(harness, ops):
    checks, where = (C.c_long * 2)(), (C.c_double * 6)()
    bad = harness(7 + ops, 1_600_000 // ops, 6, ops, checks, where)
    print(f"{checks[0]} bounds, {checks[1]} replaced operators")
    assert bad == 0, f"{bad} violations, the first (kind, code, value, lo, hi, scale): {list(where)}"
    assert checks[0] > 4_000_000
    if ops > 1:
        assert checks[1] > 100_000
