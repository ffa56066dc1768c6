"""Edges of the GPU paths' dispatch rules and tilings, at the sizes where they can go wrong.

Positions, keys, sign bits, triangles and invalid-quad counts are compared for equality with
the oracle's, or with those of the general path of the same call: the paths evaluate the same
fp32 expressions, so no tolerance applies (normals against the oracle: 1e-5, as everywhere).
"""
import numpy as np
import pytest

import sdf2mesh_amd as s2m
from sdf2mesh_amd import tape
from test_gpu_parity import assert_same_mesh, reference_mesh
from test_gpu_readback import device_mesh_copied

pytestmark = pytest.mark.gpu


def same(a, b):
    assert len(a.vertices) == len(b.vertices)
    assert np.array_equal(a.vertices.view(np.uint32), b.vertices.view(np.uint32))
    assert np.array_equal(a.triangles, b.triangles)
    assert np.array_equal(a.cell_keys, b.cell_keys)
    assert np.array_equal(a.signs, b.signs)
    assert a.invalid_quads == b.invalid_quads


def grid(res, flags, slab=0):
    return s2m.Params((-1.0, -1.1, -0.9), (1.05, 1.0, 1.1), res, 1e-4, flags, slab)


# Dense slabs: lattice bricks of 4 (one cell, partial bricks, exact corners with two
# coordinates per cell face), brick words and ranks over runs of 64 cells, several slabs.
@pytest.mark.parametrize("res", [(1, 1, 1), (2, 3, 5), (3, 4, 8), (5, 9, 7), (17, 33, 12), (64, 65, 9)])
@pytest.mark.parametrize("flags", [0, s2m.CORNERS_EXACT | s2m.COMPAT_DROP_LAST_SLICE])
def test_dense_bricks(ctx, res, flags):
    node = tape.random_csg(3)
    for slab in (0, 1, 5):
        print(f"dense {res} flags={flags} slab={slab}", flush=True)
        p = grid(res, flags | s2m.DENSE_EVAL, slab)
        assert_same_mesh(ctx.mesh(ctx.program(node), p), reference_mesh(node, p))


# The Mandelbulb's signs decided early (bailout 1.5 .. 16, offset >= 0) and in full, against
# the interpreter: min(M, M) is M bit for bit and runs on the tape interpreter.
@pytest.mark.parametrize("iterations,bailout,offset,swap", [
    (8, 2.0, 0.003, True), (8, 1.5, 0.003, False), (8, 1.49, 0.003, True), (8, 16.0, 0.003, True),
    (8, 16.5, 0.003, True), (1, 2.0, 0.003, True), (2, 4.0, 0.0, True), (8, 2.0, -0.01, True),
    (40, 2.0, 0.05, False)])
def test_mandelbulb_signs(ctx, iterations, bailout, offset, swap):
    m = tape.mandelbulb(iterations, bailout=bailout, offset=offset, swap_yz=swap)
    for res, flags in (((72, 61, 67), 0), ((40, 40, 40), s2m.CORNERS_EXACT)):
        print(f"mandelbulb {iterations} {bailout} {offset} {swap} {res}", flush=True)
        p = grid(res, flags | s2m.DENSE_EVAL)
        same(ctx.mesh(ctx.program(m), p), ctx.mesh(ctx.program(tape.union(m, m)), p))


# Orbits of many steps: the derivative grows past 2^126, where the reciprocal the value takes is
# 0.  With offset 0 that decides the sign, so an early positive one would leave cells out.
@pytest.mark.parametrize("iterations,swap", [(256, True), (1024, False)])
def test_mandelbulb_signs_of_deep_orbits(ctx, iterations, swap):
    m = tape.mandelbulb(iterations, bailout=2.0, offset=0.0, swap_yz=swap)
    p = s2m.Params((-1.25,) * 3, (1.25,) * 3, (160, 160, 160), 1e-4, s2m.DENSE_EVAL)
    print(f"deep orbits {iterations}", flush=True)
    a, b = ctx.program(m), ctx.program(tape.union(m, m))
    same(ctx.mesh(a, p), ctx.mesh(b, p))


# Signs are decided early from 2^20 lattice points per iteration on: grids around that line and past
# it, with bailouts and offsets at their limits, and one whose orbits take 256 iterations.
@pytest.mark.parametrize("iterations,bailout,offset,swap,res", [
    (1, 2.0, 0.003, True, 100), (1, 2.0, 0.003, True, 101), (2, 4.0, 0.0, True, 131), (8, 2.0, 0.003, True, 202),
    (8, 2.0, 0.003, False, 203), (8, 1.5, 0.003, True, 206), (8, 16.0, 0.003, False, 206), (8, 2.0, 1.0, True, 206),
    (256, 2.0, 0.0, True, 646)])
def test_mandelbulb_early_signs(ctx, iterations, bailout, offset, swap, res):
    m = tape.mandelbulb(iterations, bailout=bailout, offset=offset, swap_yz=swap)
    a, b = ctx.program(m), ctx.program(tape.union(m, m))
    for flags in (0, s2m.CORNERS_EXACT) if res < 300 else (0,):
        print(f"early signs {iterations} {bailout} {offset} {swap} {res} {flags}", flush=True)
        p = s2m.Params((-1.25,) * 3, (1.25, 1.25, 1.2), (res, res, res), 1e-4, flags)
        same(ctx.mesh(a, p), ctx.mesh(b, s2m.Params(p.bb_min, p.bb_max, p.res, p.eps, flags | s2m.DENSE_EVAL)))


OPS = [tape.union, tape.intersection, tape.subtraction] + [
    (lambda f: lambda a, b: f(a, b, 0.08))(f)
    for f in (tape.smooth_union, tape.smooth_intersection, tape.smooth_subtraction)]


def parts(n, seed):
    rng = np.random.default_rng(seed)
    out = []
    for i in range(n):
        c = list(rng.uniform(-0.5, 0.5, 3))
        out.append([tape.sphere(c, rng.uniform(0.25, 0.5)), tape.box(c, list(rng.uniform(0.4, 0.9, 3))),
                    tape.torus(c, [0.4, 0.15]), tape.cylinder(c, 0.4, 0.3),
                    tape.capsule(c, [-x for x in c], 0.25)][(i + seed) % 5])
    return out


def right_nested(nodes, ops):
    node = nodes[-1]
    for i, n in enumerate(reversed(nodes[:-1])):
        node = ops[i % len(ops)](n, node)
    return node


# Trees that become folds by swapping operands (each operator keeps a primitive), with every
# operator outermost; a primitive joined to a fold from the left and from the right in turn.
@pytest.mark.parametrize("first", range(len(OPS)))
def test_swapped_folds(ctx, first):
    ops = OPS[first:] + OPS[:first]
    a = parts(7, first)
    nested = right_nested(a[:4], ops[::-1])
    for node in (nested, ops[0](ops[1](nested, a[4]), a[5]), ops[2](a[6], ops[0](ops[1](nested, a[4]), a[5]))):
        for res, flags in (((33, 40, 31), 0), ((24, 24, 24), s2m.REFERENCE_COMPAT)):
            print(f"swapped folds {first} {res}", flush=True)
            p = grid(res, flags)
            assert_same_mesh(ctx.mesh(ctx.program(node), p), reference_mesh(node, p))


# Trees that are no folds anywhere: operand stacks up to and past the depth at which several
# points share an op, one with a Mandelbulb; and programs past the staged length, alone and in
# a pass with short ones (lists by tile instead of by slot).
def unfoldable(depth, seed, leaf=None):
    a = parts(2 * depth + 2, seed)
    pairs = [tape.smooth_union(a[2 * i], a[2 * i + 1], 0.05) for i in range(depth + 1)]
    if leaf is not None:
        pairs[-1] = tape.union(pairs[-1], leaf)
    return right_nested(pairs, [tape.union, lambda x, y: tape.smooth_union(x, y, 0.1)])


def pairs_fold(n, seed):  # a left fold of pairs: two values below the top at most
    a = parts(2 * n, seed)
    return tape.fold([tape.smooth_union(a[2 * i], a[2 * i + 1], 0.05) for i in range(n)], tape.union)


# (at most 16 values on the operand stack)
GENERAL = [unfoldable(2, 1), unfoldable(7, 2), unfoldable(8, 3), unfoldable(13, 4),
           unfoldable(3, 5, tape.mandelbulb(3)), pairs_fold(32, 6), pairs_fold(40, 7),
           tape.fold(parts(64, 7)), tape.fold(parts(65, 8))]


@pytest.mark.parametrize("which", range(len(GENERAL)))
def test_general_trees(ctx, which):
    node = GENERAL[which]
    p = grid((25, 32, 30), s2m.COMPAT_DROP_LAST_SLICE)
    print(f"general tree {which}: {len(node.tape())} ops", flush=True)
    m = ctx.mesh(ctx.program(node), p)
    d = grid((25, 32, 30), s2m.COMPAT_DROP_LAST_SLICE | s2m.DENSE_EVAL)
    same(m, ctx.mesh(ctx.program(node), d))
    if which != 4:  # (the oracle's Mandelbulb differs in rounding)
        assert_same_mesh(m, reference_mesh(node, p))
    nodes = [GENERAL[which], tape.torus_example(), GENERAL[(which + 5) % len(GENERAL)]]
    progs = [ctx.program(n) for n in nodes]
    for b, prog in zip(ctx.mesh_batch(progs, [p] * 3), progs):
        same(b, ctx.mesh(prog, p))


# Folds and other slots in one launch up to 128 k tiles, in two above it.
@pytest.mark.parametrize("res", [(408, 400, 408), (416, 416, 408)])
def test_kinds_of_slots(ctx, res):
    prog = ctx.program(unfoldable(3, 11))
    print(f"both kinds {res}", flush=True)
    a = ctx.mesh(prog, grid(res, 0))
    same(a, device_mesh_copied(ctx, prog, grid(res, 0)))
    same(a, ctx.mesh(prog, grid(res, s2m.DENSE_EVAL)))


# Rows (z, y) around the 4096-row chunks of the offset scan and its waves' 1024 rows, and
# fewer rows than lanes.
@pytest.mark.parametrize("res", [(9, 1, 1), (16, 7, 9), (8, 31, 33), (8, 32, 32), (9, 63, 65), (8, 64, 64),
                                 (8, 17, 241), (12, 91, 91)])
def test_row_scan(ctx, res):
    node = tape.csg64()
    print(f"row scan {res}", flush=True)
    p = grid(res, 0)
    assert_same_mesh(ctx.mesh(ctx.program(node), p), reference_mesh(node, p))


# Meshes that a kernel writes to host memory (2 MB in all, arrays below 256 KB staged) and
# larger ones: around both limits, against the device-resident mesh copied afterwards.
@pytest.mark.parametrize("res", [24, 80, 84, 88, 92, 112, 120, 152, 160, 168, 200])
def test_small_meshes_land(ctx, res):
    prog = ctx.program(tape.torus_example())
    p = grid((res, res, res), 0)
    a = ctx.mesh(prog, p)
    print(f"land {res}: {len(a.vertices)} vertices", flush=True)
    same(a, device_mesh_copied(ctx, prog, p))
    b = ctx.mesh_to_host(prog, p)
    assert np.array_equal(np.asarray(b.vertices()).view(np.uint32).reshape(-1, 6), a.vertices.view(np.uint32))
    assert np.array_equal(np.asarray(b.triangles()).reshape(-1, 3), a.triangles)


# Boxes with an axis (or all) running from its maximum to its minimum: the coordinate tables
# descend, and the intervals of bricks, tiles and super-tiles are still ordered.
@pytest.mark.parametrize("axes", [(0,), (1,), (2,), (0, 1, 2)])
@pytest.mark.parametrize("flags", [0, s2m.CORNERS_EXACT])
def test_reversed_axes(ctx, axes, flags):
    a = parts(5, 2)
    lo, hi = [-1.0, -1.1, -0.9], [1.05, 1.0, 1.1]
    for k in axes:
        lo[k], hi[k] = hi[k], lo[k]
    for node in (tape.sphere((0.0, 0.0, 0.0), 0.5), tape.csg64(), right_nested(a, OPS[::-1]), unfoldable(3, 5)):
        print(f"reversed {axes} flags={flags} ops={len(node.tape())}", flush=True)
        p = s2m.Params(tuple(lo), tuple(hi), (70, 66, 72), 1e-4, flags)
        d = s2m.Params(tuple(lo), tuple(hi), (70, 66, 72), 1e-4, flags | s2m.DENSE_EVAL)
        m = ctx.mesh(ctx.program(node), p)
        assert len(m.vertices) > 0
        same(m, ctx.mesh(ctx.program(node), d))
        assert_same_mesh(m, reference_mesh(node, p))


# A dense job with more sign changes per slab than the first estimate of the staging buffer
# repeats once with the device's count; the context keeps that size, so the same job runs once
# when it comes again.  A cube in one slab, one in slabs, and one streamed to host memory.
@pytest.mark.parametrize("res,slab", [(64, 0), (96, 40), (188, 0)])
def test_staging_capacity_kept(res, slab):
    wave = """use sdf3d::*;
fn sdf3d(p: vec3f) -> f32 {
    let q = p * %s;
    return sin(q.x) * cos(q.y) + sin(q.y) * cos(q.z) + sin(q.z) * cos(q.x);
}
""" % tape.wgsl_float(0.6 * res)
    with s2m.Context(0) as fresh:
        prog = fresh.program_from_source(wave)
        p = s2m.Params.reference(res, 2.0, flags=0)
        p.slab = slab
        print(f"staging {res} slab={slab}", flush=True)
        first = fresh.mesh(prog, p)
        t = fresh.last_timing()
        assert t["eval_launches"] > t["slabs"]  # more than the estimate holds
        for _ in range(2):
            same(first, fresh.mesh(prog, p))
            t = fresh.last_timing()
            assert t["eval_launches"] == t["slabs"]
        fresh.mesh(prog, s2m.Params.reference(32, 2.0))
        same(first, fresh.mesh(prog, p))
        assert fresh.last_timing()["eval_launches"] == t["slabs"]
