"""The surface brick shape the grid decides on: set and read back, seen in the
number of (triangle, brick) pairs; and the shapes it picks, bit-compared with the
oracle where a shape could go wrong: slices, partitions, matSplitRes intervals
that end inside a brick, and bricks cut along z by the learned schedule."""
import threading
import time

import numpy as np
import pytest

import voxelizer_amd as va
from voxelizer_amd import workloads as W

pytestmark = pytest.mark.gpu

BY_GRID = (0, 0, 0)


@pytest.fixture(scope="module")
def ctx():
    c = va.Context(0)
    yield c
    c.close()


def load(ctx, m):
    ctx.set_mesh(m.vertices, m.indices)
    ctx.set_materials(m.materials, int(m.materials.max()) + 1)


def pairs(ctx, g, kind):
    ctx.enable_timing(True)
    ctx.voxelize_nodes(g, kind, True)
    n = ctx.stage_times()["surface_pairs"]
    ctx.enable_timing(False)
    return n


@pytest.mark.parametrize("ext,kind,picked,other", [
    ((5.0, 4.0, 3.0), va.NODE_SHORT, (32, 8, 16), (128, 4, 8)),
    ((5.0, 4.0, 0.1), va.NODE_SHORT, (32, 16, 8), (128, 4, 8)),
    ((5.0, 4.0, 3.0), va.NODE_LONG_FCC, (32, 8, 16), (64, 4, 4)),
])
def test_shape_set_and_read_back(ctx, ext, kind, picked, other):
    fcc = kind == va.NODE_LONG_FCC
    m = W.shoebox_room(seed=41, n_boxes=6, size=(5.0, 4.0, 3.0), subdiv=4)
    m.vertices = (m.vertices * (np.array(ext) / [5.0, 4.0, 3.0])).astype(np.float32)
    load(ctx, m)
    g = ctx.plan_grid(va.PLAN_CUBE_LENGTH, 0.03)
    assert ctx.brick_dims(fcc) == BY_GRID
    by_grid = pairs(ctx, g, kind)
    ctx.set_brick_dims(other, fcc)
    assert ctx.brick_dims(fcc) == other and pairs(ctx, g, kind) != by_grid
    ctx.set_brick_dims(picked, fcc)
    assert ctx.brick_dims(fcc) == picked and pairs(ctx, g, kind) == by_grid
    ctx.set_brick_dims(other, fcc)
    ctx.set_brick_dims(BY_GRID, fcc)
    assert ctx.brick_dims(fcc) == BY_GRID and pairs(ctx, g, kind) == by_grid
    with pytest.raises(va.VoxError):
        ctx.set_brick_dims((0, 8, 16), fcc)
    assert ctx.brick_dims(fcc) == BY_GRID


@pytest.mark.parametrize("brick", [BY_GRID, (32, 8, 16), (32, 16, 8)])
@pytest.mark.parametrize("kind", [va.NODE_SHORT, va.NODE_LONG, va.NODE_PARTIAL, va.NODE_SHORT_FCC,
                                  va.NODE_LONG_FCC])
def test_shapes_match_oracle(ctx, oracle, kind, brick):
    m = W.shoebox_room(seed=31, n_boxes=12, subdiv=3)
    load(ctx, m)
    g = ctx.plan_grid(va.PLAN_CUBE_LENGTH, 0.037)
    og = oracle.plan_grid(m.vertices, va.PLAN_CUBE_LENGTH, 0.037)
    fcc = kind in (va.NODE_SHORT_FCC, va.NODE_LONG_FCC)
    ctx.set_brick_dims(brick, fcc)
    try:
        for ms in (va.DEFAULT_MAT_SPLIT, (13, 11, 7), (512, 512, 5)):
            print(f"kind {kind} brick {brick} mat split {ms}", flush=True)
            assert np.array_equal(ctx.voxelize_nodes(g, kind, True, mat_split=ms),
                                  oracle.voxelize_nodes(m, og, kind, True, mat_split=ms)), ms
    finally:
        ctx.set_brick_dims(BY_GRID, fcc)


@pytest.mark.parametrize("kind", [va.NODE_SHORT, va.NODE_LONG])
def test_slices_and_partitions_match_oracle(ctx, oracle, kind):
    m = W.shoebox_room(seed=8, n_boxes=16, subdiv=3)
    load(ctx, m)
    mode, param = va.PLAN_CUBE_LENGTH, 0.025
    for axis in range(3):
        for at in (1, 58, 119):
            print(f"slice {axis} {at} kind {kind}", flush=True)
            a = (mode, param, kind, axis, at, True, (1024, 1024), (33, 20))
            got, gd = ctx.voxelize_slice(*a)
            ref, rd = oracle.voxelize_slice(m, *a)
            assert gd == rd and np.array_equal(got, ref)
    g = ctx.plan_grid(mode, param)
    og = oracle.plan_grid(m.vertices, mode, param)
    ry, rz = g.res[1], g.res[2]
    for lo, hi in (((0, 0), (ry // 2, rz // 2)), ((ry // 3, rz // 4), (2 * ry // 3, 3 * rz // 4)),
                   ((0, rz - 1), (ry, rz)), ((5, 0), (6, rz)), ((7, 20), (ry, 26))):
        print(f"partition {lo} {hi} kind {kind}", flush=True)
        assert np.array_equal(ctx.voxelize_partition(g, kind, lo, hi, True),
                              oracle.voxelize_part(m, og, kind, lo, hi, True))


@pytest.mark.parametrize("kind,brick", [(va.NODE_SHORT, BY_GRID), (va.NODE_LONG, (32, 16, 8)),
                                        (va.NODE_PARTIAL, BY_GRID), (va.NODE_LONG_FCC, BY_GRID)])
def test_cut_bricks_match_oracle(ctx, oracle, kind, brick):
    """Every listed brick predicted heavy, so each is cut into four along z."""
    m = W.shoebox_room(seed=23, n_boxes=16, subdiv=3)
    load(ctx, m)
    ctx.cost_record(True)
    g = ctx.plan_grid(va.PLAN_CUBE_LENGTH, 0.012)
    ctx.voxelize_nodes(g, va.NODE_SHORT, True)
    f, c = ctx.cost_samples()
    ctx.cost_record(False)
    ctx.cost_train(f, c, epochs=5, batch=128, lr=3e-3, seed=2)
    fcc = kind == va.NODE_LONG_FCC
    d = 0.02 if fcc else 0.012
    g, og = ctx.plan_grid(va.PLAN_CUBE_LENGTH, d), oracle.plan_grid(m.vertices, va.PLAN_CUBE_LENGTH, d)
    try:
        ctx.set_brick_dims(brick, fcc)
        ctx.set_schedule(va.SCHEDULE_LEARNED)
        ctx.set_heavy_threshold(-1e6)
        ctx.set_screen_ratio(0.0)
        ctx.set_split_parts(4)
        ctx.enable_timing(True)
        got = ctx.voxelize_nodes(g, kind, True)
        used = ctx.stage_times()["learned_schedule"]
    finally:
        ctx.enable_timing(False)
        ctx.set_schedule(va.SCHEDULE_PLAIN)
        ctx.set_heavy_threshold(1.5)
        ctx.set_screen_ratio(24.0)
        ctx.set_split_parts(0)
        ctx.set_brick_dims(BY_GRID, fcc)
    assert used == 1
    assert np.array_equal(got, oracle.voxelize_nodes(m, og, kind, True))


def test_autotune_keeps_the_grids_shape_when_its_first_runs_are_slow():
    """The autotuner starts while another context keeps the device busy for about
    as long as one shape's three runs: the shape it keeps is no slower than the
    grid's own (the best of the hall's; the next is 7% slower)."""
    m = W.hall(seed=0)
    split = (1024, 1024, 1024)
    c, other = va.Context(0), va.Context(0)
    try:
        for x in (c, other):
            load(x, m)
        g = c.plan_grid(va.PLAN_CUBE_LENGTH, 1.0 / 64.0)
        n = c.node_count(g, va.NODE_SHORT)
        out, out2 = va.DeviceBuffer(c, n), va.DeviceBuffer(other, n)

        def call(x, o):
            t = time.perf_counter()
            x.voxelize_nodes_device(g, va.NODE_SHORT, o.ptr.value, True, split)
            x.sync()
            return time.perf_counter() - t

        def busy():
            end = time.perf_counter() + 0.008
            while time.perf_counter() < end:
                call(other, out2)

        call(other, out2)
        by_grid = min(call(c, out) for _ in range(10))
        load_thread = threading.Thread(target=busy)
        load_thread.start()
        dims, _ = c.autotune_bricks(g, va.NODE_SHORT, out.ptr.value, 2, split)
        load_thread.join()
        tuned = min(call(c, out) for _ in range(10))
        out.free()
        out2.free()
    finally:
        other.close()
        c.close()
    print(f"by the grid {by_grid * 1e6:.0f} us, tuned {dims} {tuned * 1e6:.0f} us", flush=True)
    assert tuned < 1.04 * by_grid
