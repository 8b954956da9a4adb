"""Meshes most of whose triangles have no candidates (degenerate, or outside the
slice or partition): outputs bit-compared with the oracle around the 256
triangles from which a block's candidates are searched for, and the time of a
call, which must not grow with where those triangles lie in the mesh."""
import time

import numpy as np
import pytest

import voxelizer_amd as va
from voxelizer_amd import workloads as W

pytestmark = pytest.mark.gpu


def sparse(runs, seed, flat=None):
    """Small triangles in the unit box in runs of (count, empty): an empty run's
    are degenerate, or with `flat` lie above that z."""
    rng = np.random.default_rng(seed)
    n = sum(k for k, _ in runs)
    top = 1.0 if flat is None else flat
    c = rng.random((n, 1, 3)) * [0.9, 0.9, 0.9 * top] + 0.05 * top
    v = c + rng.standard_normal((n, 3, 3)) * 0.02
    at, used = 0, []
    for k, empty in runs:
        if empty and flat is None:
            v[at:at + k, 1:] = v[at:at + k, :1]
        elif empty:
            v[at:at + k, :, 2] = top + (1.0 - top) * rng.random((k, 3))
        else:
            v[at:at + k, :, 2] = np.minimum(v[at:at + k, :, 2], top)
        used += [] if empty else [at, at + k - 1]
        at += k
    # The first and the last triangle that is not empty reach the box's corners.
    v[used[0]] = [[0, 0, 0], [0.1, 0.02, 0.1], [0, 0.1, 0]]
    v[used[-1]] = [[1, 1, 1], [0.9, 1, 1], [1, 0.9, 1]]
    v = np.clip(v, 0, 1).reshape(-1, 3).astype(np.float32)
    return W.Mesh(v, np.arange(3 * n, dtype=np.uint32).reshape(-1, 3),
                  rng.integers(1, 8, n).astype(np.uint8))


def load(ctx, oracle, m, dim):
    ctx.set_mesh(m.vertices, m.indices)
    ctx.set_materials(m.materials, 8)
    g = ctx.plan_grid(va.PLAN_MAX_DIMENSION, dim)
    og = oracle.plan_grid(m.vertices, va.PLAN_MAX_DIMENSION, dim)
    assert g.same(og)
    return g, og


@pytest.mark.parametrize("gap", [1, 253, 254, 255, 256, 257, 511, 70000])
@pytest.mark.parametrize("kind", [va.NODE_SHORT, va.NODE_LONG_FCC])
def test_gaps_match_oracle(gpu_ctx, oracle, gap, kind):
    """Candidates in a first, a middle and a last run; `gap` empty triangles
    around the middle one."""
    m = sparse([(40, False), (gap, True), (300, False), (gap, True), (3, False)], seed=gap)
    g, og = load(gpu_ctx, oracle, m, 40)
    print(f"gap {gap} kind {kind}", flush=True)
    assert np.array_equal(gpu_ctx.voxelize_nodes(g, kind, True),
                          oracle.voxelize_nodes(m, og, kind, True))


def test_slice_and_partition_of_a_large_mesh_match_oracle(gpu_ctx, oracle):
    m = sparse([(500, False), (60000, True), (900, False), (60000, True), (2, False)], seed=3,
               flat=0.1)
    g, og = load(gpu_ctx, oracle, m, 90)
    for axis, at in ((0, 30), (1, 40), (2, 3), (2, 7)):
        print(f"slice {axis} {at}", flush=True)
        a = (va.PLAN_MAX_DIMENSION, 90, va.NODE_LONG, axis, at, True, (1024, 1024))
        got, gd = gpu_ctx.voxelize_slice(*a)
        ref, rd = oracle.voxelize_slice(m, *a)
        assert gd == rd and np.array_equal(got, ref)
    for lo, hi in (((0, 2), (g.res[1], 5)), ((30, 0), (33, g.res[2]))):
        print(f"partition {lo} {hi}", flush=True)
        assert np.array_equal(gpu_ctx.voxelize_partition(g, va.NODE_SHORT, lo, hi, True),
                              oracle.voxelize_part(m, og, va.NODE_SHORT, lo, hi, True))


def test_time_does_not_depend_on_where_the_empty_triangles_lie(gpu_ctx, oracle):
    """The same 1500 triangles with two million empty ones before them all, and
    in their middle.  The second call may take half as long again; a walk over
    the two million takes several times as long."""
    n = 2_000_000
    best = []
    for runs in ([(n, True), (1500, False)], [(750, False), (n, True), (750, False)]):
        m = sparse(runs, seed=9)
        gpu_ctx.set_mesh(m.vertices, m.indices)
        g = gpu_ctx.plan_grid(va.PLAN_MAX_DIMENSION, 60)
        out = va.DeviceBuffer(gpu_ctx, 4 * (g.alloc[0] // 32) * g.alloc[1] * g.alloc[2])
        times = []
        for _ in range(12):
            gpu_ctx.sync()
            t = time.perf_counter()
            gpu_ctx.solid_bits_device(g, out.ptr.value)
            gpu_ctx.sync()
            times.append(time.perf_counter() - t)
        out.free()
        best.append(min(times))
    print(f"{best[0] * 1e6:.0f} and {best[1] * 1e6:.0f} us", flush=True)
    assert best[1] < 1.5 * best[0]
