"""Calls of vox_voxelize_nodes_noalloc near the end of its 128 MiB of scratch:
meshes with many (triangle, brick) pairs for their grid, whose lists fit with
wide bricks and no array beside them, and their nodes as vox_voxelize_nodes
writes them."""
import numpy as np
import pytest

import voxelizer_amd as va
from voxelizer_amd import workloads as W

pytestmark = pytest.mark.gpu


def mesh(v, seed):
    n = len(v)
    return W.Mesh(v.reshape(-1, 3).astype(np.float32), np.arange(3 * n, dtype=np.uint32).reshape(-1, 3),
                  np.random.default_rng(seed).integers(1, 8, n).astype(np.uint8))


def across(n):
    """n triangles across the whole box: every brick and every tile of it."""
    rng = np.random.default_rng(1)
    v = np.empty((n, 3, 3))
    v[:, 0], v[:, 1], v[:, 2] = [0, 0, 0], [1, 1, 0.5], [0.5, 0.2, 1]
    v[:, 1, 0], v[:, 2, 0] = 1.0, rng.random(n)
    return mesh(v * 254.0, 1), 1.0


def slivers(n):
    """n thin triangles along x: eight bricks of 32 voxels each, two of 128."""
    rng = np.random.default_rng(2)
    v = np.repeat(rng.random((n, 1, 3)) * [0, 28.5, 28.5], 3, axis=1) + rng.random((n, 3, 3)) * 0.3
    v[:, 0, 0], v[:, 1, 0], v[:, 2, 0] = 0.0, 254.0, 127.0
    v[0, :, 1:], v[1, :, 1:] = 0.0, 29.0
    return mesh(v, 2), 1.0


@pytest.mark.parametrize("make,n,kind", [(across, 1450, va.NODE_SHORT), (across, 1450, va.NODE_LONG),
                                         (slivers, 880000, va.NODE_SHORT)])
def test_calls_that_need_most_of_the_scratch(make, n, kind):
    m, d = make(n)
    ctx = va.Context(0)
    try:
        ctx.set_mesh(m.vertices, m.indices)
        ctx.set_materials(m.materials, 8)
        g = ctx.plan_grid(va.PLAN_CUBE_LENGTH, d)
        print(f"{make.__name__} {n} alloc {tuple(g.alloc)} kind {kind}", flush=True)
        split = (1024, 1024, 1024)
        ref = ctx.voxelize_nodes(g, kind, True, split)
        nb = ctx.node_count(g, kind) * va.NODE_SIZE[kind]
        out = va.DeviceBuffer(ctx, nb)
        for _ in range(2):  # the second call starts from the first one's scratch
            out.upload(np.full(nb, 0xA5, np.uint8))
            ctx.voxelize_nodes_noalloc_device(g, kind, out.ptr.value, True, split)
            assert np.array_equal(out.download(np.uint8, nb), ref)
        out.free()
    finally:
        ctx.close()
