"""The brick pass off its usual path, bit-compared with the oracle: its list, and
coordinates, voxel lengths and normals too large or too small for the reciprocal
divisions (whole grids, and single triangles of a grid), and matSplitRes
intervals that end inside a brick."""
import numpy as np
import pytest

import voxelizer_amd as va
from voxelizer_amd import workloads as W

pytestmark = pytest.mark.gpu


def check(ctx, oracle, m, dim, mat_split=va.DEFAULT_MAT_SPLIT):
    ctx.set_mesh(m.vertices, m.indices)
    ctx.set_materials(m.materials, 8)
    g = ctx.plan_grid(va.PLAN_MAX_DIMENSION, dim)
    og = oracle.plan_grid(m.vertices, va.PLAN_MAX_DIMENSION, dim)
    assert g.same(og)
    got = ctx.voxelize_nodes(g, va.NODE_SHORT, True, mat_split=mat_split)
    ref = oracle.voxelize_nodes(m, og, va.NODE_SHORT, True, mat_split=mat_split)
    assert np.array_equal(got, ref)


def rough(subdiv, scale, offset=0.0):
    m = W.icosphere(seed=4, subdiv=subdiv)
    m.vertices = ((m.vertices.astype(np.float64) + offset) * scale).astype(np.float32)
    return m


@pytest.mark.parametrize("dim", [37, 126])
@pytest.mark.parametrize("subdiv", [2, 4])
@pytest.mark.parametrize("log2_scale,offset", [
    (0, 0.0), (0, 900.0), (23, 0.0), (26, 0.0), (40, 0.0),  # up to 2^24 and past it
    (-12, 0.0), (-16, 0.0), (-24, 0.0), (-40, 0.0),         # normals, then voxel lengths
])
def test_scales_match_oracle(gpu_ctx, oracle, dim, subdiv, log2_scale, offset):
    print(f"2^{log2_scale} +{offset} subdiv {subdiv} dim {dim}", flush=True)
    check(gpu_ctx, oracle, rough(subdiv, 2.0 ** log2_scale, offset), dim)


@pytest.mark.parametrize("mat_split", [(9, 512, 512), (512, 7, 512), (512, 512, 5), (13, 11, 3)])
def test_split_inside_brick_matches_oracle(gpu_ctx, oracle, mat_split):
    check(gpu_ctx, oracle, rough(1, 1.0), 61, mat_split)


def test_slivers_match_oracle(gpu_ctx, oracle):
    """Triangles with tiny normals (beside large ones) take the divisions one by one."""
    m = W.icosphere(seed=7, subdiv=2)
    rng = np.random.default_rng(3)
    n, base = 40, m.nv
    a = rng.random((n, 3)) * 0.7 - 0.35
    d = rng.standard_normal((n, 3)) * 0.1
    eps = rng.standard_normal((n, 3)) * 2.0 ** -rng.integers(18, 44, (n, 1)).astype(np.float64)
    v = np.stack([a, a + d, a + 0.5 * d + eps], 1).reshape(-1, 3).astype(np.float32)
    m.vertices = np.concatenate([m.vertices, v])
    m.indices = np.concatenate(
        [m.indices.reshape(-1, 3), (base + np.arange(3 * n, dtype=np.uint32)).reshape(-1, 3)])
    m.materials = np.concatenate([m.materials, rng.integers(1, 8, n).astype(np.uint8)])
    check(gpu_ctx, oracle, m, 90)


@pytest.mark.parametrize("ext", [(20, 1, 1), (20, 9, 17), (61, 150, 150), (200, 149, 301),
                                 (200, 161, 317), (200, 163, 325), (330, 201, 333)])
def test_brick_lists_match_oracle(gpu_ctx, oracle, ext):
    """Boxes whose shells take from one brick to about three per resident
    workgroup (1280), on either side of one each, so that the parts of the
    list are empty, short and of uneven length."""
    m = W.box(hi=ext, subdiv=3)
    m.materials = (1 + np.arange(m.nt) % 7).astype(np.uint8)
    gpu_ctx.set_mesh(m.vertices, m.indices)
    gpu_ctx.set_materials(m.materials, 8)
    g = gpu_ctx.plan_grid(va.PLAN_CUBE_LENGTH, 1.0)
    og = oracle.plan_grid(m.vertices, va.PLAN_CUBE_LENGTH, 1.0)
    assert g.same(og)
    got = gpu_ctx.voxelize_nodes(g, va.NODE_SHORT, True)
    assert np.array_equal(got, oracle.voxelize_nodes(m, og, va.NODE_SHORT, True))
