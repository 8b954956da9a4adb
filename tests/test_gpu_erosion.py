"""Erosion of open sheets, whose removals travel from their free edges across the
blocks of 256 words and 8 planes, bit-compared with the oracle: tilted squares
of every dominant axis, rows of 1 to 9 words, one or several erosion subspaces."""
import numpy as np
import pytest

import voxelizer_amd as va
from voxelizer_amd import workloads as W

pytestmark = pytest.mark.gpu


def sheets(ext, seed):
    """Three tilted squares (one per axis) over a box of `ext` voxels."""
    rng = np.random.default_rng(seed)
    v, t = [], []
    for a in range(3):
        u, w = (a + 1) % 3, (a + 2) % 3
        q = np.zeros((4, 3))
        q[[1, 2], u] = 1.0
        q[[2, 3], w] = 1.0
        slope = rng.uniform(0.05, 0.9, 2)
        q[:, a] = q[:, u] * slope[0] + q[:, w] * slope[1] * (1.0 - slope[0])
        t += [[4 * a, 4 * a + 1, 4 * a + 2], [4 * a, 4 * a + 2, 4 * a + 3]]
        v.append(q)
    v = np.concatenate(v)
    v = (v - v.min(0)) / (v.max(0) - v.min(0)) * np.array(ext)
    return W.Mesh(v.astype(np.float32), np.array(t, np.uint32),
                  rng.integers(1, 8, 6).astype(np.uint8))


@pytest.mark.parametrize("ext", [(29, 29, 6), (29, 300, 40), (61, 90, 75), (90, 61, 5),
                                 (157, 120, 77), (250, 40, 100)])
@pytest.mark.parametrize("split", [(1024, 512, 512), (1024, 37, 29)])
def test_sheets_match_oracle(gpu_ctx, oracle, ext, split):
    m = sheets(ext, seed=sum(ext))
    gpu_ctx.set_mesh(m.vertices, m.indices)
    gpu_ctx.set_materials(m.materials, 8)
    g = gpu_ctx.plan_grid(va.PLAN_CUBE_LENGTH, 1.0)
    og = oracle.plan_grid(m.vertices, va.PLAN_CUBE_LENGTH, 1.0)
    assert g.same(og)
    print(f"sheets {ext} split {split}", flush=True)
    got = gpu_ctx.voxelize_nodes(g, va.NODE_SHORT, True, split)
    assert np.array_equal(got, oracle.voxelize_nodes(m, og, va.NODE_SHORT, True, split))
