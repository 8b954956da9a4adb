"""Node passes at the edges of their blocks, bit-compared with the oracle: grids
one to three words wide whose planes end just before, at and after the runs of
62 and 248 FCC words, the 256-word chunks of the Cartesian pass and the 64-word
blocks of the PartialNode expansion, filled with an open triangle soup (every
kind of boundary pattern)."""
import numpy as np
import pytest

import voxelizer_amd as va
from voxelizer_amd import workloads as W

pytestmark = pytest.mark.gpu


# Extents in voxels: x gives 1, 2 or 3 words per row (x + 3 rounded up to 32),
# y and z give y + 3 and z + 3 rows and planes.
@pytest.mark.parametrize("ext", [(29, 28, 5), (29, 29, 6), (29, 121, 3), (29, 122, 9),
                                 (61, 28, 4), (61, 61, 1), (93, 40, 7), (93, 83, 2)])
@pytest.mark.parametrize("kind", [va.NODE_SHORT, va.NODE_LONG, va.NODE_PARTIAL,
                                  va.NODE_SHORT_FCC, va.NODE_LONG_FCC])
def test_node_block_edges_match_oracle(gpu_ctx, oracle, ext, kind):
    m = W.random_soup(seed=sum(ext), n_tris=70)
    lo, hi = m.vertices.min(0), m.vertices.max(0)
    m.vertices = ((m.vertices - lo) / (hi - lo) * np.array(ext)).astype(np.float32)
    gpu_ctx.set_mesh(m.vertices, m.indices)
    gpu_ctx.set_materials(m.materials, 9)
    g = gpu_ctx.plan_grid(va.PLAN_CUBE_LENGTH, 1.0)
    og = oracle.plan_grid(m.vertices, va.PLAN_CUBE_LENGTH, 1.0)
    assert g.same(og)
    print(f"edges {ext} kind {kind}", flush=True)
    got = gpu_ctx.voxelize_nodes(g, kind, True)
    assert np.array_equal(got, oracle.voxelize_nodes(m, og, kind, True))
