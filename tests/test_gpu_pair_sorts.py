"""The counting sorts of (triangle, tile) and (triangle, brick) pairs where their
blocks of 256 candidates and tiles of 4096 scan entries begin and end, bit-compared
with the oracle: triangles without candidates (degenerate, or outside) before,
between and after the others, one large triangle with many, and numbers of
triangles and of tiles just below, at and above the limits."""
import numpy as np
import pytest

import voxelizer_amd as va
from voxelizer_amd import workloads as W

pytestmark = pytest.mark.gpu


def soup(n, empty, seed):
    """n triangles over a box, `empty` of them degenerate at random places (a run
    at either end), after one triangle across the whole box."""
    rng = np.random.default_rng(seed)
    c = rng.random((n, 1, 3)) * 0.9 + 0.05
    v = c + rng.standard_normal((n, 3, 3)) * 0.02
    v[0] = [[0, 0, 0], [0.3, 1, 0], [1, 0.4, 1]]
    off = rng.choice(np.arange(1, n), empty, replace=False) if empty else np.array([], int)
    if empty > 8:
        off[:4], off[4:8] = np.arange(1, 5), np.arange(n - 4, n)
    v[off, 1:] = v[off, :1]
    v = np.clip(v, 0, 1).reshape(-1, 3).astype(np.float32)
    return W.Mesh(v, np.arange(3 * n, dtype=np.uint32).reshape(-1, 3),
                  rng.integers(1, 8, n).astype(np.uint8))


SIZES = [(1, 0, 5), (2, 1, 33), (255, 0, 40), (256, 0, 40), (257, 200, 40), (600, 580, 70),
         (4095, 100, 60), (4096, 4000, 60), (4097, 5, 97)]


@pytest.mark.parametrize("n,empty,dim,kind",
                         [(*s, k) for s in SIZES for k in (va.NODE_SHORT, va.NODE_LONG_FCC)] +
                         [(40, 30, 250, va.NODE_SHORT), (9000, 0, 300, va.NODE_LONG)])
def test_soups_match_oracle(gpu_ctx, oracle, n, empty, dim, kind):
    m = soup(n, empty, seed=n + dim)
    gpu_ctx.set_mesh(m.vertices, m.indices)
    gpu_ctx.set_materials(m.materials, 8)
    g = gpu_ctx.plan_grid(va.PLAN_MAX_DIMENSION, dim)
    og = oracle.plan_grid(m.vertices, va.PLAN_MAX_DIMENSION, dim)
    assert g.same(og)
    print(f"soup {n} empty {empty} dim {dim} kind {kind}", flush=True)
    got = gpu_ctx.voxelize_nodes(g, kind, True)
    assert np.array_equal(got, oracle.voxelize_nodes(m, og, kind, True))


@pytest.mark.parametrize("ext", [(60, 60, 4), (60, 60, 5), (60, 60, 6), (29, 125, 13), (29, 126, 14),
                                 (500, 3, 40), (3, 300, 3), (200, 140, 90)])
@pytest.mark.parametrize("kind", [va.NODE_SHORT, va.NODE_SHORT_FCC, va.NODE_PARTIAL])
def test_brick_choice_matches_oracle(gpu_ctx_auto, oracle, ext, kind):
    """Grids on either side of the rules that pick the brick (8 planes, padding)."""
    m = soup(300, 20, seed=sum(ext))
    m.vertices = (m.vertices * np.array(ext)).astype(np.float32)
    gpu_ctx_auto.set_mesh(m.vertices, m.indices)
    gpu_ctx_auto.set_materials(m.materials, 8)
    g = gpu_ctx_auto.plan_grid(va.PLAN_CUBE_LENGTH, 1.0)
    og = oracle.plan_grid(m.vertices, va.PLAN_CUBE_LENGTH, 1.0)
    assert g.same(og)
    print(f"brick {ext} kind {kind}", flush=True)
    ref = oracle.voxelize_nodes(m, og, kind, True)
    assert np.array_equal(gpu_ctx_auto.voxelize_nodes(g, kind, True), ref)


@pytest.fixture(scope="module")
def gpu_ctx_auto():
    ctx = va.Context(0)
    yield ctx
    ctx.close()
