"""The solid fill at row widths around its 64-word steps and at tiles whose triangles
pass few, many or all of their centres, bit-compared with the oracle."""
import numpy as np
import pytest

import voxelizer_amd as va
from voxelizer_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("words", [1, 5, 16, 31, 33, 63, 64, 65, 100, 1023, 1024])
@pytest.mark.parametrize("layers", [1, 3, 70])
def test_row_widths_match_oracle(gpu_ctx, oracle, words, layers):
    """`layers` squares across x over 6 x 9 rows, and small triangles on them."""
    rng = np.random.default_rng(words + layers)
    ext = np.array([words * 32 - 3, 6, 9], float)
    x = np.sort(rng.uniform(0, ext[0], layers + 1))
    x[0], x[-1] = 0.0, ext[0]
    v, t = [], []
    for k in range(layers):
        q = np.array([[x[k], 0, 0], [x[k], ext[1], 0], [x[k + 1], ext[1], ext[2]],
                      [x[k + 1], 0, ext[2]]])
        t += [[4 * k, 4 * k + 1, 4 * k + 2], [4 * k, 4 * k + 2, 4 * k + 3]]
        v.append(q)
    c = rng.random((40, 1, 3)) * ext
    small = np.clip(c + rng.standard_normal((40, 3, 3)), 0, ext).reshape(-1, 3)
    t = np.array(t + (4 * layers + np.arange(120).reshape(-1, 3)).tolist(), np.uint32)
    m = W.Mesh(np.concatenate(v + [small]).astype(np.float32), t)
    gpu_ctx.set_mesh(m.vertices, m.indices)
    g = gpu_ctx.plan_grid(va.PLAN_CUBE_LENGTH, 1.0)
    og = oracle.plan_grid(m.vertices, va.PLAN_CUBE_LENGTH, 1.0)
    assert g.same(og)
    print(f"words {words} layers {layers}", flush=True)
    got = gpu_ctx.solid_bits(g)
    assert np.array_equal(got, oracle.solid_bits(m, og))
