"""Vertex merging at query counts that leave batches, rounds and groups partly filled, for each number
of lanes per range search, against the CPU restatement. Both sum a pixel's photons in single precision
in different orders (up to some hundred terms of one sign): 100 x 2^-24 = 6e-6 relative."""
import numpy as np
import pytest

import oracle as O
from selas_amd import native as N
from selas_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def scene(gpu_ctx):
    sc = W.sized_vcm_scene(5, 1e4, textures=False)
    s = N.build_render_scene(gpu_ctx, sc)
    yield sc, s, O.RenderScene(sc)
    s.release()


@pytest.mark.parametrize("lanes", [8, 16, 32])
@pytest.mark.parametrize("w,h", [(1, 1), (5, 3), (16, 1), (17, 1), (13, 10), (65, 33)])
def test_partly_filled_batches_match_oracle(gpu_ctx, scene, lanes, w, h):
    sc, s, rs = scene
    radius = 4.0 * sc["merge_radius"]  # few photons at these sizes: a wide radius still merges
    before = gpu_ctx.tuning()["vcm_merge_lanes"]
    gpu_ctx.set_tuning(vcm_merge_lanes=lanes)
    try:
        got = N.render_vcm(s, sc["camera"], w, h, 3, 8, radius, sc["radius_alpha"], 7)
    finally:
        gpu_ctx.set_tuning(vcm_merge_lanes=before)
    want, _ = O.render_vcm(rs, sc["camera"], w, h, 3, 8, radius, sc["radius_alpha"], 7)
    np.testing.assert_allclose(got.reshape(-1), np.asarray(want).reshape(-1), rtol=6e-6, atol=1e-6 * max(1e-6, float(np.max(want))))


@pytest.mark.parametrize("order", [0, N.ORDER_MERGE_CELLS])
@pytest.mark.parametrize("lanes", [8, 16, 32])
@pytest.mark.parametrize("w,h", [(101, 102), (145, 146), (205, 206), (300, 300)])
def test_batches_of_every_size_match_oracle(gpu_ctx, scene, lanes, w, h, order):
    """Counts between which a wave's batch grows by a round: one round holds 64 / lanes queries and 5,120
    waves are resident on 256 CUs, so 16 lanes take 1 to 4 rounds and 32 lanes 2 to 8 over these sizes
    (nearly every first-bounce ray hits and asks)."""
    sc, s, rs = scene
    radius = 2.0 * sc["merge_radius"]
    before = gpu_ctx.tuning()
    gpu_ctx.set_tuning(vcm_merge_lanes=lanes, vcm_order=order)
    try:
        got = N.render_vcm(s, sc["camera"], w, h, 1, 4, radius, sc["radius_alpha"], 7)
    finally:
        gpu_ctx.set_tuning(vcm_merge_lanes=before["vcm_merge_lanes"], vcm_order=before["vcm_order"])
    want, _ = O.render_vcm(rs, sc["camera"], w, h, 1, 4, radius, sc["radius_alpha"], 7)
    np.testing.assert_allclose(got.reshape(-1), np.asarray(want).reshape(-1), rtol=6e-6, atol=1e-6 * max(1e-6, float(np.max(want))))
