"""The device tree build at the sizes where its passes have remainders: blocks of 256 leaves in the
box pyramid, levels that do not halve evenly, the smallest trees. A box that missed one of its
triangles would lose hits, so hits are compared bit for bit with brute force."""
import numpy as np
import pytest

import oracle as O
from selas_amd import native as N
from selas_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 3, 5, 9, 255, 256, 257, 511, 513, 4095, 65537])
def test_tree_of_every_remainder_keeps_its_hits(gpu_ctx, n):
    t9 = N.gen_cluster_soup(n, -(-n // 32), 32, 0.2, 2e-2, 3e-1)[:n]
    n_rays = 64 if n > 4096 else 2048
    cam = N.gen_camera_rays(W.CAMERA_POS, W.CAMERA_LOOK_AT, W.CAMERA_UP, 50.0, 8, 8, 1)
    bounce = N.gen_bounce_rays(n, t9, n_rays)
    rays = {k: np.concatenate([cam[k], bounce[k]]) for k in N.RAY_FIELDS}
    scene = N.Scene(gpu_ctx)
    scene.add_soup(t9)
    scene.commit()
    dr, dh = N.DeviceRays(gpu_ctx, rays), N.DeviceHits(gpu_ctx, rays["org_x"].shape[0])
    scene.intersect(dr, dh)
    N.synchronize()
    scene.check()
    got = dh.to_host()
    scene.release()
    want = O.closest_brute_f32(t9, rays)
    assert np.array_equal(got["prim_id"], want["prim"])
    for k in ("t", "u", "v"):
        assert np.array_equal(got[k].view(np.uint32), want[k].view(np.uint32)), k
