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


def test_top_tree_of_many_instances(gpu_ctx):
    """Every one of 300,000 instances is found: the top tree's last level is collapsed in several parts
    (131,072 tasks at a time)."""
    n, side = 300000, 550
    model = N.Scene(gpu_ctx)
    model.add_soup(np.array([[0.2, 0, 0.2, 0.8, 0, 0.2, 0.2, 0, 0.8], [0.8, 0, 0.8, 0.2, 0, 0.8, 0.8, 0, 0.2]], np.float32))
    model.commit()
    top = N.Scene(gpu_ctx)
    at = np.stack([np.arange(n) % side, np.zeros(n), np.arange(n) // side], 1).astype(np.float32)
    m = np.eye(4, dtype=np.float32).T.copy().reshape(-1)
    for k in range(n):
        m[12:15] = at[k]
        N.check(N.lib.sgpu_scene_add_instance(top.handle, model.handle, N.fptr(m), None))
    top.commit()
    rng = np.random.default_rng(1)
    o = at + np.stack([rng.uniform(0.25, 0.75, n), np.full(n, 5.0), rng.uniform(0.25, 0.75, n)], 1)
    full = lambda v: np.full(n, v, np.float32)
    rays = {"org_x": o[:, 0], "org_y": o[:, 1], "org_z": o[:, 2], "dir_x": full(0), "dir_y": full(-1), "dir_z": full(0),
            "tnear": full(0), "tfar": full(np.inf)}
    dr, dh = N.DeviceRays(gpu_ctx, rays), N.DeviceHits(gpu_ctx, n, with_inst=True)
    top.intersect(dr, dh)
    N.synchronize()
    top.check()
    got = dh.to_host()
    top.release()
    model.release()
    assert np.array_equal(got["inst_id0"], np.arange(n, dtype=np.uint32))
    np.testing.assert_allclose(got["t"], 5.0, rtol=1e-6)
