"""The curve pass's 8-wide tree and its steps by many lanes at once, at the sizes where they have
remainders (one segment, fewer than a node's children, more than a block of leaves; ray counts that
leave waves partly filled), with rays aimed at the curves' axes at the joints of segments and between:
such rays do not graze, so every one hits, at the oracle's distance (1e-5 relative: the device searches
in float, the oracle in double), on the oracle's segment or, at a joint, the one that shares its ball."""
import numpy as np
import pytest

import oracle as O
from selas_amd import native as N

pytestmark = pytest.mark.gpu


def _strand(seed, n_seg):
    rng = np.random.default_rng(seed)
    d, p, pts = np.array([0.0, 1.0, 0.0]), np.zeros(3), []
    for _ in range(n_seg + 3):
        pts.append(p)
        d = d + 0.15 * rng.normal(size=3)
        d /= np.linalg.norm(d)
        p = p + 0.1 * d
    return np.concatenate([np.array(pts), np.full((n_seg + 3, 1), 0.01)], 1).astype(np.float32)


@pytest.mark.parametrize("n_seg,n_rays", [(1, 1), (1, 65), (2, 7), (3, 64), (8, 200), (9, 257), (257, 999), (600, 4097)])
def test_axis_rays_hit_where_the_oracle_says(gpu_ctx, n_seg, n_rays):
    verts, idx = _strand(n_seg, n_seg), np.arange(n_seg, dtype=np.uint32)
    rng = np.random.default_rng(n_rays)
    seg, u = rng.integers(0, n_seg, n_rays), np.where(rng.random(n_rays) < 0.5, 0.0, rng.random(n_rays))
    cp = verts[:, :3].astype(np.float64)
    b = np.stack([(1 - u) ** 3, 3 * u ** 3 - 6 * u ** 2 + 4, -3 * u ** 3 + 3 * u ** 2 + 3 * u + 1, u ** 3], 1) / 6
    axis = sum(b[:, j:j + 1] * cp[seg + j] for j in range(4))
    way = rng.normal(size=(n_rays, 3))
    way /= np.linalg.norm(way, axis=1, keepdims=True)
    o, d = (axis - 2.0 * way).astype(np.float32), way.astype(np.float32)
    rays = {"org_x": o[:, 0], "org_y": o[:, 1], "org_z": o[:, 2], "dir_x": d[:, 0], "dir_y": d[:, 1], "dir_z": d[:, 2],
            "tnear": np.zeros(n_rays, np.float32), "tfar": np.full(n_rays, np.inf, np.float32)}
    rays = {k: np.ascontiguousarray(v) for k, v in rays.items()}
    scene = N.Scene(gpu_ctx)
    scene.add_curves(verts, idx)
    scene.commit()
    dr, dh = N.DeviceRays(gpu_ctx, rays), N.DeviceHits(gpu_ctx, n_rays)
    scene.intersect(dr, dh)
    occ = gpu_ctx.empty(4 * n_rays)
    scene.occluded(dr, occ)
    N.synchronize()
    scene.check()
    got = dh.to_host()
    want = O.curves_closest(O.curve_segments({"curve_vertices": verts, "curves": idx}), dict(rays, tfar=np.full(n_rays, 1e30, np.float32)))
    assert (got["geom_id"] == 0).all() and (occ.download(np.uint32, n_rays) == 1).all()
    np.testing.assert_allclose(got["t"], want["t"], rtol=1e-5)
    gp, wp = got["prim_id"].astype(np.int64), want["prim"].astype(np.int64)
    joint = (np.abs(gp - wp) == 1) & ((got["u"] < 1e-2) | (got["u"] > 1 - 1e-2))
    assert ((gp == wp) | joint).all()
    scene.release()


@pytest.mark.parametrize("factor", [1, 5, 20])
def test_axis_rays_from_afar(gpu_ctx, factor):
    """The pass culls in single precision with a rounded reciprocal: rays whose origins are `factor` times
    the scene's largest coordinate away still hit every segment aimed at. (Their own rounding, half an ulp
    of the origin, is 2e-6 at 50: a five-thousandth of the radius.)"""
    n_seg, n_rays = 300, 20000
    verts, idx = _strand(1, n_seg), np.arange(n_seg, dtype=np.uint32)
    verts[:, :3] *= np.float32(2.5 / np.abs(verts[:, :3]).max())
    rng = np.random.default_rng(factor)
    seg, u = rng.integers(0, n_seg, n_rays), rng.random(n_rays)
    cp = verts[:, :3].astype(np.float64)
    b = np.stack([(1 - u) ** 3, 3 * u ** 3 - 6 * u ** 2 + 4, -3 * u ** 3 + 3 * u ** 2 + 3 * u + 1, u ** 3], 1) / 6
    axis = sum(b[:, j:j + 1] * cp[seg + j] for j in range(4))
    way = rng.normal(size=(n_rays, 3))
    way /= np.linalg.norm(way, axis=1, keepdims=True)
    way[::5] = np.eye(3)[rng.integers(0, 3, way[::5].shape[0])] * rng.choice([-1.0, 1.0], (way[::5].shape[0], 1))
    o, d = (axis - 2.5 * factor * way).astype(np.float32), way.astype(np.float32)
    rays = {"org_x": o[:, 0], "org_y": o[:, 1], "org_z": o[:, 2], "dir_x": d[:, 0], "dir_y": d[:, 1], "dir_z": d[:, 2],
            "tnear": np.zeros(n_rays, np.float32), "tfar": np.full(n_rays, np.inf, np.float32)}
    rays = {k: np.ascontiguousarray(v) for k, v in rays.items()}
    scene = N.Scene(gpu_ctx)
    scene.add_curves(verts, idx)
    scene.commit()
    dr, dh = N.DeviceRays(gpu_ctx, rays), N.DeviceHits(gpu_ctx, n_rays)
    scene.intersect(dr, dh)
    occ = gpu_ctx.empty(4 * n_rays)
    scene.occluded(dr, occ)
    N.synchronize()
    scene.check()
    got = dh.to_host()
    scene.release()
    want = O.curves_closest(O.curve_segments({"curve_vertices": verts, "curves": idx}), dict(rays, tfar=np.full(n_rays, 1e30, np.float32)))
    hit = want["prim"] != N.INVALID_ID
    # a ray along the strand may start inside it; and one that grazes an earlier turn of it may go either way
    assert hit.mean() > 0.999 and np.array_equal(got["geom_id"] == 0, occ.download(np.uint32, n_rays) == 1)
    close = np.abs(got["t"] - want["t"]) <= 1e-5 * want["t"]
    assert (hit & ~close).sum() <= 1 + 2e-4 * n_rays, (hit & ~close).sum()
