"""Launches of few rays (eight lanes a ray) give the bits of large ones (one lane a ray): prefixes of one
set of rays at counts that leave groups and waves partly filled, and on both sides of the counts where
the kernel changes, over geometries with doubled triangles (ties) and over instances."""
import numpy as np
import pytest

import instancing as I
from selas_amd import native as N
from test_instances_gpu import _rays, _soup

pytestmark = pytest.mark.gpu

COUNTS = [1, 7, 8, 9, 31, 33, 1000, 98304, 98305, 131072]
N_RAYS = 131073  # past both lines


@pytest.fixture(scope="module", params=["one", "flat", "instanced"])
def scene(gpu_ctx, request):
    top = N.Scene(gpu_ctx)
    parts = [top]
    if request.param == "instanced":
        rng = np.random.default_rng(3)
        m = I.Model([("soup", _soup(4, 900))])
        dm = m.device(gpu_ctx)
        parts.append(dm)
        for _ in range(90):
            x = np.asarray(I.random_transform(rng, scale=(0.3, 1.5), spread=6.0), np.float32).reshape(4, 4).T
            top.add_instance(dm, x)
            top.add_instance(dm, x)  # twice in one place: the ties go by instance
    else:
        t = _soup(5, 1 if request.param == "one" else 6000, spread=4.0)
        top.add_soup(np.concatenate([t, t[::2]]) if request.param == "flat" else t)
    top.commit()
    rays = _rays(6, N_RAYS)
    yield top, rays, _trace(gpu_ctx, top, rays, N_RAYS)
    for s in parts:
        s.release()


def _trace(ctx, scene, rays, n):
    dr = N.DeviceRays(ctx, {k: v[:n] for k, v in rays.items()})
    dh = N.DeviceHits(ctx, n, with_inst=True)
    occ = ctx.array(np.full(n, 7, np.uint32))
    scene.intersect(dr, dh)
    scene.occluded(dr, occ)
    N.synchronize()
    scene.check()
    out = dh.to_host()
    out["occluded"] = occ.download(np.uint32, n)
    return out


@pytest.mark.parametrize("n", COUNTS)
def test_prefix_equals_large_launch(gpu_ctx, scene, n):
    top, rays, want = scene
    got = _trace(gpu_ctx, top, rays, n)
    assert (want["prim_id"] != N.INVALID_ID).any()
    for k in want:
        assert np.array_equal(got[k].view(np.uint32), want[k][:n].view(np.uint32)), (n, k)
