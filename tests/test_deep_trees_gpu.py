"""Trees too deep for the part of a traversal's stack that is in LDS: entries spilled and taken back, in
launches of one lane a ray (with the hand-over of a wave's last rays to eight lanes each), over geometries,
instances and several scenes at once, and in the curve pass; trees too deep for eight lanes a ray, whose
small launches go lane by lane. Hits are the oracle's, bit for bit. Every scene's stack words are asked
for, so that a tree that is no longer deep enough fails."""
import numpy as np
import pytest

import deep
import instancing as I
import oracle as O
from selas_amd import native as N
from selas_amd import workloads as W

pytestmark = pytest.mark.gpu

# octant levels of the scenes whose stacks spill and still fit eight lanes a ray, and of those that don't
SPILLS, TOO_DEEP = 13, 21
CORE = {SPILLS: 0, TOO_DEEP: 2048}


def _trace(ctx, scene, rays, noalloc=False):
    n = rays["org_x"].size
    dr, dh = N.DeviceRays(ctx, rays), N.DeviceHits(ctx, n, with_inst=True)
    occ = ctx.array(np.full(n, 7, np.uint32))
    (scene.intersect_noalloc if noalloc else scene.intersect)(dr, dh)
    scene.occluded(dr, occ)
    N.synchronize()
    scene.check()
    return dict(dh.to_host(), occluded=occ.download(np.uint32, n))


def _same(got, want, keys, what):
    for k in keys:
        a, b = got[k].view(np.uint32), want[k].view(np.uint32)
        bad = np.nonzero(a != b)[0]
        assert bad.size == 0, (what, k, bad.size, bad[:5])


def _check_words(scene, too_deep):
    words = deep.stack_words(scene)
    print(f"stack words: {words}", flush=True)
    assert words > deep.MOST_GROUP_WORDS if too_deep else deep.LDS_WORDS < words <= deep.MOST_GROUP_WORDS, words


@pytest.fixture(scope="module", params=[SPILLS, TOO_DEEP])
def flat(gpu_ctx, request):
    soup = deep.nested_soup(1, request.param, core=CORE[request.param])
    scene = N.Scene(gpu_ctx)
    scene.add_soup(soup)
    scene.commit()
    _check_words(scene, request.param == TOO_DEEP)
    yield scene, O.CpuBvh(soup), request.param
    scene.release()


@pytest.mark.parametrize("n", [1, 63, 1000, 131073, 600001])
def test_flat(gpu_ctx, flat, n):
    """1 and 63 rays to 1000: eight lanes a ray, or lane by lane where the tree is too deep for that;
    131,073: each wave its one chunk, then its last rays eight lanes each; 600,001: chunks from the
    counter."""
    scene, bvh, levels = flat
    rays = deep.rays(n, n, levels)
    print(f"flat, {levels} levels, {n} rays", flush=True)
    got, ref = _trace(gpu_ctx, scene, rays), bvh.closest(rays)
    want = {"t": ref["t"], "u": ref["u"], "v": ref["v"], "prim_id": ref["prim"], "occluded": bvh.occluded(rays)}
    _same(got, want, want, n)
    assert n < 1000 or 0.2 < (want["prim_id"] != N.INVALID_ID).mean() < 0.99


def test_flat_without_allocation(gpu_ctx, flat):
    """The fixed per-GPU array: the deeper tree's spill fits fewer blocks of it than the launch would
    use."""
    scene, bvh, levels = flat
    for n in (600001, 7000, 140000):
        rays = deep.rays(n + 1, n, levels)
        print(f"flat without allocation, {levels} levels, {n} rays", flush=True)
        got, ref = _trace(gpu_ctx, scene, rays, noalloc=True), bvh.closest(rays)
        _same(got, {"t": ref["t"], "u": ref["u"], "v": ref["v"], "prim_id": ref["prim"]}, ("t", "u", "v", "prim_id"), n)


@pytest.fixture(scope="module", params=[(SPILLS, 6), (SPILLS, 90), (TOO_DEEP, 6)], ids=["spills", "spills-90", "too-deep"])
def instanced(gpu_ctx, request):
    levels, count = request.param
    m = I.Model([("soup", deep.nested_soup(2, levels, core=CORE[levels]))])
    dm = m.device(gpu_ctx)
    top = N.Scene(gpu_ctx)
    rng = np.random.default_rng(3)
    xs = [np.asarray(I.random_transform(rng, scale=(0.7, 1.4), spread=1.5 if count < 10 else 4.0), np.float32) for _ in range(count)]
    xs[1] = xs[0]  # two in one place: ties go by instance
    for x in xs:
        top.add_instance(dm, x.reshape(4, 4).T)
    top.commit()
    _check_words(top, levels == TOO_DEEP)
    yield top, I.compose([(m, x) for x in xs]), [x.reshape(4, 4).T.astype(float) for x in xs], levels
    top.release()
    dm.release()


def _instance_rays(xs, seed, n, levels):
    """Rays of the model's own kinds, each batch carried by one of the placements."""
    parts = [deep.placed(deep.rays(seed + k, -(-n // len(xs)), levels), x) for k, x in enumerate(xs)]
    order = np.random.default_rng(seed).permutation(len(xs) * (-(-n // len(xs))))[:n]
    return {k: np.ascontiguousarray(np.concatenate([p[k] for p in parts])[order]) for k in N.RAY_FIELDS}


@pytest.mark.parametrize("n", [9, 2000, 131073, 600001])
def test_instances(gpu_ctx, instanced, n):
    top, composed, xs, levels = instanced
    rays = _instance_rays(xs, n, n, levels)
    print(f"{len(xs)} instances, {levels} levels, {n} rays", flush=True)
    got = _trace(gpu_ctx, top, rays)
    # the oracle for up to 40,000 rays of the launch, spread over it
    pick = np.unique(np.linspace(0, n - 1, min(n, 40000)).astype(np.int64))
    ref = I.oracle_hits(composed, {k: np.ascontiguousarray(v[pick]) for k, v in rays.items()})
    _same({k: v[pick] for k, v in got.items()}, ref, ("t", "u", "v", "prim_id", "geom_id", "inst_id0", "occluded"), n)
    assert n < 2000 or 0.2 < (ref["prim_id"] != N.INVALID_ID).mean() < 0.999
    if n > 2000:  # all of them: the same in launches of the other kind
        small = [_trace(gpu_ctx, top, {k: np.ascontiguousarray(v[a:a + 90000]) for k, v in rays.items()})
                 for a in range(0, n, 90000)]
        _same(got, {k: np.concatenate([s[k] for s in small]) for k in got}, got, n)


def _deep_scene(levels):
    """An instanced scene of two deep models over a floor, seen from one's inner corner."""
    soup = {"geoms": [deep.nested_soup(4, levels, core=CORE[levels])], "materials": np.stack([W.material(2, (0.7, 0.6, 0.5))]),
            "geom_material": np.zeros(1, np.uint32)}
    floor = {"geoms": [np.array([[-4, -0.5, -4, 4, -0.5, 4, 4, -0.5, -4], [-4, -0.5, -4, -4, -0.5, 4, 4, -0.5, 4]], np.float32)],
             "materials": np.stack([W.material(2, (0.5, 0.5, 0.5))]), "geom_material": np.zeros(1, np.uint32)}
    lights = np.zeros(1, W.LIGHT_DTYPE)
    lights[0] = (0, (0.5, 3.0, 0.5), (0.0, -1.0, 0.0), (2.0, 0.0, 0.0), (0.0, 0.0, 2.0), (6.0, 6.0, 6.0))
    far = np.eye(4)
    far[:3, 3] = (1.2, 0.1, 0.4)
    e = 2.0 ** -levels
    return {"models": [soup, floor], "instances": [("model", 0, np.eye(4)), ("model", 0, far), ("model", 1, np.eye(4))],
            "lights": lights, "background": np.zeros(3, np.float32),
            "camera": {"position": (0.3 * e, 0.4 * e, 0.2 * e), "look_at": (1.0, 1.0, 1.0), "up": (0.0, 1.0, 0.0), "fov": 60.0}}


@pytest.mark.parametrize("levels", [SPILLS, TOO_DEEP])
def test_several_scenes_at_once(gpu_ctx, levels):
    """Jobs on a deep instanced scene and on a flat one in one wavefront (the scene-table launches, as
    graphs and one by one), past the counts that eight lanes a ray take: each job's image is that of the
    job alone launched one by one (over its one scene, without the table) but for the order of its splats
    and merged photons."""
    deep_sc, flat_sc = _deep_scene(levels), W.sized_vcm_scene(5, 1e4, textures=False)
    sd, sf = N.build_render_scene(gpu_ctx, deep_sc), N.build_render_scene(gpu_ctx, flat_sc)
    _check_words(sd, levels == TOO_DEEP)
    print(f"several scenes, {levels} levels", flush=True)
    jobs = [(sd, deep_sc["camera"], 500, 500, 1, 6), (sf, flat_sc["camera"], 200, 200, 2, 7), (sd, deep_sc["camera"], 64, 64, 2, 8)]
    try:
        gpu_ctx.set_tuning(vcm_graphs=0)
        alone = [N.render_vcm(s, cam, w, h, its, 6, 0.01, 0.75, seed) for s, cam, w, h, its, seed in jobs]
        for graphs in (0, 1):
            gpu_ctx.set_tuning(vcm_graphs=graphs)
            batch = N.render_vcm_batch([dict(scene=s, camera=cam, width=w, height=h, iterations=its, max_path_length=6,
                                             base_radius=0.01, radius_alpha=0.75, seed=seed) for s, cam, w, h, its, seed in jobs])
            for a, b in zip(alone, batch):
                assert a.mean() > 1e-3
                # sums of one sign of some hundred terms in another order: 100 x 2^-24 = 6e-6 relative
                np.testing.assert_allclose(b, a, rtol=1e-5, atol=1e-6 * float(a.max()))
    finally:
        gpu_ctx.set_tuning(vcm_graphs=1)
    sd.release()
    sf.release()


def _axis_rays(seed, n, verts, idx, levels):
    """Rays from about the origin through points of the segments' axes: they do not graze the segment they
    aim at, and being short where the segments are small keep their precision there."""
    rng = np.random.default_rng(seed)
    seg, u = idx[rng.integers(0, idx.size, n)].astype(np.int64), rng.random(n)
    b = np.stack([(1 - u) ** 3, 3 * u ** 3 - 6 * u ** 2 + 4, -3 * u ** 3 + 3 * u ** 2 + 3 * u + 1, u ** 3], 1) / 6
    axis = sum(b[:, j:j + 1] * verts[seg + j, :3].astype(float) for j in range(4))
    o = rng.random((n, 3)) * 2.0 ** -(levels + 2)
    d = axis - o
    far = np.linalg.norm(d, axis=1)
    f = lambda a: np.ascontiguousarray(a, np.float32)
    d /= far[:, None]
    return {"org_x": f(o[:, 0]), "org_y": f(o[:, 1]), "org_z": f(o[:, 2]), "dir_x": f(d[:, 0]), "dir_y": f(d[:, 1]),
            "dir_z": f(d[:, 2]), "tnear": f(np.zeros(n)), "tfar": f(np.full(n, 1e30))}


@pytest.mark.parametrize("n", [500, 20000, 300001])
@pytest.mark.parametrize("levels", [14, TOO_DEEP])
def test_curves(gpu_ctx, levels, n):
    verts, idx = deep.nested_strands(6, levels)
    scene = N.Scene(gpu_ctx)
    scene.add_curves(verts, idx)
    scene.commit()
    words = deep.stack_words(scene)
    print(f"curves, {levels} levels, {n} rays, stack words {words}", flush=True)
    assert words > deep.LDS_WORDS
    rays = _axis_rays(n, n, verts, idx, levels)
    got = _trace(gpu_ctx, scene, rays)
    hit = got["geom_id"] == 0
    # a ray aimed at an axis hits its segment or one before it, but for the few that start inside one
    assert hit.mean() > 0.999 and np.array_equal(hit, got["occluded"] == 1)
    pick = np.unique(np.linspace(0, n - 1, min(n, 20000)).astype(np.int64))
    want = O.curves_closest(O.curve_segments({"curve_vertices": verts, "curves": idx}),
                            {k: np.ascontiguousarray(v[pick]) for k, v in rays.items()})
    # the search is in float, in the coordinates of the segment: t to 1e-5 of itself (as at a scale of one)
    # and 1e-6 of those, some ulps; a ray that grazes a segment before its own may take it on one side only
    at = np.max(np.abs(np.stack([rays["org_" + a][pick] + want["t"] * rays["dir_" + a][pick] for a in "xyz"])), axis=0)
    close = np.abs(got["t"][pick] - want["t"]) <= 1e-5 * want["t"] + 1e-6 * at
    assert (~close).sum() <= 1 + 2e-4 * pick.size, (~close).sum()
    scene.release()
