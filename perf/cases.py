"""The work a user of this framework has it do, as cases that can be timed and compared.

Every case goes through the public Python binding (selas_amd.native over libselas_gpu's C ABI):

  closest / any   sgpu_intersect and sgpu_occluded on a committed scene of triangles, for ray counts
                  from one pick up to a full frame's samples;
  instances       sgpu_intersect on a two-level instanced scene;
  curves          sgpu_intersect on a scene with round B-spline curves;
  commit          a scene made, filled, committed (the device tree build) and queried once;
  pt, deferred    the unidirectional and the deferred path tracer, whole images;
  vcm, batch      vertex connection and merging: one job, and several uneven jobs at once.

A state holds what such a program keeps: the resident scene, the rays or the job on the device, the
output buffers. Scenes, rays and job seeds all come from the seed. Contexts are kept per wavefront
size, as a program keeps one context per GPU.
"""
import math

import numpy as np
import torch

from selas_amd import native as N
from selas_amd import workloads as W

INF = float("inf")


# ---- the listed cases ------------------------------------------------------------------------------

def listed():
    return [
        # a pick or a probe: a handful of rays against a small model; latency and launches
        {"name": "closest 61 rays", "kind": "closest", "tris": 20480, "rays": 61, "coherent": False},
        # an interactive frame's primary and bounce rays, an odd count, a medium model
        {"name": "closest 250k rays", "kind": "closest", "tris": 65536, "rays": 250007, "coherent": False},
        # a full frame's samples against a large model: the traversal workload of the benchmark
        {"name": "closest 16M rays", "kind": "closest", "tris": 2097152, "rays": 16777216, "coherent": False},
        # the shadow rays of a large bounce
        {"name": "any 4M rays", "kind": "any", "tris": 1048576, "rays": 4194304, "coherent": False},
        # two instance levels (a model placed in a subscene, the subscene in the scene)
        {"name": "instances 4M rays", "kind": "instances", "tris": 8192, "placed": 256, "rays": 4194304},
        # hair and grass
        {"name": "curves 1M rays", "kind": "curves", "strands": 65536, "rays": 1048576},
        # a scene loaded and committed, then queried
        {"name": "commit 500k tris", "kind": "commit", "tris": 524288, "rays": 4096},
        # the path tracer's small image: many short launches
        {"name": "path tracer 256", "kind": "pt", "width": 256, "height": 256, "spp": 16, "length": 8},
        # the deferred path tracer under a sky
        {"name": "deferred 320x200", "kind": "deferred", "tris": 65536, "width": 320, "height": 200, "spp": 4, "length": 10,
         "sort": 0},
        # the smallest VCM request: a thumbnail, one iteration
        {"name": "vcm 64", "kind": "vcm", "tris": 10000, "width": 64, "height": 64, "iterations": 1, "paths": 1 << 20},
        # the headline job: 512 x 512, 32 iterations, 1M triangles, at the stored launch shape
        {"name": "vcm 512", "kind": "vcm", "tris": 1048576, "width": 512, "height": 512, "iterations": 32, "paths": 1 << 24},
        # uneven jobs on scenes of their own, rendered together
        {"name": "batch of 8", "kind": "batch", "tris": 65536, "jobs": 8, "side": 384, "iterations": 24, "paths": 1 << 22},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["closest", "closest", "any", "instances", "curves", "commit", "pt", "deferred", "vcm", "vcm", "batch"])
    if kind in ("closest", "any"):
        return {"kind": kind, "tris": _log(rng, 256, 2e6), "rays": _log(rng, 1, 1.6e7), "coherent": rng.random() < 0.3}
    if kind == "instances":
        return {"kind": kind, "tris": _log(rng, 256, 3e4), "placed": rng.choice([4, 16, 64, 256]), "rays": _log(rng, 1e3, 4e6)}
    if kind == "curves":
        return {"kind": kind, "strands": _log(rng, 1e3, 1e5), "rays": _log(rng, 1e3, 1e6)}
    if kind == "commit":
        return {"kind": kind, "tris": _log(rng, 1e3, 1e6), "rays": _log(rng, 64, 65536)}
    if kind == "pt":
        return {"kind": kind, "width": _log(rng, 32, 400), "height": _log(rng, 32, 400), "spp": rng.choice([1, 4, 9, 16, 25]),
                "length": rng.choice([4, 8, 10])}
    if kind == "deferred":
        return {"kind": kind, "tris": _log(rng, 1e4, 3e5), "width": _log(rng, 48, 400), "height": _log(rng, 48, 400),
                "spp": rng.choice([1, 2, 4]), "length": rng.choice([6, 10]), "sort": rng.choice([0, 0, 1, 2])}
    if kind == "vcm":
        return {"kind": kind, "tris": _log(rng, 1e4, 3e5), "width": _log(rng, 48, 400), "height": _log(rng, 48, 400),
                "iterations": rng.randint(1, 16), "paths": rng.choice([1 << 20, 1 << 22])}
    return {"kind": kind, "tris": _log(rng, 1e4, 1e5), "jobs": rng.randint(2, 8), "side": _log(rng, 64, 384),
            "iterations": rng.randint(2, 24), "paths": rng.choice([1 << 20, 1 << 22])}


# ---- states ----------------------------------------------------------------------------------------

_contexts = {}


def _context(paths=1 << 20):
    """The program's context for this wavefront size (sgpu_tuning.vcm_wavefront_paths)."""
    if paths not in _contexts:
        c = N.Context(0)
        c.set_tuning(vcm_wavefront_paths=paths)
        _contexts[paths] = c
    return _contexts[paths]


class Buffer:
    """A torch tensor as the binding's device buffer (its `ptr`)."""

    def __init__(self, shape, dtype=torch.float32):
        self.tensor = torch.zeros(shape, dtype=dtype, device="cuda")
        self.ptr = self.tensor.data_ptr()


class Rays:
    """SoA rays in torch tensors."""

    def __init__(self, org, direction, tnear, tfar):
        cols = [org[:, 0], org[:, 1], org[:, 2], direction[:, 0], direction[:, 1], direction[:, 2], tnear, tfar]
        self.cols = [c.to(torch.float32).contiguous().clone() for c in cols]
        self.n = int(org.shape[0])
        self.soa = N.RaysSoA(*[c.data_ptr() for c in self.cols])


class Hits:
    """The closest-hit outputs in torch tensors (instance ids where the scene has instances)."""

    def __init__(self, n, instances=False):
        ids = ("prim_id", "geom_id") + (("inst_id0", "inst_id1") if instances else ())
        self.out = {k: torch.zeros(n, dtype=torch.float32, device="cuda") for k in ("t", "u", "v", "ng_x", "ng_y", "ng_z")}
        self.out.update({k: torch.zeros(n, dtype=torch.int32, device="cuda") for k in ids})
        self.soa = N.HitsSoA(*[self.out[f].data_ptr() if f in self.out else None for f, _ in N.DeviceHits.FIELDS])


class State:
    def __init__(self, case):
        self.kind = case["kind"]
        self.scenes = []  # released in this order

    def __del__(self):
        try:
            torch.cuda.synchronize()
            for s in self.scenes:
                s.release()
        except Exception:
            pass


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _camera_rays(g, n):
    """Jittered pinhole rays over a square image of the unit box, in scanline order."""
    side = max(1, int(math.isqrt(n)))
    i = torch.arange(n, device="cuda")
    j = torch.rand((n, 2), generator=g, device="cuda", dtype=torch.float64)
    spp = max(1, n // (side * side))
    x = ((i // spp) % side + j[:, 0]) / side
    y = (((i // spp) // side) % side + j[:, 1]) / side
    s = 2 * math.tan(math.radians(W.CAMERA_FOV) / 2)
    d = torch.stack([(x - 0.5) * s, (0.5 - y) * s, torch.ones_like(x)], 1)
    o = torch.tensor(W.CAMERA_POS, device="cuda", dtype=torch.float64).expand(n, 3)
    return o, d / d.norm(dim=1, keepdim=True)


def _surface_points(g, tri, n):
    """Points uniform on uniformly chosen triangles, and those triangles' unit normals."""
    k = torch.randint(tri.shape[0], (n,), generator=g, device="cuda")
    t = tri[k].view(n, 3, 3).double()
    u = torch.rand((n, 2), generator=g, device="cuda", dtype=torch.float64)
    u = torch.where(u.sum(1, keepdim=True) > 1, 1 - u, u)
    e1, e2 = t[:, 1] - t[:, 0], t[:, 2] - t[:, 0]
    ng = torch.linalg.cross(e1, e2)
    return t[:, 0] + u[:, :1] * e1 + u[:, 1:] * e2, ng / ng.norm(dim=1, keepdim=True).clamp_min(1e-30)


def _sphere(g, n):
    d = torch.randn((n, 3), generator=g, device="cuda", dtype=torch.float64)
    return d / d.norm(dim=1, keepdim=True)


def _trace_rays(g, tri, n, coherent):
    """Half camera rays and half cosine rays leaving the surfaces (all camera rays if coherent)."""
    nb = 0 if coherent else n // 2
    o, d = _camera_rays(g, n - nb)
    if nb:
        p, ng = _surface_points(g, tri, nb)
        b = ng + 0.999 * _sphere(g, nb)
        o, d = torch.cat([o, p]), torch.cat([d, b / b.norm(dim=1, keepdim=True)])
    return Rays(o, d, torch.full((n,), 1e-4, device="cuda"), torch.full((n,), INF, device="cuda"))


def _shadow_rays(g, tri, n, coherent):
    """Segments from surface points (in triangle order, if coherent) to one of two lights above the box."""
    p, _ = _surface_points(g, tri, n)
    if coherent:
        p = p[p[:, 0].argsort()]
    lights = torch.tensor([[0.3, 1.4, 0.4], [1.2, 1.1, -0.2]], device="cuda", dtype=torch.float64)
    to = lights[torch.randint(2, (n,), generator=g, device="cuda")] - p
    dist = to.norm(dim=1)
    return Rays(p, to / dist[:, None], torch.full((n,), 1e-4, device="cuda"), dist * 0.999)


def _soup(seed, tris):
    per = max(1, min(8192, tris // 16))
    return N.gen_cluster_soup(seed, -(-tris // per), per, 0.02 if tris > 1e5 else 0.05, 1e-3, 2e-2 if tris > 1e5 else 8e-2)[:tris]


def _rotation(rng):
    q, r = np.linalg.qr(rng.normal(size=(3, 3)))
    return q * np.sign(np.diag(r))


def _placement(rng, lo, hi):
    return np.vstack([np.hstack([_rotation(rng), rng.uniform(lo, hi, (3, 1))]), [0, 0, 0, 1]])


def _grass(rng, ns):
    """Blades of 10 control points (7 segments), radius 3 mm tapering to 1 mm, 10-25 cm tall, on 2 m x 2 m."""
    ncp = 10
    height = rng.uniform(0.10, 0.25, ns)
    d = np.tile([0.0, 1.0, 0.0], (ns, 1)) + 0.3 * rng.normal(size=(ns, 3)) * [1, 0, 1]
    pts = [np.stack([rng.uniform(-1, 1, ns), np.zeros(ns), rng.uniform(-1, 1, ns)], 1)]
    for _ in range(ncp - 1):
        d = d + 0.15 * rng.normal(size=(ns, 3)) * [1, 0.2, 1]
        d /= np.linalg.norm(d, axis=1, keepdims=True)
        pts.append(pts[-1] + d * (height / (ncp - 1))[:, None])
    rad = np.broadcast_to(np.linspace(0.003, 0.001, ncp)[None, :, None], (ns, ncp, 1))
    verts = np.concatenate([np.stack(pts, 1), rad], 2).reshape(-1, 4).astype(np.float32)
    return verts, (np.arange(ns)[:, None] * ncp + np.arange(ncp - 3)[None, :]).reshape(-1).astype(np.uint32)


def _render_scene(seed, tris, sky):
    nv = max(2, int(round(math.sqrt(tris / 256.0))))
    sc = W.vcm_scene(seed=seed % (1 << 31), n_meshes=64, nu=2 * nv, nv=nv, textures=True, res_log2=3)
    if sky:
        sc["ibl"] = {"rgb": W.sky_map(64, 128), "rotation": 0.0, "exposure": 1.0}
    return sc


def _batch_shape(case):
    """(side, iterations) of each job: sides down to a quarter, uneven iteration counts."""
    n = case["jobs"]
    return [(max(32, int(round(case["side"] * 0.25 ** (k / max(1, n - 1))))), 1 + (case["iterations"] - 1) * ((5 * k + 3) % n) // max(1, n - 1))
            for k in range(n)]


def prepare(case, seed):
    kind, st = case["kind"], State(case)
    if kind in ("closest", "any"):
        tri = _soup(seed, case["tris"])
        scene = N.Scene(_context())
        scene.add_soup(tri)
        scene.commit()
        st.scenes, st.scene = [scene], scene
        g, dev = _generator(seed), torch.from_numpy(tri).cuda()
        if kind == "any":
            st.rays, st.hits = _shadow_rays(g, dev, case["rays"], case["coherent"]), Buffer(case["rays"], torch.int32)
        else:
            st.rays, st.hits = _trace_rays(g, dev, case["rays"], case["coherent"]), Hits(case["rays"])
    elif kind == "instances":
        rng = np.random.default_rng(seed)
        model = N.gen_cluster_soup(seed, 1, case["tris"], 0.02, 1e-4, 1e-2)
        model = (model.reshape(-1, 3) - model.reshape(-1, 3).mean(0)).astype(np.float32).reshape(-1, 9)
        side = max(1, int(math.isqrt(case["placed"])))
        scenes = [N.Scene(_context()) for _ in range(3)]
        scenes[2].add_soup(model)
        scenes[2].commit()
        for _ in range(side):
            scenes[1].add_instance(scenes[2], _placement(rng, -0.15, 0.15))
        scenes[1].commit()
        for _ in range(case["placed"] // side):
            scenes[0].add_instance(scenes[1], _placement(rng, 0.2, 0.8))
        scenes[0].commit()
        st.scenes, st.scene = scenes, scenes[0]
        n, g = case["rays"], _generator(seed)
        o, d = _camera_rays(g, n - n // 2)
        p = torch.rand((n // 2, 3), generator=g, device="cuda", dtype=torch.float64)
        st.rays = Rays(torch.cat([o, p]), torch.cat([d, _sphere(g, n // 2)]), torch.full((n,), 1e-4, device="cuda"),
                       torch.full((n,), INF, device="cuda"))
        st.hits = Hits(n, instances=True)
    elif kind == "curves":
        verts, idx = _grass(np.random.default_rng(seed), case["strands"])
        scene = N.Scene(_context())
        scene.add_soup(np.array([[-1.2, 0, -1.2, 1.2, 0, -1.2, 1.2, 0, 1.2], [-1.2, 0, -1.2, 1.2, 0, 1.2, -1.2, 0, 1.2]], np.float32))
        scene.add_curves(verts, idx)
        scene.commit()
        st.scenes, st.scene = [scene], scene
        n, g = case["rays"], _generator(seed)
        # a camera above the field looking down at it, and cosine rays up from the ground
        o, d = _camera_rays(g, n - n // 2)
        eye, look = np.array([0.0, 1.2, -1.9]), np.array([0.0, 0.05, 0.0])
        f = (look - eye) / np.linalg.norm(look - eye)
        r = np.cross([0.0, 1.0, 0.0], f)
        r /= np.linalg.norm(r)
        basis = torch.tensor(np.stack([r, np.cross(f, r), f]), device="cuda")
        p = torch.rand((n // 2, 3), generator=g, device="cuda", dtype=torch.float64) * 2 - 1
        p[:, 1] = 1e-3
        up = torch.tensor([0.0, 1.0, 0.0], device="cuda", dtype=torch.float64) + 0.999 * _sphere(g, n // 2)
        st.rays = Rays(torch.cat([torch.tensor(eye, device="cuda").expand(n - n // 2, 3), p]),
                       torch.cat([d @ basis, up / up.norm(dim=1, keepdim=True)]), torch.zeros(n, device="cuda"),
                       torch.full((n,), INF, device="cuda"))
        st.hits = Hits(n)
    elif kind == "commit":
        st.tri = _soup(seed, case["tris"])
        st.context = _context()
        st.rays = _trace_rays(_generator(seed), torch.from_numpy(st.tri).cuda(), case["rays"], False)
        st.hits = Hits(case["rays"])
    elif kind == "pt":
        sc = W.room_scene(seed % (1 << 31))
        scene = N.build_render_scene(_context(), sc)
        st.scenes, st.scene, st.camera = [scene], scene, sc["camera"]
        st.args = (case["width"], case["height"], case["spp"], case["length"], seed)
        st.frame = Buffer((2, case["height"], case["width"], 3))
    elif kind == "deferred":
        sc = _render_scene(seed, case["tris"], sky=True)
        scene = N.build_render_scene(_context(), sc)
        st.scenes, st.scene, st.camera = [scene], scene, sc["camera"]
        st.args = (case["width"], case["height"], case["spp"], case["spp"], case["length"], seed)
        st.flags = (0, N.DPT_SORT_HITS, N.DPT_SORT_RAYS)[case["sort"]]
        st.frame = Buffer((case["height"], case["width"], 3))
    elif kind == "vcm":
        sc = _render_scene(seed, case["tris"], sky=False)
        scene = N.build_render_scene(_context(case["paths"]), sc)
        st.scenes, st.scene, st.camera = [scene], scene, sc["camera"]
        st.args = (case["width"], case["height"], case["iterations"], sc["max_path_length"], sc["merge_radius"], sc["radius_alpha"], seed)
        st.frame = Buffer((case["height"], case["width"], 3))
    else:
        st.jobs, st.frames = [], []
        scs = [_render_scene(seed + 7 * k, case["tris"] >> (2 * k), sky=False) for k in range(2)]
        st.scenes = [N.build_render_scene(_context(case["paths"]), sc) for sc in scs]
        for k, (side, its) in enumerate(_batch_shape(case)):
            sc = scs[k % 2]
            st.jobs.append({"scene": st.scenes[k % 2], "camera": sc["camera"], "width": side, "height": side, "iterations": its,
                            "max_path_length": sc["max_path_length"], "base_radius": sc["merge_radius"],
                            "radius_alpha": sc["radius_alpha"], "seed": seed + k})
            st.frames.append(Buffer((side, side, 3)))
    return st


# ---- one pass --------------------------------------------------------------------------------------

def run(st):
    kind = st.kind
    if kind in ("closest", "instances", "curves"):
        st.scene.intersect(st.rays, st.hits)
        return st.hits.out
    if kind == "any":
        st.scene.occluded(st.rays, st.hits)
        return st.hits.tensor
    if kind == "commit":
        scene = N.Scene(st.context)
        scene.add_soup(st.tri)
        scene.commit()
        scene.intersect(st.rays, st.hits)
        scene.release()  # a new scene takes the old one's place
        return st.hits.out
    if kind == "pt":
        N.render_pt(st.scene, st.camera, *st.args, framebuffer=st.frame)
    elif kind == "deferred":
        N.render_deferred_pt(st.scene, st.camera, *st.args, flags=st.flags, framebuffer=st.frame)
    elif kind == "vcm":
        N.render_vcm(st.scene, st.camera, *st.args, framebuffer=st.frame)
    else:
        N.render_vcm_batch(st.jobs, framebuffers=st.frames)
        return [f.tensor for f in st.frames]
    return st.frame.tensor


# ---- what a pass cannot do without ------------------------------------------------------------------

def _query_flops(prims):
    """One path down an 8-wide tree to one primitive: 8 boxes of 6 planes (a multiply-add and a
    compare each) a level, and one triangle test of about 60 operations."""
    return max(1, math.ceil(math.log(max(2, prims), 8))) * 8 * 6 * 3 + 60


def work(case):
    kind = case["kind"]
    if kind in ("closest", "any", "instances", "commit"):
        prims = case["tris"] * case.get("placed", 1)
        out = 4 if kind == "any" else 40 if kind == "instances" else 32
        return {"bytes": 36 * case["tris"] + case["rays"] * (32 + out),
                "flops": case["rays"] * _query_flops(prims) + (60 * case["tris"] if kind == "commit" else 0)}
    if kind == "curves":
        # a segment's 64 bytes; a hit's search along one segment is some 20 steps of 50 operations
        return {"bytes": 64 * 7 * case["strands"] + case["rays"] * 64, "flops": case["rays"] * (_query_flops(7 * case["strands"]) + 1000)}
    if kind == "pt":
        # each path sample is at least one closest-hit ray, one shadow ray and one shaded vertex a bounce; about 3.5 bounces
        return {"bytes": 24 * case["width"] * case["height"] + 36 * 20504,
                "flops": case["width"] * case["height"] * case["spp"] * 3.5 * (2 * _query_flops(20504) + 300)}
    if kind == "deferred":
        return {"bytes": 12 * case["width"] * case["height"] + (36 + 96) * case["tris"],
                "flops": case["width"] * case["height"] * case["spp"] ** 2 * 3.0 * (2 * _query_flops(case["tris"]) + 300)}
    # VCM: about 5.8 rays a sample and 18 photons merged a sample at some 300 operations each
    jobs = _batch_shape(case) if kind == "batch" else None
    samples = sum(s * s * i for s, i in jobs) if jobs else case["width"] * case["height"] * case["iterations"]
    pixels = sum(s * s for s, _ in jobs) if jobs else case["width"] * case["height"]
    return {"bytes": 12 * pixels + (36 + 96) * case["tris"], "flops": samples * (5.8 * _query_flops(case["tris"]) + 18 * 300)}


# ---- how far another correct implementation may be ---------------------------------------------------

def tolerance(case):
    kind = case["kind"]
    if kind in ("closest", "any", "instances", "commit"):
        # the intersection arithmetic is specified operation by operation and the hit does not depend
        # on the tree: results are the same bits
        return "exact"
    if kind == "curves":
        # the hit along a curve is found by a search in 32 bits, to 1.5e-6 of the ray's parameter
        return {"rel": 2e-5, "max": 1e-2, "differ": 1e-5}
    # images: the path tracers equal the CPU restatement bit for bit; VCM's splats and merges add in
    # another order (2-norm 4.5e-8, largest 2.2e-7 against it and against other merge group sizes)
    return {"rel": 1e-6, "max": 1e-5}


# ---- the same in 64 bits -----------------------------------------------------------------------------

def exact(case, seed):
    """Closest hits by testing every ray against every triangle in 64 bits (plain torch); None where that
    is too much, and for images and curves, which have no closed form."""
    if case["kind"] not in ("closest", "commit") or case["rays"] * case["tris"] > 3e10:
        return None
    tri = torch.from_numpy(_soup(seed, case["tris"])).cuda()
    rays = _trace_rays(_generator(seed), tri, case["rays"], case.get("coherent", False))
    c = [x.double() for x in rays.cols]
    o, d, tnear = torch.stack(c[0:3], 1), torch.stack(c[3:6], 1), c[6]
    v = tri.double().view(-1, 3, 3)
    # the edges as the 32-bit records hold them: the differences rounded once
    e1 = (v[:, 1].float() - v[:, 0].float()).double()
    e2 = (v[:, 2].float() - v[:, 0].float()).double()
    v0 = v[:, 0]
    ng = torch.linalg.cross(e1, e2)
    moment = torch.linalg.cross(o, d)
    n, m = o.shape[0], tri.shape[0]
    out = {k: torch.zeros(n, dtype=torch.float64, device="cuda") for k in ("t", "u", "v", "ng_x", "ng_y", "ng_z")}
    out["t"].fill_(INF)
    # with a = v0: det = -d.ng, T = (o - a).ng, U = e2.(o x d) - d.(e2 x a), V = -(e1.(o x d) - d.(e1 x a))
    c2, c1, c0 = torch.linalg.cross(e2, v0), torch.linalg.cross(e1, v0), (v0 * ng).sum(1)
    rows, cols = 4096, 16384
    for r in range(0, n, rows):
        dr, mr, orr, tn = d[r:r + rows], moment[r:r + rows], o[r:r + rows], tnear[r:r + rows, None]
        best = torch.full((dr.shape[0],), INF, dtype=torch.float64, device="cuda")
        bu, bv = torch.zeros_like(best), torch.zeros_like(best)
        bk = torch.zeros(dr.shape[0], dtype=torch.int64, device="cuda")
        for k in range(0, m, cols):
            s = slice(k, min(m, k + cols))
            det = -(dr @ ng[s].t().contiguous())
            T = orr @ ng[s].t().contiguous() - c0[s]
            U = mr @ e2[s].t().contiguous() - dr @ c2[s].t().contiguous()
            V = dr @ c1[s].t().contiguous() - mr @ e1[s].t().contiguous()
            inv = 1.0 / det
            T, U, V = T * inv, U * inv, V * inv
            ok = (U >= 0) & (V >= 0) & (U + V <= 1) & (T > tn) & (det != 0)
            T = torch.where(ok, T, INF)
            t, at = T.min(dim=1)
            better = t < best
            at1 = at[:, None]
            bu = torch.where(better, U.gather(1, at1)[:, 0], bu)
            bv = torch.where(better, V.gather(1, at1)[:, 0], bv)
            bk = torch.where(better, at + k, bk)
            best = torch.where(better, t, best)
        hit = best < INF
        out["t"][r:r + rows] = best
        out["u"][r:r + rows] = torch.where(hit, bu, 0.0)
        out["v"][r:r + rows] = torch.where(hit, bv, 0.0)
        for a, key in enumerate(("ng_x", "ng_y", "ng_z")):
            out[key][r:r + rows] = torch.where(hit, ng[bk, a], 0.0)
    out["prim_id"] = out["geom_id"] = None
    return out

