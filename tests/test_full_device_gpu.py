"""Calls on a device with no memory left but what contexts hold idle and what its pool holds freed: they
get it and give the same results. The device is not really filled: a child process loads
tests/alloc_limit, which refuses the library's allocations past a limit."""
import ctypes
import os
import subprocess
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

HERE = os.path.dirname(os.path.abspath(__file__))
LIMIT_SRC = os.path.join(HERE, "alloc_limit", "alloc_limit.c")


@pytest.fixture(scope="module")
def limit_lib(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("alloc_limit") / "liballoc_limit.so")
    subprocess.run(["gcc", "-std=c11", "-O2", "-Wall", "-Wextra", "-Werror", "-shared", "-fPIC", "-o", so, LIMIT_SRC,
                    "-ldl", "-pthread"], check=True)
    return so


def _child(limit_lib, call):
    r = subprocess.run([sys.executable, "-u", os.path.abspath(__file__), limit_lib, call], capture_output=True, text=True,
                       timeout=100)
    print(r.stdout, r.stderr, flush=True)
    assert r.returncode == 0, (r.returncode, r.stdout[-2000:], r.stderr[-2000:])


CALLS = ["commit", "commit curves", "commit instances", "other context", "materials", "attributes", "texture", "ibl",
         "query", "curve query", "stats", "vcm", "server", "hdr", "pool"]


@pytest.mark.parametrize("call", CALLS)
def test_call_takes_idle_memory(limit_lib, call):
    _child(limit_lib, call)


@pytest.mark.parametrize("kind", ["triangles", "curves", "instances"])
def test_refused_commit_leaves_nothing(limit_lib, kind):
    """Whichever of a commit's allocations is refused: an error, nothing left allocated, and the same
    scene commits once there is memory."""
    _child(limit_lib, "refused " + kind)


# bytes a primitive of device memory that a commit gets by with, the scene's own included
COMMIT_BYTES = {"triangles": 480, "curves": 580, "instances": 613}


@pytest.mark.parametrize("kind", list(COMMIT_BYTES))
def test_commit_memory(limit_lib, kind):
    _child(limit_lib, "memory " + kind)


# ---- the child ---------------------------------------------------------------------------------------

def _main(so, call):
    lim = ctypes.CDLL(so, mode=ctypes.RTLD_GLOBAL)
    lim.alloc_limit_used.restype = lim.alloc_limit_refused.restype = ctypes.c_size_t
    lim.alloc_limit_set.argtypes = [ctypes.c_size_t]
    sys.path[:0] = [os.path.dirname(HERE), HERE]
    from selas_amd import native as N
    from selas_amd import workloads as W
    from test_curve_tree_gpu import _strand

    ctx = N.Context(0)
    ctx.set_tuning(vcm_wavefront_paths=1 << 12)
    soup = lambda seed, n: N.gen_cluster_soup(seed, 16, n // 16, 0.1, 1e-2, 1e-1)
    cam = N.gen_camera_rays(W.CAMERA_POS, W.CAMERA_LOOK_AT, W.CAMERA_UP, 50.0, 800, 800, 1)
    strands = _strand(1, 2000)

    def scene(c, n, curves=False, commit=True):
        s = N.Scene(c)
        s.add_soup(soup(n, n))
        if curves:
            s.add_curves(strands, np.arange(2000, dtype=np.uint32))
        if commit:
            s.commit()
        return s

    def hits(s):
        lim_off()
        dr, dh = N.DeviceRays(ctx, cam), N.DeviceHits(ctx, cam["org_x"].size)
        s.intersect(dr, dh)
        N.synchronize()
        return dh.to_host()

    lim_off = lambda: lim.alloc_limit_set(ctypes.c_size_t(-1).value)
    if call.startswith("memory"):
        kind, n = call.split()[1], 64000
        s = N.Scene(ctx)
        if kind == "triangles":
            s.add_soup(soup(1, n))
        elif kind == "curves":
            for k in range(n // 2000):
                s.add_curves(strands + np.float32([0.1 * k, 0, 0, 0]), np.arange(2000, dtype=np.uint32))
        else:
            model, n = scene(ctx, 16), 400000
            m = np.eye(4, dtype=np.float32).reshape(-1)
            for k in range(n):
                m[12:15] = (k % 71, k // 71 % 73, k // 5183)
                N.check(N.lib.sgpu_scene_add_instance(s.handle, model.handle, N.fptr(m), None))
        lim.alloc_limit_set(lim.alloc_limit_used() + COMMIT_BYTES[kind] * n)
        s.commit()
        lim_off()
        print(f"{call}: ok", flush=True)
        return
    sc = W.room_scene(1)
    room = N.build_render_scene(ctx, sc)
    bare = scene(ctx, 1600)  # (a small scratch block for the calls that take one)
    with_curves = scene(ctx, 1600, curves=True)
    drays, dhits = N.DeviceRays(ctx, cam), N.DeviceHits(ctx, cam["org_x"].size)
    occ = ctx.empty(4 * drays.n)
    frame = ctx.empty(12 * 32 * 32)
    other = N.Context(0)
    for c in (ctx, other):
        scene(c, 3200, curves=True).release()  # scratch for the small commits below
    scene(ctx, 3200000).release()  # 1.8 GB more that stay idle
    job = {"camera": sc["camera"], "width": 32, "height": 32, "iterations": 1, "max_path_length": 5, "base_radius": 0.05,
           "radius_alpha": 0.75, "seed": 3}

    if call.startswith("refused"):
        def make():
            s = N.Scene(ctx)
            if call == "refused instances":
                for k in range(500):
                    m = np.eye(4)
                    m[:3, 3] = (k % 13, k // 13, 0)
                    s.add_instance(bare if k % 250 else with_curves, m)
                return s
            s.release()
            return scene(ctx, 3200, curves=call == "refused curves", commit=False)

        want_scene = make()
        want_scene.commit()
        want = hits(want_scene)
        s = make()

        def held():  # with the idle blocks given back
            lim.alloc_limit_set(1)
            with pytest.raises(N.SgpuError):
                ctx.empty(1 << 20)
            return lim.alloc_limit_used()

        before, refusals, codes = held(), 0, set()
        for slack in range(0, 1 << 24, 24 << 10):
            lim.alloc_limit_set(before + slack)
            try:
                s.commit()
                break
            except N.SgpuError as e:
                assert e.code in (N.SGPU_E_NOMEM, N.SGPU_E_HIP), str(e)
                codes.add(e.code)
            refusals += 1
            assert held() == before, (slack, before, lim.alloc_limit_used())
        assert refusals > 20
        assert N.SGPU_E_NOMEM in codes  # the records' allocation says what it was
        got = hits(s)
        for k in want:
            assert np.array_equal(got[k].view(np.uint32), want[k].view(np.uint32)), k
        print(f"{call}: ok after {refusals} refusals", flush=True)
        return

    def vcm():
        N.render_vcm(room, sc["camera"], 32, 32, 1, 5, 0.05, 0.75, 3, framebuffer=frame)
        return {"image": frame.download(np.float32, 3 * 32 * 32)}

    def server():
        sv = N.VcmServer(ctx, 1 << 12, 5)
        sv.submit(room, job, frame)
        while sv.step()[1]:
            pass
        N.synchronize()
        sv.close()
        return {"image": frame.download(np.float32, 3 * 32 * 32)}

    def instances():
        s = N.Scene(ctx)
        for k in range(2000):
            m = np.eye(4)
            m[:3, 3] = (k % 13, k // 13 % 13, k // 169)
            s.add_instance(bare, m)
        s.commit()
        return hits(s)

    def materials():
        fresh = scene(ctx, 1600)
        m = np.ascontiguousarray(np.tile(np.asarray(sc["materials"], np.float32)[:1], (4000, 1)))
        gm = np.zeros(1, np.uint32)
        lim_set()
        N.check(N.lib.sgpu_scene_set_materials(fresh.handle, N.fptr(m), 4000, N.uptr(gm), 1))

    def attributes():
        fresh = scene(ctx, 160000, commit=False)
        lim_set()
        fresh.set_vertex_attributes(0, 480000, normals=np.ones((480000, 3), np.float32))

    def texture():
        fresh = N.Scene(ctx)
        fresh.add_quads(np.array([[0, 0, 0], [1, 0, 0], [1, 1, 0], [0, 1, 0]], np.float32), np.arange(4, dtype=np.uint32))
        lim_set()
        fresh.set_ptex(0, 8, np.zeros(3 << 16, np.uint8), np.full((1, 4), -1, np.int32), np.zeros((1, 4), np.int32))

    def intersect(s):
        s.intersect(drays, dhits)
        N.synchronize()
        return dhits.to_host()

    def hdr():
        N.save_hdr(ctx, os.path.join(os.path.dirname(so), "frame"), big_frame, 640, 640)

    def pool():
        s = scene(ctx, 80000)
        return hits(s)

    lim_set = lambda: lim.alloc_limit_set(lim.alloc_limit_used() + 4096)
    big_frame = ctx.empty(12 * 640 * 640)
    run, late = {
        "commit": (lambda: hits(scene(ctx, 3200)), False), "commit curves": (lambda: hits(scene(ctx, 3200, curves=True)), False),
        "commit instances": (instances, False), "other context": (lambda: hits(scene(other, 3200)), False),
        "materials": (materials, True), "attributes": (attributes, True), "texture": (texture, True),
        "ibl": (lambda: room.set_ibl(np.ones((64, 128, 3), np.float32)), False),
        "query": (lambda: intersect(bare), False), "curve query": (lambda: intersect(with_curves), False),
        "stats": (lambda: bare.intersect_stats(drays, any_hit=True) and None, False),
        "vcm": (vcm, False), "server": (server, False), "hdr": (hdr, False),
        "pool": (pool, False)}[call]
    if call == "pool":  # a server's arrays, freed to the pool, and no scratch block left idle
        sv = N.VcmServer(ctx, 1 << 16, 10)
        sv.close()
        N.synchronize()
        N.check(N.lib.sgpu_context_destroy(other.handle))
        lim.alloc_limit_set(1)
        try:
            ctx.empty(1 << 20)
        except N.SgpuError:
            pass
        lim_off()
        sv = N.VcmServer(ctx, 1 << 16, 10)
        sv.close()
        N.synchronize()
    if not late:
        lim_set()
    before = lim.alloc_limit_refused()
    got = run()
    lim_off()
    assert lim.alloc_limit_refused() > before, "the call met no limit"
    want = run() if not late else None
    if isinstance(got, dict):
        for k in got:
            # images add their splats in no fixed order
            np.testing.assert_allclose(got[k], want[k], rtol=1e-5 if k == "image" else 0, atol=1e-6 if k == "image" else 0,
                                       err_msg=k)
    print(f"{call}: ok", flush=True)


if __name__ == "__main__":
    _main(sys.argv[1], sys.argv[2])
