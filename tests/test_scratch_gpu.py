"""Calls share their context's scratch blocks one after another, never at the same time: images and
trees made by several threads on streams of their own equal those made alone, whatever sizes the
blocks were last used for."""
import ctypes as C
import threading

import numpy as np
import pytest

from selas_amd import native as N
from selas_amd import workloads as W

pytestmark = pytest.mark.gpu

SIZES = [(64, 48, 4), (17, 9, 1), (96, 96, 9), (64, 48, 4)]


def _stream():
    s = C.c_void_p()
    N.check(N.lib.sgpu_stream_create(C.byref(s)))
    return s


def test_threads_render_and_commit_as_alone(gpu_ctx):
    sc = W.room_scene(3)
    scene = N.build_render_scene(gpu_ctx, sc)
    soup = W.traversal_scene(0.02)
    infos = []

    def image(k, stream=None):
        w, h, spp = SIZES[k]
        return N.render_pt(scene, sc["camera"], w, h, spp, 6, 11 + k, stream=stream)

    def commit(stream=None):
        s = N.Scene(gpu_ctx)
        s.add_soup(soup)
        s.commit(stream)
        infos.append(s.info())
        s.release()

    alone = [image(k) for k in range(len(SIZES))]
    commit()
    got = [None] * len(SIZES)

    def work(k):
        st = _stream()
        for _ in range(3):
            got[k] = image(k, st)
            commit(st)
        N.check(N.lib.sgpu_stream_destroy(st))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(len(SIZES))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for k in range(len(SIZES)):
        assert np.array_equal(got[k].view(np.uint32), alone[k].view(np.uint32)), SIZES[k]
    assert all(i == infos[0] for i in infos)
    scene.release()
