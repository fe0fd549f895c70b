"""Scenes whose 8-wide trees are deep: content in the seven outer octants of a cube at the origin, of the
eighth's, of that one's eighth's, and so on. An octant level is one level of the 8-wide tree, and rays
from the origin outwards pass an inner octant and an outer one on every level, so that the stacks of a
traversal fill."""
import ctypes as C
import itertools

import numpy as np

from selas_amd import native as N

# a lane's stack words: these many are in LDS, and above kMostGroupWords small launches go lane by lane
LDS_WORDS = 16
MOST_GROUP_WORDS = 34


def stack_words(scene):
    f = N.lib._Z22sgpu_trace_stack_wordsP12sgpu_scene_s
    f.argtypes, f.restype = [C.c_void_p], C.c_uint32
    return f(scene.handle)


def octants(levels):
    """(corner, side) of every octant, the innermost cube last."""
    out = []
    for k in range(levels):
        h = 2.0 ** -(k + 1)
        out += [(h * np.array(c, float), h) for c in itertools.product((0, 1), repeat=3) if any(c)]
    return out + [(np.zeros(3), 2.0 ** -levels)]


def nested_soup(seed, levels, per=16, core=0):
    """`per` triangles in each octant, and one more triangle `core` times in the innermost, for a few more
    levels (the octants themselves stop at the builder's growth of all boxes, 2^-18 of the scene)."""
    rng = np.random.default_rng(seed)
    tris = [(corner + h * rng.random((per, 1, 3)) + rng.normal(scale=0.12 * h, size=(per, 3, 3))).reshape(per, 9)
            for corner, h in octants(levels)]
    tris.append(np.tile(2.0 ** -levels * np.array([[0.5, 0.4, 0.4, 0.4, 0.5, 0.4, 0.4, 0.4, 0.5]]), (core, 1)))
    return np.concatenate(tris).astype(np.float32)


def nested_strands(seed, levels, per=16):
    """Curve vertices and segment indices: a strand of `per` segments in each octant."""
    rng = np.random.default_rng(seed)
    verts, idx = [], []
    for corner, h in octants(levels):
        step = rng.normal(size=(per + 3, 3))
        walk = np.cumsum(step / np.linalg.norm(step, axis=1, keepdims=True) * 0.1 + [0.03, 0.02, 0.01], axis=0)
        idx.append(np.arange(per) + (per + 3) * len(verts))
        verts.append(np.concatenate([corner + h * (0.2 + 0.6 * walk / 1.5), np.full((per + 3, 1), 0.01 * h)], 1))
    return np.concatenate(verts).astype(np.float32), np.concatenate(idx).astype(np.uint32)


def rays(seed, n, levels):
    """Half outwards from about the origin, half of those past hits nearer than a random octant level; a
    quarter inwards from a random level's octants; a quarter anywhere. (Rays that come a long way to the
    smallest triangles would be bent by more than the boxes' growth in the triangle test's rounding.)"""
    rng = np.random.default_rng(seed)
    kind = rng.integers(0, 4, n)
    scale = 2.0 ** -rng.integers(0, levels + 1, (n, 1)).astype(float)
    out = rng.random((n, 3)) * np.where(kind[:, None] < 2, 2.0 ** -levels, scale / 8)
    o = np.choose(kind[:, None], [out, out, scale * rng.uniform(0.5, 2.0, (n, 3)), rng.uniform(-1.0, 2.0, (n, 3))])
    d = np.choose(kind[:, None], [0.2 + rng.random((n, 3)), 0.2 + rng.random((n, 3)), out - o, rng.normal(size=(n, 3))])
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    tnear = np.where(kind == 0, 2.0 ** -rng.integers(0, levels + 1, n).astype(float), 0.0)
    tfar = np.where(rng.random(n) < 0.2, tnear + rng.random(n), np.inf)
    f = lambda a: np.ascontiguousarray(a, np.float32)
    return {"org_x": f(o[:, 0]), "org_y": f(o[:, 1]), "org_z": f(o[:, 2]), "dir_x": f(d[:, 0]), "dir_y": f(d[:, 1]),
            "dir_z": f(d[:, 2]), "tnear": f(tnear), "tfar": f(tfar)}


def placed(r, l2w):
    """The rays carried by a 4 x 4 local-to-world matrix."""
    o = np.stack([r["org_x"], r["org_y"], r["org_z"]], 1) @ l2w[:3, :3].T + l2w[:3, 3]
    d = np.stack([r["dir_x"], r["dir_y"], r["dir_z"]], 1) @ l2w[:3, :3].T
    f = lambda a: np.ascontiguousarray(a, np.float32)
    return dict(r, org_x=f(o[:, 0]), org_y=f(o[:, 1]), org_z=f(o[:, 2]), dir_x=f(d[:, 0]), dir_y=f(d[:, 1]), dir_z=f(d[:, 2]))
