"""The narrowphase with a wave per convex or triangle-mesh pair, where its loops change over:
hulls with more vertices than a wave has lanes (a support query in two rounds, more than 64
faces) and with four, smooth shapes that run EPA to its end, a body over more candidate
triangles than a wave has lanes, and a BVH stored in another order than its triangles'."""
import struct

import numpy as np
import pytest

from gpu_util import lockstep, log
from physecs_amd import api, scenes

pytestmark = pytest.mark.gpu


def _hull(rng, points, lo=0.3, hi=0.6):
    return scenes.ellipsoid_hull(rng, n_points=points, lo=lo, hi=hi)


@pytest.mark.parametrize("points", [4, 24, 63, 65, 130])
def test_hull_sizes_lockstep_bitexact(points):
    rng = np.random.default_rng(points)
    sc = scenes.Scene()
    sc.add_static(scenes.BOX, [20, 0.5, 20], [0, -0.5, 0])
    meshes = [sc.add_convex_mesh(*_hull(rng, points)) for _ in range(3)]
    for i in range(24):
        p = [rng.uniform(-1.2, 1.2), 0.6 + 0.35 * i, rng.uniform(-1.2, 1.2)]
        q = scenes.random_quats(rng, 1)[0]
        k = i % 6
        if k < 3:
            sc.add_convex_body(meshes[k], p, q, scale=(1, 1, 1) if i < 12 else tuple(rng.uniform(0.6, 1.4, 3)))
        else:
            sc.add_body(k - 3, {0: [0.35], 1: [0.3, 0.2], 2: [0.3, 0.2, 0.35]}[k - 3], p, q)
    log(f"[wave] hulls of {points} points, 45 steps")
    lockstep(sc, 45, check_every=5)


@pytest.mark.parametrize("kind", ["convex", "box", "capsule", "sphere"])
def test_many_candidate_triangles_lockstep_bitexact(kind):
    """One large body over a fine terrain: 65 to 256 candidates."""
    rng = np.random.default_rng(5)
    sc = scenes.Scene()
    verts, tris, _ = scenes.terrain_mesh(3, quads=24, spacing=0.25, amplitude=0.3)
    tm = sc.add_triangle_mesh(verts, tris)
    sc.add_collider(sc.add_actor([0, 0, 0]), scenes.TRIANGLE_MESH, [0, 0, 0, float(tm)])
    p = [0.1, 1.4, 0.05]
    if kind == "convex":
        sc.add_convex_body(sc.add_convex_mesh(*_hull(rng, 24, 0.9, 1.2)), p, scenes.random_quats(rng, 1)[0])
    else:
        prm = {"box": (scenes.BOX, [0.9, 0.5, 0.8]), "capsule": (scenes.CAPSULE, [0.6, 0.5]),
               "sphere": (scenes.SPHERE, [1.0])}[kind]
        sc.add_body(prm[0], prm[1], p, scenes.random_quats(rng, 1)[0])
    g, _ = lockstep(sc, 60, check_every=5)
    assert g.counts()["manifolds"] > 0


def _fnv(data):
    h = 1469598103934665603
    for b in data:
        h = ((h ^ b) * 1099511628211) & 0xFFFFFFFFFFFFFFFF
    return h


def test_mesh_stored_out_of_order_gives_the_same_manifolds():
    """The root's children exchanged: the walk meets the triangles in another order, the same
    triangles touch."""
    sc = scenes.terrain_drop(11, quads=8, n=24)
    v, t = sc.trimesh[0]
    raw = bytearray(api.trimesh_cache(v, t))
    magic, version, nv, nt, nodes, depth, size, mesh_hash, _ = struct.unpack_from("<IIiiiiQQQ", raw)
    first = 48 + 3 * 16 * nt
    a, b = first + 32, first + 64              # nodes 1 and 2: the root's children
    raw[a:a + 32], raw[b:b + 32] = raw[b:b + 32], raw[a:a + 32]
    struct.pack_into("<Q", raw, 40, _fnv(bytes(raw[48:])))
    assert api.trimesh_cache_validate(v, t, bytes(raw)) == 0
    got = []
    for cache in (None, bytes(raw)):
        sc.tri_bvh_cache = [cache]
        w = api.World(sc, substeps=4, iterations=2)
        seen = []
        for _ in range(30):
            w.step(1 / 60)
            keys, ints, f = w.manifolds()
            order = np.lexsort(keys.T[::-1])
            seen.append((keys[order], ints[order][:, 2], f[order][:, :28]))
            if len(keys):
                break
        got.append(seen)
    assert len(got[0]) == len(got[1]) and len(got[0][-1][0]) > 0
    for x, y in zip(*got):
        for p, q in zip(x, y):
            assert np.array_equal(p, q)
