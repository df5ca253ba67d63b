"""The triangle-mesh passes keep the candidate triangles of all pairs in one list. Where it is
too short for a call's candidates, an MTD query asks again with a longer one, and beyond 2^24 of
them query by query range; it must give what the same queries give in smaller calls. A step
raises the capacity error."""
import numpy as np
import pytest

from gpu_util import bits, log
from physecs_amd import scenes

pytestmark = pytest.mark.gpu
INITIAL = 1 << 18    # slots of the first attempt and of a small world's step


N, CELL = 61, 0.2


def _carpet(sc):
    """A flat mesh of N x N vertices around the origin; returns its index."""
    n = N
    x = (np.arange(n) - (n - 1) / 2) * CELL
    gx, gz = np.meshgrid(x, x, indexing="ij")
    a = (np.arange(n - 1)[:, None] * n + np.arange(n - 1)).ravel()
    tris = np.concatenate([np.stack([a, a + 1, a + n], 1), np.stack([a + 1, a + n + 1, a + n], 1)])
    return sc.add_triangle_mesh(np.stack([gx.ravel(), np.zeros(n * n), gz.ravel()], 1), tris)


def _under(mn, mx):
    """The mesh's triangles whose bounds overlap these boxes, which reach through y = 0."""
    n = 2.0
    for k in (0, 2):
        lo, hi = (np.floor(x / CELL + (N - 1) / 2) for x in (mn[:, k], mx[:, k]))
        n = n * (hi - lo + 1)
    return int(n.sum())


def _queries(n, hulls):
    """Boxes (or boxes and hulls in turn) of about 1 m sunk into the mesh, some 100 candidates each."""
    rng = np.random.default_rng(n)
    kinds = np.where(np.arange(n) % 2 * hulls > 0, scenes.CONVEX_MESH, scenes.BOX)
    prm = np.tile(np.float32([0.45, 0.3, 0.45, 0.0]), (n, 1))
    prm[kinds == scenes.CONVEX_MESH, :3] = 0.8
    pos = rng.uniform((-4, 0, -4), (4, 0.25, 4), (n, 3)).astype(np.float32)
    return kinds, prm, pos, scenes.random_quats(rng, n).astype(np.float32)


def _world(hulls):
    from physecs_amd import api
    sc = scenes.Scene()
    sc.add_collider(sc.add_actor([0, 0, 0]), scenes.TRIANGLE_MESH, [0, 0, 0, float(_carpet(sc))])
    if hulls:
        sc.add_convex_mesh(*scenes.ellipsoid_hull(np.random.default_rng(1)))
    sc.add_body(scenes.SPHERE, [0.3], [0, 0.5, 0])
    return api.World(sc)


def _same_in_parts(q, part, hulls):
    n = len(q[0])
    log(f"[candidates] {n} queries, hulls {hulls}, in one call and in calls of {part}")
    whole, parts = _world(hulls), _world(hulls)
    got, _ = whole.overlap_mtd(*q)
    for lo in range(0, n, part):
        for k, (c, m) in enumerate(parts.overlap_mtd(*(x[lo:lo + part] for x in q))[0]):
            assert np.array_equal(c, got[lo + k][0]) and np.array_equal(bits(m), bits(got[lo + k][1])), lo + k
    whole.close()
    parts.close()
    total = sum(len(c) for c, _ in got)
    assert total > n
    return total


@pytest.mark.parametrize("hulls", [0, 1])
def test_more_candidates_than_the_first_list_holds(hulls):
    q = _queries(12007, hulls)
    assert _under(q[2] - 0.24, q[2] + 0.24) > INITIAL     # within every shape's bounds
    _same_in_parts(q, 1000, hulls)


def test_more_candidates_than_a_pass_takes():
    """Spheres of 1.8 m, which overlap some 180 triangles and touch few."""
    from physecs_amd import api
    n = 105001
    pos = np.random.default_rng(2).uniform((-4, 0.7, -4), (4, 0.8, 4), (n, 3)).astype(np.float32)
    assert _under(pos - 0.9, pos + 0.9) > 1 << 24
    q = np.full(n, scenes.SPHERE), np.tile(np.float32([0.9]), (n, 1)), pos, np.tile(np.float32([0, 0, 0, 1]), (n, 1))
    total = _same_in_parts(q, 20000, 0)
    w = _world(0)
    with pytest.raises(api.PgxError, match=f"{total} hits exceed the capacity {total - 1}"):
        w.overlap_mtd(*q, capacity=total - 1)
    w.close()


def test_a_step_with_too_many_candidates_says_so():
    """Spheres that rest on the mesh: many candidates and few contacts."""
    from physecs_amd import api
    sc = scenes.Scene()
    mesh, worlds = _carpet(sc), 48
    at = [[1.3 * i, 0.59, 1.3 * j] for i in range(-4, 5) for j in range(-4, 5)]
    for w in range(worlds):
        sc.add_collider(sc.add_actor([0, 0, 0], world=w), scenes.TRIANGLE_MESH, [0, 0, 0, float(mesh)])
        for p in at:
            sc.add_body(scenes.SPHERE, [0.6], p, world=w)
    at = np.array(at)
    assert worlds * _under(at - 0.59, at + 0.59) > INITIAL
    log(f"[candidates] a step of {worlds * len(at)} spheres on meshes")
    g = api.World(sc)
    with pytest.raises(api.PgxError, match="CAPACITY"):
        g.step(1 / 60)
    g.close()
