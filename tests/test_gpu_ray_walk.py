"""The raycast walk at the places where its order or its skipping could show: trees deeper
than its stack, grazing rays, distant origins, directions and orientations that are not
normalised (nothing is skipped) or very long (walked in the tree's order), batches that end within a wave, capsules whose
bounds reach far from them. Against the oracle's Scene::raycastClosest on the same state, bit
for bit."""
import numpy as np
import pytest

import oracle_lib as ol
from gpu_util import bits, lockstep, log
from physecs_amd import scenes

pytestmark = pytest.mark.gpu


def _deep():
    """Morton codes with one further bit each and 64 equal ones: a path of more than 30 nodes,
    all of whose boxes overlap."""
    sc = scenes.Scene()
    at = [[0, 0, 0]] * 64 + [[1, 1, 1]] * 64
    for k in range(2, 10):
        at += [[2.0 ** -k, 0, 0], [0, 2.0 ** -k, 0], [0, 0, 2.0 ** -k]]
    for i, p in enumerate(at):
        sc.add_body(scenes.SPHERE, [4.0 + 0.01 * (i * 37 % 61)], p)
    sc.add_static(scenes.BOX, [20, 0.5, 20], [0, -9, 0])
    return sc


def _mixed():
    return scenes.mixed_lattice(3, side=7)


def _loose():
    """Orientations that are not unit quaternions."""
    sc = scenes.Scene()
    rng = np.random.default_rng(8)
    for i in range(60):
        q = rng.normal(size=4)
        q *= rng.uniform(0.9, 1.1) / np.linalg.norm(q)
        kind = (scenes.SPHERE, scenes.CAPSULE, scenes.BOX)[i % 3]
        sc.add_body(kind, [[0.5], [0.5, 0.3], [0.4, 0.2, 0.6]][i % 3], rng.uniform(-4, 4, 3), q)
    return sc


def _rays(kind, sc, rng, n):
    pos = sc.arrays()["pos"].reshape(-1, 3)[:sc.n_actors]
    target = pos[rng.integers(0, len(pos), n)].astype(np.float64)
    away = rng.normal(size=(n, 3))
    away /= np.linalg.norm(away, axis=1, keepdims=True)
    side = np.cross(away, rng.normal(size=(n, 3)))
    side /= np.linalg.norm(side, axis=1, keepdims=True)
    reach = 10.0 ** rng.uniform(0, 5 if kind == "far" else 1.5, (n, 1))
    offset = {"graze": 0.5 + 1e-4 * rng.normal(size=(n, 1))}.get(kind, rng.uniform(0, 0.5, (n, 1)))
    d = -away * (rng.uniform(0.5, 2.0, (n, 1)) if kind == "length" else 1.0)
    if kind == "odd":     # lengths of 1 among very short and long ones and none at all
        d *= 10.0 ** np.where(rng.random((n, 1)) < 0.3, 0, rng.uniform(-4, 8, (n, 1)))
        d[::17] = 0
    return (target + away * reach + side * offset).astype(np.float32), d.astype(np.float32)


def _same(g, o, origins, dirs, maxd):
    gc, gt, _ = g.raycast(origins, dirs, maxd)
    oc, ot = o.raycast(origins, dirs, np.full(len(origins), maxd, np.float32))
    assert np.array_equal(gc, oc), np.flatnonzero(gc != oc)
    assert np.array_equal(bits(gt[gc >= 0]), bits(ot[gc >= 0]))
    return oc, ot


@pytest.mark.parametrize("scene,kind,n", [("deep", "near", 1), ("deep", "near", 257), ("deep", "length", 65),
                                          ("mixed", "graze", 1023), ("mixed", "far", 1000), ("mixed", "length", 300),
                                          ("loose", "near", 500), ("mixed", "odd", 900), ("deep", "odd", 200)])
def test_walk_matches_oracle(scene, kind, n):
    log(f"[ray walk] {scene}, {kind}, {n} rays")
    sc = {"deep": _deep, "mixed": _mixed, "loose": _loose}[scene]()
    g, o = lockstep(sc, 10 if scene == "mixed" else 0)
    origins, dirs = _rays(kind, sc, np.random.default_rng(n), n)
    for maxd in (3e5, 20.0):
        c, _ = _same(g, o, origins, dirs, maxd)
    assert (c >= 0).any() or kind == "far"


def test_capsule_met_behind_the_origin():
    """The line meets the tilted capsule behind the origin, which is a hit at 0; its bounds are
    entered 8.5 m ahead, behind a sphere that is met at 2.7 m."""
    sc = scenes.Scene()
    d = np.array([-1, -1.5, 0]) / np.hypot(1, 1.5)
    o = np.array([12.0, 1, 0])
    sc.add_body(scenes.CAPSULE, [10, 0.1], [0, 0, 0], [0, 0, np.sin(-np.pi / 8), np.cos(-np.pi / 8)])
    sc.add_body(scenes.SPHERE, [0.3], o + 3 * d)
    c, t = _same(*lockstep(sc, 0), np.array([o], np.float32), np.array([d], np.float32), 200.0)
    assert c[0] == 0 and t[0] == 0


@pytest.mark.parametrize("half", [0.5, 1.0, 6.0, 10.0])
def test_rays_that_start_beside_poles(half):
    """The same of random poles, each alone with 48 balls: rays from beside the pole, on a line
    that comes from its axis beyond the end, each with a ball a little way ahead."""
    rng = np.random.default_rng(int(10 * half))
    ahead = 0
    for _ in range(20):
        sc = scenes.Scene()
        a = rng.normal(size=3)
        a /= np.linalg.norm(a)
        q = np.array([a[2], 0, -a[0], 1 + a[1]])      # the turn that takes the y axis to a
        sc.add_body(scenes.CAPSULE, [half, 0.02 * half], [0, 0, 0], q / np.linalg.norm(q))
        p = np.cross(rng.normal(size=(48, 3)), a)
        end = a * half * rng.choice([-1, 1], (48, 1))
        origins = end * rng.uniform(0, 0.9, (48, 1)) + \
            p / np.linalg.norm(p, axis=1, keepdims=True) * half * rng.uniform(0.05, 0.6, (48, 1))
        dirs = origins - end * rng.uniform(1.05, 2.0, (48, 1))
        dirs /= np.linalg.norm(dirs, axis=1, keepdims=True)
        for at in origins + dirs * half * rng.uniform(0.02, 0.2, (48, 1)):
            sc.add_body(scenes.SPHERE, [0.01 * half], at)
        origins, dirs = origins.astype(np.float32), dirs.astype(np.float32)
        g, o = lockstep(sc, 0)
        c, t = _same(g, o, origins, dirs, 200.0)
        mn, mx = o.bounds()[0, :3], o.bounds()[0, 3:]
        entry = (np.minimum((mn - origins) / dirs, (mx - origins) / dirs)).max(1)
        ahead += ((c == 0) & (t == 0) & (entry > 0.3 * half)).sum()
    assert ahead > 5


@pytest.mark.parametrize("at", [2.0 ** 20, -2.0 ** 20, 2.0 ** 23, 1e8])
def test_far_from_the_worlds_origin(at):
    """The nearer sphere's box is rounded to begin behind the other sphere's surface: 9.75 or 10
    for 9.7, with a hit at 9.72 before it (both at 2^20 and 2^23; rounded further at 1e8)."""
    sc = scenes.Scene()
    sc.add_body(scenes.SPHERE, [1.3], [at + 11, 0, 0])
    sc.add_body(scenes.SPHERE, [0.28], [at + 10, 0, 0])
    g, o = lockstep(sc, 0)
    for origin, d in ((at, 1), (at + 21, -1)):
        _same(g, o, np.array([[origin, 0, 0]], np.float32), np.array([[d, 0, 0]], np.float32), 200.0)


def _prism():
    """A box's faces without the top one: the half-spaces of the others have no upper end."""
    v, f, n, c = scenes.convex_hull(np.array([[x, y, z] for x in (-1, 1) for y in (-1, 1) for z in (-1, 1)], float))
    keep = [k for k in range(len(f)) if n[k][1] < 0.5]
    return v, [f[k] for k in keep], n[keep], c[keep]


def test_hull_that_its_faces_do_not_close():
    """The ray meets a side's plane above the bounds, at 4.12 m, and enters them 7.2 m ahead,
    behind a sphere that is met at 5.2 m."""
    sc = scenes.Scene()
    sc.add_convex_body(sc.add_convex_mesh(*_prism()), [0, 0, 0])
    sc.add_body(scenes.SPHERE, [0.2], [-0.7, 2.8, 0])
    d = np.array([1, -4, 0.01]) / np.sqrt(17.0001)
    c, t = _same(*lockstep(sc, 0), np.array([[-2, 8, 0]], np.float32), d[None].astype(np.float32), 200.0)
    assert c[0] == 0 and 4 < t[0] < 4.2


@pytest.mark.parametrize("scale", [(1, 1, 1), (1, -0.5, 2), (1, 0.002, 1), (0.001, 1, 0.001)])
def test_hulls_of_any_scale(scale):
    """Rays past the rims of hulls, flat and needle-like ones too, with spheres around them."""
    rng = np.random.default_rng(9)
    sc = scenes.Scene()
    mesh = sc.add_convex_mesh(*scenes.ellipsoid_hull(rng))
    at, q = rng.uniform(-3, 3, (40, 3)), scenes.random_quats(rng, 40)
    for k in range(40):
        sc.add_convex_body(mesh, at[k], q[k], scale)
        sc.add_body(scenes.SPHERE, [0.1], at[k] + rng.uniform(-0.8, 0.8, 3))
    g, o = lockstep(sc, 0)
    origins = rng.uniform(-8, 8, (2000, 3))
    dirs = at[rng.integers(0, 40, 2000)] + rng.uniform(-0.4, 0.4, (2000, 3)) * np.abs(scale) - origins
    dirs /= np.linalg.norm(dirs, axis=1, keepdims=True)
    _same(g, o, origins.astype(np.float32), dirs.astype(np.float32), 200.0)


def test_poses_written_without_bounds():
    """write_state moves bodies and leaves their bounds, which rays go on to enter, as they were:
    a hit can lie far before its collider's box."""
    rng = np.random.default_rng(4)
    sc = scenes.Scene()
    n = 60
    for at in rng.uniform(-6, 6, (n, 3)):
        sc.add_body(scenes.SPHERE, [0.5], at)
    g, o = lockstep(sc, 0)
    box = o.bounds()
    pos = g.state()[0]
    pos[:, 0] -= rng.uniform(0, 6, n).astype(np.float32)
    g.write_state(pos=pos)
    origins = rng.uniform(-8, 8, (400, 3)).astype(np.float32)
    origins[:, 0] = -20
    dirs = np.tile(np.float32([[1, 0, 0]]), (400, 1))
    gc, gt, _ = g.raycast(origins, dirs, 200.0)
    jumps = 0
    for k in range(len(origins)):
        best, dist, first = -1, 0.0, np.inf
        for c in range(n):
            met, entry = ol.ray_aabb("orc", origins[k], dirs[k], box[c, :3], box[c, 3:])
            hit, t = ol.ray_geometry("orc", origins[k], dirs[k], scenes.SPHERE, [0.5], pos[c], [0, 0, 0, 1])
            if met and hit and (best < 0 or t < dist):
                best, dist, first = c, t, entry
        assert gc[k] == best and bits(gt[k]) == bits(np.float32(dist)), k
        jumps += best >= 0 and first > dist + 1
    assert jumps > 20
