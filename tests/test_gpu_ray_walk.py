"""The raycast walk at the places where its order or its skipping could show: trees deeper
than its stack, grazing rays, distant origins, directions and orientations that are not
normalised (walked in the tree's order), batches that end within a wave. Against the
oracle's Scene::raycastClosest on the same state, bit for bit."""
import numpy as np
import pytest

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
    return (target + away * reach + side * offset).astype(np.float32), d.astype(np.float32)


@pytest.mark.parametrize("scene,kind,n", [("deep", "near", 1), ("deep", "near", 257), ("deep", "length", 65),
                                          ("mixed", "graze", 1023), ("mixed", "far", 1000), ("mixed", "length", 300),
                                          ("loose", "near", 500)])
def test_walk_matches_oracle(scene, kind, n):
    log(f"[ray walk] {scene}, {kind}, {n} rays")
    sc = {"deep": _deep, "mixed": _mixed, "loose": _loose}[scene]()
    g, o = lockstep(sc, 10 if scene == "mixed" else 0)
    origins, dirs = _rays(kind, sc, np.random.default_rng(n), n)
    for maxd in (3e5, 20.0):
        gc, gt, _ = g.raycast(origins, dirs, maxd)
        oc, ot = o.raycast(origins, dirs, np.full(n, maxd, np.float32))
        assert np.array_equal(gc, oc)
        assert np.array_equal(bits(gt[gc >= 0]), bits(ot[gc >= 0]))
    assert (gc >= 0).any() or kind == "far"
