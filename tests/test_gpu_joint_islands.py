"""Joint islands at the edges of a workgroup's pass: fewer and more joints than one pass
stages (32), colours that end inside a pass, every joint type, joints to a static body.
In lockstep with the oracle, bit for bit."""
import numpy as np
import pytest

from gpu_util import lockstep, log
from physecs_amd import scenes

pytestmark = pytest.mark.gpu


def _web(n, seed):
    """A chain of n joints of every type in turn, its bodies also joined to a hub that hangs
    from a static body: two to eight colours, joints of 3 to 7 rows."""
    rng = np.random.default_rng(seed)
    sc = scenes.Scene()
    top = sc.add_static(scenes.BOX, [0.2, 0.2, 0.2], [0, 8, 0])
    hub = sc.add_body(scenes.SPHERE, [0.3], [0, 7, 0])
    sc.add_joint(scenes.REVOLUTE, top, hub, (0, -0.5, 0), (0, 0.5, 0), drive=(1.5, 20.0))
    kinds = (scenes.SPHERICAL, scenes.REVOLUTE, scenes.PRISMATIC, scenes.UNIVERSAL, scenes.FIXED, scenes.SERVO,
             scenes.GEAR)
    prev = hub
    for i in range(n):
        at = [0.5 * (i + 1), 7 + 0.3 * (i % 2), 0.1 * (i % 3)]
        body = sc.add_body(scenes.BOX, [0.1, 0.1, 0.1], at, vel=rng.normal(size=3))
        args = {}
        if kinds[i % 7] == scenes.PRISMATIC:
            args = dict(lower_limit=-0.05, upper_limit=0.02, target=0.01, drive_enabled=1)
        sc.add_joint(kinds[i % 7], prev, body, (0.25, 0, 0), (-0.25, 0, 0), **args)
        if 0 < i < 6:
            sc.add_joint(scenes.SPHERICAL, hub, body, (0.1 * i, 0, 0), (0, 0.2, 0))
        prev = body
    return sc


@pytest.mark.parametrize("n", [1, 26, 27, 33, 62, 250])
def test_islands_lockstep_bitexact(n):
    log(f"[islands] a web of {n} bodies")
    lockstep(_web(n, n), 25, check_every=5)


@pytest.mark.parametrize("n", [33, 34, 65, 66, 140])
def test_chains_lockstep_bitexact(n):
    """Two colours: up to 64 joints are two chunks of an island's pass, more are solved in a
    launch per colour."""
    log(f"[islands] a chain of {n} bodies")
    sc = scenes.Scene()
    sc.add_static(scenes.BOX, [60, 0.5, 20], [0, -0.5, 0])
    scenes.capsule_chain(sc, [-n / 4, 0.6, 0], n=n)
    lockstep(sc, 20, check_every=5)


def test_islands_of_different_sizes_lockstep_bitexact():
    sc = _web(5, 2)
    for k in range(9):
        a = sc.add_body(scenes.BOX, [0.1, 0.1, 0.1], [0, 2.0 * k, 5])
        b = sc.add_body(scenes.BOX, [0.1, 0.1, 0.1], [0.4, 2.0 * k, 5])
        sc.add_joint(scenes.REVOLUTE, a, b, (0.2, 0, 0), (-0.2, 0, 0))
    lockstep(sc, 20, check_every=5)
