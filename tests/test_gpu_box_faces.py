"""Face contacts of box pairs, eight lanes a pair: polygons of three to eight corners, corners
on the reference face's sides, thin and very unequal boxes, either box's face as the
reference, around the number of pairs a workgroup takes (32). In lockstep with the oracle,
bit for bit."""
import numpy as np
import pytest

from gpu_util import lockstep, log
from physecs_amd import scenes

pytestmark = pytest.mark.gpu


def _pairs(n, kind, seed):
    rng = np.random.default_rng(seed)
    sc = scenes.Scene()
    for i in range(n):
        at = np.array([6.0 * (i % 8), 0.0, 6.0 * (i // 8)])
        h0, h1 = rng.uniform(0.3, 1.0, 3), rng.uniform(0.3, 1.0, 3)
        yaw, tilt, off = rng.uniform(0, 2 * np.pi), 0.02 * rng.normal(), rng.uniform(-0.6, 0.6, 2)
        if kind == "aligned":      # sides and corners coincide
            h1, yaw, tilt, off = h0.copy(), (i % 4) * np.pi / 2, 0.0, np.array([0.0, h0[2]]) * (i % 2)
        elif kind == "octagon":    # 45 degrees: eight corners
            h0[:] = h1[:] = 0.5
            yaw, tilt, off = np.pi / 4, 0.0, np.zeros(2)
        elif kind == "unequal":    # a plate on a needle, a needle on a plate
            h0, h1 = (np.array([1.5, 0.02, 1.5]), np.array([0.02, 0.6, 0.02])) if i % 2 else \
                     (np.array([0.02, 0.6, 0.02]), np.array([1.5, 0.02, 1.5]))
        q = np.array([np.sin(tilt / 2), np.cos(tilt / 2) * np.sin(yaw / 2), 0.0, np.cos(tilt / 2) * np.cos(yaw / 2)])
        q /= np.linalg.norm(q)
        top = at + [off[0], h0[1] + h1[1] - 0.01, off[1]]
        lower = sc.add_static if i % 3 else sc.add_body
        if i % 5 == 0:             # the other order of the pair
            sc.add_body(scenes.BOX, h1, top, q)
            lower(scenes.BOX, h0, at)
        else:
            lower(scenes.BOX, h0, at)
            sc.add_body(scenes.BOX, h1, top, q)
    return sc


@pytest.mark.parametrize("kind", ["turned", "aligned", "octagon", "unequal"])
@pytest.mark.parametrize("n", [1, 31, 33, 70])
def test_box_faces_lockstep_bitexact(kind, n):
    log(f"[box faces] {n} pairs, {kind}")
    lockstep(_pairs(n, kind, n), 6)
