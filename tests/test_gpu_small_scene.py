"""Small scenes list and colour their manifolds in one workgroup; larger ones in a launch per
phase. A world's colouring does not depend on the worlds beside it, so the same worlds alone
(one workgroup) and in a batch of more than 4,096 bodies (a launch per phase) must step to the
same bits; and a pile on either side of the limits must be coloured properly and match the
oracle fed its order."""
import numpy as np
import pytest

from gpu_util import bits, lockstep, log
from physecs_amd import scenes

pytestmark = pytest.mark.gpu


def test_worlds_alone_and_in_a_large_batch():
    from physecs_amd import api
    sc = scenes.batched_worlds(8, n_worlds=60, lo=60, hi=140, ragdoll_frac=0.3)
    assert sc.n_dyn > 4096
    log(f"[small] {sc.n_dyn} bodies in 60 worlds against worlds alone")
    big = api.World(sc, substeps=4, iterations=2)
    arr = sc.arrays()
    picks = {w: api.World(sc.world_subscene(w), substeps=4, iterations=2) for w in (0, 7, 33, 59)}
    for k in range(40):
        big.step(1 / 60)
        for g in picks.values():
            g.step(1 / 60)
    pos = big.state()[0]
    for w, g in picks.items():
        assert np.array_equal(bits(pos[arr["world"] == w]), bits(g.state()[0])), w
        assert 0 < g.counts()["manifolds"] < 4096
        g.close()
    big.close()


@pytest.mark.parametrize("side", [1, 2, 10, 15, 17])
def test_piles_lockstep_bitexact(side):
    """1 to 4,913 bodies: one to four manifolds a thread, and beyond the limit."""
    log(f"[small] a pile of {side ** 3} bodies")
    g, _ = lockstep(scenes.mixed_lattice(5, side=side), 30 if side < 15 else 12, check_every=6)
    assert g.grid_fallbacks() == 0


@pytest.mark.parametrize("bodies,statics", [(64, 2100), (65, 2048), (65, 2049), (300, 4097), (3, 7000)])
def test_statics_packed_in_the_grid_or_apart(bodies, statics):
    """The grid's workgroup (256 threads for up to 256 bodies, 512 for up to 512) packs the
    non-dynamic colliders of up to 64 bodies, and up to eight a thread of more bodies; beyond,
    they have a launch of their own."""
    sc = scenes.Scene()
    side = int(np.ceil(statics ** 0.5))
    for i in range(statics):
        sc.add_static(scenes.BOX, [0.5, 0.3, 0.5], [i % side - side / 2, -0.3, i // side - side / 2])
    for i in range(bodies):
        sc.add_body((scenes.SPHERE, scenes.BOX)[i % 2], [[0.4], [0.3, 0.3, 0.3]][i % 2],
                    [0.9 * (i % 16) - 7, 0.35, 0.9 * (i // 16) - 9])
    g, _ = lockstep(sc, 4)
    assert g.counts()["pairs"] >= bodies


def test_a_full_cell_hands_the_step_to_the_tree_walk():
    """729 small bodies in one cell, made large by one large body: more than a cell may hold."""
    sc = scenes.Scene()
    for i in range(729):
        sc.add_body(scenes.SPHERE, [0.3], [0.7 * (i % 9), 0.7 * (i // 9 % 9), 0.7 * (i // 81)])
    sc.add_body(scenes.SPHERE, [4.0], [20, 3, 3])
    sc.add_static(scenes.BOX, [30, 0.5, 30], [0, -0.85, 0])
    g, _ = lockstep(sc, 6, check_every=3)
    assert g.grid_fallbacks() == 6
