"""The contact solve with a lane per side of a manifold, at the edges of its passes: one
iteration (the substep's first pass is the last with a bias), none (the relaxation is the
first pass too), one substep (no velocity integration after the write-back), with hard,
bouncy and soft contacts and points without a friction mass, in lockstep with the oracle."""
import numpy as np
import pytest

from gpu_util import lockstep, log
from physecs_amd import scenes

pytestmark = pytest.mark.gpu


def _scene(seed, n):
    sc = scenes.random_cluster(seed, n=n, extent=1.0 + 0.01 * n)
    mat = sc.col_material
    kinds = np.random.default_rng(seed).integers(0, 4, len(mat))
    mat[kinds == 1] = np.array([0.4, 0.5, 0.0], np.float32)     # bouncy
    mat[kinds == 2] = np.array([0.6, 20.0, 0.7], np.float32)    # soft
    mat[kinds == 3] = np.array([0.0, 0.0, 0.0], np.float32)     # no friction
    sc._frozen = None
    return sc


@pytest.mark.parametrize("substeps,iterations", [(1, 0), (1, 1), (3, 1), (2, 3)])
@pytest.mark.parametrize("n,mode", [(1, "colors"), (33, "colors"), (90, "flow"), (90, "worlds"), (90, "xpass")])
def test_passes_lockstep_bitexact(substeps, iterations, n, mode):
    log(f"[sides] {n} bodies, {substeps} x {iterations}, {mode}")
    lockstep(_scene(3, n), 25, substeps=substeps, iterations=iterations, mode=mode)


@pytest.mark.parametrize("color_batch", [0, 1 << 30])
def test_colour_launches_and_runs_lockstep_bitexact(color_batch):
    """Colours of more manifolds than a run's workgroup has lane pairs (512), by launch and in a run."""
    sc = scenes.mixed_lattice(2, side=12)
    lockstep(sc, 40, check_every=10, tuning={"color_batch": color_batch})
