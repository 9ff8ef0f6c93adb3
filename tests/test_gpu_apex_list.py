"""GPU check of the FP64 apex pass beside the surrogate (from the position lists) against the same pass without it (from
G2P's masks), at the counts where waves, blocks and groups of 64 waves end: with a network whose outputs are NaN every
candidate takes the exact projection, so the two runs give equal bits and as many FP64 projections."""
import numpy as np
import pytest

from anisotropicelastoplasticity_amd import Solver, _lib, scenes
from oracle import mlp_oracle as mo

pytestmark = pytest.mark.gpu

COUNTS = {1: (1, 1, 1), 64: (4, 4, 4), 65: (13, 5, 1), 256: (4, 8, 8), 257: (257, 1, 1), 4096: (16, 16, 16), 4097: (17, 241, 1),
          16400: (25, 16, 41)}


def _scene(n, seed, predicted):
    sc = scenes.small_scene(_lib.SAND, 2, predicted, _lib.FRICTION_COULOMB, seed=seed, res=(32, 32, 32), cells=COUNTS[n], ppa=1,
                            dt=1e-5)
    sc.params.fp64_apex_radius = 1.5e-3  # of the order of the strains: some particles on either side
    rng = np.random.default_rng(seed)
    F = np.tile(np.eye(3).reshape(9, 1), (1, n)) * (1 - rng.uniform(1e-4, 1e-3, n)) + 6e-4 * rng.normal(size=(9, n))
    sc.particles["F"] = F.astype(np.float32)
    return sc


@pytest.mark.parametrize("predicted", [0, 1])
@pytest.mark.parametrize("counts", [(1,), (64,), (65,), (256,), (257,), (4096,), (4097,), (16400,), (257, 1, 4097, 64)])
def test_apex_beside_surrogate(counts, predicted):
    batch = [_scene(n, k, predicted) for k, n in enumerate(counts)]
    w = np.zeros(mo.NPARAM, np.float32)
    w[mo.active_mask()] = np.nan
    outs = []
    for sur in (False, True):
        with Solver(0) as s:
            s.load_batch(batch)
            if sur:
                s.surrogate_set_weights(w)
                s.set_surrogate(True, 1e-5)
            s.run(batch[0].dt, 3)
            outs.append((s.get_particles(), s.stats()))
    (a, sa), (b, sb) = outs
    print(counts, predicted, "apex", sa["fp64_apex_count"], sb["fp64_apex_count"], "candidates", sb["surrogate_candidates"], flush=True)
    if sum(counts) > 64:
        assert sa["fp64_apex_count"] > 0 and sb["surrogate_candidates"] > 0
    assert sa["fp64_apex_count"] == sb["fp64_apex_count"]
    for k in ("x", "v", "B", "F", "plastic"):
        assert np.array_equal(a[k].view(np.uint32), b[k].view(np.uint32)), k
