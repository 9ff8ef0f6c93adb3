"""GPU check of the stress at the predicted F (one thread per particle, then the force pass) against the
FP64 oracle: one substep of strained particles at the counts where its 64-lane waves and 256-particle
blocks end, for both spline orders and materials, in the interior and against three faces of the grid,
where stencil nodes are dropped.

Bars, as for the staged substeps of the other parity tests: relative L2 error 2e-5 for v and B,
|dF| <= 2e-5, |dx| <= 1e-5 cells.
"""
import numpy as np
import pytest

from anisotropicelastoplasticity_amd import Solver, _lib, scenes
from oracle.bind import Oracle

pytestmark = pytest.mark.gpu

COUNTS = {1: (1, 1, 1), 63: (7, 3, 3), 64: (4, 4, 4), 65: (13, 5, 1), 256: (4, 8, 8), 257: (257, 1, 1)}


@pytest.mark.parametrize("n", sorted(COUNTS))
@pytest.mark.parametrize("order", [2, 3])
@pytest.mark.parametrize("material", [_lib.SAND, _lib.SNOW])
@pytest.mark.parametrize("corner", [False, True])
def test_predicted_stress(n, order, material, corner):
    lo, hi = ((0.0, 0.0, 0.0), (0.2, 0.2, 0.2)) if corner else ((0.4, 0.3, 0.4), (0.6, 0.5, 0.55))
    sc = scenes.small_scene(material, order, 1, _lib.FRICTION_STICKY, seed=n, res=(16, 16, 16), cells=COUNTS[n], ppa=1,
                            lo=lo, hi=hi, prims=[], dt=1e-4)
    assert sc.n == n
    rng = np.random.default_rng(n)
    p = sc.particles
    p["v"] = p["v"] + rng.normal(size=(3, n)).astype(np.float32)
    p["B"] = (1e-3 * rng.normal(size=(9, n))).astype(np.float32)
    F = np.tile(np.eye(3).reshape(9, 1), (1, n)) + 5e-3 * rng.normal(size=(9, n)) - 3e-3 * np.eye(3).reshape(9, 1)
    p["F"] = F.astype(np.float32)
    with Solver(0) as s:
        sc.load_into(s)
        s.substep(sc.dt)
        q = s.get_particles()
        assert s.stats()["status"] == 0
    o = Oracle(sc.params, sc.gmin, sc.gmax, sc.res, prims=sc.prims)
    o.load_scene(sc)
    o.substep(sc.dt)
    r = o.get_particles()
    o.close()
    rel = {k: np.linalg.norm(q[k] - r[k]) / np.linalg.norm(r[k]) for k in ("v", "B")}
    dF, dx = np.max(np.abs(q["F"] - r["F"])), np.max(np.abs(q["x"] - r["x"])) * 16
    print(n, order, material, corner, rel, dF, dx, flush=True)
    assert rel["v"] <= 2e-5 and rel["B"] <= 2e-5 and dF <= 2e-5 and dx <= 1e-5
