"""GPU check of the P2G schedule a context takes by itself (mpm_run, from the active tiles): few tiles, many
tiles of ordinary filling and many crowded tiles, for each kernel mode, with ragged edges. Both schedules
keep every order of summation, so the bar is equal bits against each schedule set by hand.
"""
import numpy as np
import pytest

from anisotropicelastoplasticity_amd import Solver, _lib, scenes

pytestmark = pytest.mark.gpu

# resolution, lattice cells, particles per cell and axis, block extent in grid cells, schedule taken
FILLS = {"few tiles": ((24, 23, 25), (9, 8, 7), 2, 9.0, _lib.P2G_ROWS),
         "many tiles": ((61, 62, 63), (38, 37, 35), 2, 38.0, _lib.P2G_LAYERS),
         "crowded": ((61, 62, 63), (31, 30, 30), 3, 31.0, _lib.P2G_ROWS)}


@pytest.mark.parametrize("fill", sorted(FILLS))
@pytest.mark.parametrize("order,predicted", [(2, 0), (2, 1), (3, 0), (3, 1)])
def test_schedule_chosen(fill, order, predicted):
    res, cells, ppa, edge, expect = FILLS[fill]
    lo = tuple(0.2 for _ in range(3))
    hi = tuple(0.2 + edge * c / max(cells) / max(res) for c in cells)
    sc = scenes.small_scene(_lib.SAND, order, predicted, _lib.FRICTION_STICKY, seed=5, res=res, cells=cells, ppa=ppa,
                            lo=lo, hi=hi, prims=[], dt=1e-5)
    sc.particles["v"] = sc.particles["v"] + np.random.default_rng(5).normal(size=(3, sc.n)).astype(np.float32)
    outs = []
    for shape in (None, (8, 512, 4096, _lib.SORT_COUNTING, _lib.P2G_ROWS), (4, 768, 4096, _lib.SORT_COUNTING, _lib.P2G_LAYERS)):
        with Solver(0) as s:
            sc.load_into(s)
            if shape:
                s.set_tuning(*shape)
            s.run(sc.dt, 6)
            print(fill, order, predicted, sc.n, s.stats()["n_active_tiles"], s.tuning(), flush=True)
            assert s.tuning()["p2g_pass"] == (shape[4] if shape else expect)
            outs.append(s.get_particles())
    for o in outs[1:]:
        for k in ("x", "v", "B", "F", "plastic"):
            assert np.array_equal(o[k].view(np.uint32), outs[0][k].view(np.uint32)), k
