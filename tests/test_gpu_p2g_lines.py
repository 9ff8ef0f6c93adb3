"""GPU check of the lines between P2G's rows and layers for untuned contexts: scenes on either side of each line, with
equal bits against the schedule not taken."""
import numpy as np
import pytest
import torch

from anisotropicelastoplasticity_amd import Solver, _lib, scenes

pytestmark = pytest.mark.gpu

# tiles along each axis, lattice cells of 8 particles: 512 tiles (two per CU) and 576
LINES = {"two per CU, 216 per tile": ((8, 8, 8), (24, 24, 24), _lib.P2G_ROWS),
         "two per CU, 343 per tile": ((8, 8, 8), (28, 28, 28), _lib.P2G_LAYERS),
         "more than two, 64 per tile": ((9, 8, 8), (18, 16, 16), _lib.P2G_LAYERS),
         "more than two, 720 per tile": ((9, 8, 8), (40, 36, 36), _lib.P2G_LAYERS),
         "more than two, 799 per tile": ((9, 8, 8), (42, 37, 37), _lib.P2G_ROWS)}


@pytest.mark.parametrize("line", sorted(LINES))
def test_line(line):
    tiles, cells, expect = LINES[line]
    n_cu = torch.cuda.get_device_properties(0).multi_processor_count
    if n_cu != 256:
        pytest.skip("the scenes are made for 256 CUs")
    lo, hi = (24.5 / 96,) * 3, tuple((24 + 4 * k - 0.5) / 96 for k in tiles)
    sc = scenes.small_scene(_lib.SAND, 2, 0, _lib.FRICTION_STICKY, seed=6, res=(96,) * 3, cells=cells, lo=lo, hi=hi, prims=[],
                            dt=1e-6)
    sc.particles["v"] = sc.particles["v"] + np.random.default_rng(6).normal(size=(3, sc.n)).astype(np.float32)
    outs = []
    for shape in (None, (8, 512, 4096, _lib.SORT_COUNTING, _lib.P2G_ROWS), (4, 768, 4096, _lib.SORT_COUNTING, _lib.P2G_LAYERS)):
        with Solver(0) as s:
            sc.load_into(s)
            if shape:
                s.set_tuning(*shape)
            s.run(sc.dt, 5)
            print(line, sc.n, s.stats()["n_active_tiles"], s.tuning()["p2g_pass"], flush=True)
            assert s.stats()["n_active_tiles"] == tiles[0] * tiles[1] * tiles[2]
            assert s.tuning()["p2g_pass"] == (shape[4] if shape else expect)
            outs.append(s.get_particles())
    for o in outs[1:]:
        for k in ("x", "v", "B", "F", "plastic"):
            assert np.array_equal(o[k].view(np.uint32), outs[0][k].view(np.uint32)), k
