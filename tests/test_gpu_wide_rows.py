"""GPU check of P2G's rows by 16 waves: the kernel of every launch shape with 8 ranks, the row pass and no more
workgroups than CUs. Several scenes with ragged grids in one context, so that a workgroup's next tile may be
another scene's, with one workgroup, fewer workgroups than tiles and one per CU, for each kernel mode. It keeps
every order of summation, so the bar is equal bits against the other row kernel and the layers.
"""
import numpy as np
import pytest
import torch

from anisotropicelastoplasticity_amd import Solver, _lib, scenes

pytestmark = pytest.mark.gpu

KEYS = ("x", "v", "B", "F", "plastic")


def _batch(order, predicted):
    out = []
    for k, (res, cells, ppa) in enumerate((((24, 23, 25), (9, 8, 7), 2), ((31, 17, 29), (5, 4, 6), 3),
                                           ((19, 26, 22), (1, 1, 1), 1))):
        sc = scenes.small_scene(_lib.SAND if k % 2 else _lib.SNOW, order, predicted, _lib.FRICTION_STICKY, seed=k, res=res,
                                cells=cells, ppa=ppa, lo=(0.2,) * 3, hi=(0.55, 0.5, 0.45), prims=[], dt=1e-5)
        rng = np.random.default_rng(k)
        sc.particles["v"] = sc.particles["v"] + rng.normal(size=(3, sc.n)).astype(np.float32)
        sc.particles["F"] = (np.tile(np.eye(3).reshape(9, 1), (1, sc.n)) +
                             5e-3 * rng.normal(size=(9, sc.n))).astype(np.float32)
        out.append(sc)
    return out


def _same(a, b, what):
    for k in KEYS:
        assert np.array_equal(a[k].view(np.uint32), b[k].view(np.uint32)), (what, k)


@pytest.mark.parametrize("order,predicted", [(2, 0), (2, 1), (3, 0), (3, 1)])
def test_wide_rows_bits(order, predicted):
    n_cu = torch.cuda.get_device_properties(0).multi_processor_count
    batch = _batch(order, predicted)
    outs = []
    for shape in ((8, n_cu + 1, 4096, _lib.SORT_COUNTING, _lib.P2G_ROWS), (8, n_cu, 4096, _lib.SORT_COUNTING, _lib.P2G_ROWS),
                  (8, 7, 4096, _lib.SORT_COUNTING, _lib.P2G_ROWS), (8, 1, 4096, _lib.SORT_RADIX, _lib.P2G_ROWS),
                  (4, 3 * n_cu, 4096, _lib.SORT_COUNTING, _lib.P2G_LAYERS)):
        with Solver(0) as s:
            s.load_batch(batch)
            s.set_tuning(*shape)
            s.run(batch[0].dt, 6)
            print(order, predicted, shape, s.stats()["n_active_tiles"], flush=True)
            assert s.stats()["n_active_tiles"] > 7
            outs.append(s.get_particles())
    for o in outs[1:]:
        _same(o, outs[0], (order, predicted))


def test_chosen_shape_can_be_set():
    """An untuned context with few tiles takes the 16-wave rows; setting what it reports keeps them."""
    n_cu = torch.cuda.get_device_properties(0).multi_processor_count
    batch = _batch(2, 0)
    outs, shapes = [], []
    for given in (None, 0):
        with Solver(0) as s:
            s.load_batch(batch)
            if given is not None:
                t = shapes[given]
                s.set_tuning(t["p2g_ranks"], t["p2g_blocks"], t["grid_blocks"], t["sort_mode"], t["p2g_pass"])
            s.run(batch[0].dt, 6)
            shapes.append(s.tuning())
            outs.append(s.get_particles())
    print(shapes, flush=True)
    assert shapes[0]["p2g_pass"] == _lib.P2G_ROWS and shapes[0]["p2g_ranks"] == 8 and shapes[0]["p2g_blocks"] == n_cu
    assert shapes[1] == shapes[0]
    _same(outs[1], outs[0], "set again")
