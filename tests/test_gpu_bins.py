"""GPU checks of the sort's bins, which each substep's G2P counts for the next one (a cloth's elements by the kernel
that moves them). Whatever comes between two substeps - another sort, the other sort mode, new particles, a
frame's end - the sorted order stays the stable order of the keys, and the state's bits do not change.
The keys themselves are compared with floor((x - min) / h) in double at the cells' boundaries and beside them.
"""
import ctypes

import numpy as np
import pytest

from anisotropicelastoplasticity_amd import Solver, _lib, scenes

pytestmark = pytest.mark.gpu

KEYS = ("x", "v", "B", "F", "plastic")


def _scene(kind):
    if kind == "cloth":
        return scenes.config3_cloth_sand(n_side=17, edge=1.0 / 60.0, sand_cells=(7, 5, 6))
    return scenes.small_scene(_lib.SAND, 2, 0, _lib.FRICTION_STICKY, seed=9, res=(29, 31, 27), cells=(9, 8, 7), dt=1e-4)


def _load(sc, s):
    sc, mesh = sc if isinstance(sc, tuple) else (sc, None)
    sc.load_into(s)
    if mesh:
        s.set_mesh(mesh["x"], mesh["faces"], **{k: v for k, v in mesh.items() if k not in ("x", "faces")})
    return sc


def _between(s, what, sc):
    if what == "autotune":
        s.autotune(sc.dt, reps=1)
    elif what == "radix":
        t = s.tuning()
        s.set_tuning(t["p2g_ranks"], t["p2g_blocks"], t["grid_blocks"], _lib.SORT_RADIX, t["p2g_pass"])
    elif what == "eager":
        s.time_substeps(sc.dt, 2)
        s.substep(sc.dt)


@pytest.mark.parametrize("kind", ["sand", "cloth"])
@pytest.mark.parametrize("what", ["autotune", "radix", "eager"])
def test_substeps_after(kind, what):
    scene = _scene(kind)
    outs = []
    for interrupted in (False, True):
        with Solver(0) as s:
            sc = _load(scene, s)
            s.run(sc.dt, 5)
            if interrupted:
                _between(s, what, sc)
            elif what == "eager":
                s.run(sc.dt, 3)
            s.run(sc.dt, 6)
            if kind == "sand":
                keys, ids, bins = s.get_sorted()
                assert np.array_equal(np.diff(bins), np.bincount(keys, minlength=len(bins) - 1))
                order = np.lexsort((ids, keys))
                assert np.array_equal(order, np.arange(s.n)) and np.array_equal(np.sort(ids), np.arange(s.n))
            outs.append((s.get_particles(), s.stats()["n_active_tiles"], s.stats()["n_active_blocks"]))
    print(kind, what, outs[0][1:], outs[1][1:], flush=True)
    assert outs[0][1:] == outs[1][1:]
    for k in KEYS:
        assert np.array_equal(outs[0][0][k].view(np.uint32), outs[1][0][k].view(np.uint32)), k


@pytest.mark.parametrize("steps", [1, 4, 7])
def test_new_particles(steps):
    # counts that no sort has used are dropped with the particles they belong to
    sc, other = _scene("sand"), _scene("sand")
    other.particles["x"] = (other.particles["x"] + 0.1).astype(np.float32)
    outs = []
    for first in (None, other):
        with Solver(0) as s:
            (first or sc).load_into(s)
            if first:
                s.run(sc.dt, steps)
                p = sc.particles
                s.set_particles(p["x"], p["mass"], v=p.get("v"), B=p.get("B"), F=p.get("F"), plastic=p.get("plastic"),
                                volume=p.get("volume"), phi=p.get("phi"))
            s.run(sc.dt, 5)
            outs.append(s.get_particles())
    for k in KEYS:
        assert np.array_equal(outs[0][k].view(np.uint32), outs[1][k].view(np.uint32)), k


@pytest.mark.parametrize("lo,size", [(0.0, 1.0), (0.37, 1.0), (-5.3, 7.7), (1000.1, 1.0), (-64.0, 128.0)])
def test_keys_at_cell_boundaries(lo, size):
    res = (37, 41, 23)
    mn, mx = [lo, lo + 0.11, lo - 0.23], [lo + size, lo + 0.11 + size, lo - 0.23 + size]
    axes, rng = [], np.random.default_rng(3)
    for d in range(3):
        h = (mx[d] - mn[d]) / res[d]
        c = np.float32(mn[d] + h * np.arange(1, res[d]))
        near = [c]
        for _ in range(3):
            near.append(np.nextafter(near[-1], np.float32(np.inf)))
        near.append(np.nextafter(c, np.float32(-np.inf)))
        near.append(np.nextafter(near[-1], np.float32(-np.inf)))
        near.append(np.float32(mn[d] + h * rng.uniform(0.01, res[d] - 0.01, 500)))
        axes.append(np.concatenate(near))
    n = max(map(len, axes))
    x = np.stack([rng.permutation(np.resize(a, n)) for a in axes]).astype(np.float32)
    want = np.zeros(n, np.int64)
    for d, mult in ((0, 1), (1, res[0]), (2, res[0] * res[1])):
        h = (mx[d] - mn[d]) / res[d]
        want += np.floor((x[d].astype(np.float64) - mn[d]) / h).astype(np.int64) * mult
    with Solver(0) as s:
        s.set_grid(mn, mx, res)
        s.set_params(scenes.sand_params())
        s.set_particles(x, np.ones(n, np.float32))
        s.stage(_lib.STAGE_SORT, 1e-4)
        keys, ids, _ = s.get_sorted()
    got = np.empty(n, np.int64)
    got[ids] = keys
    print(lo, size, n, int((got != want).sum()), flush=True)
    assert np.array_equal(got, want)


@pytest.mark.parametrize("kind", ["sand", "predicted", "cloth"])
def test_read_between_stages(kind):
    # the readback uses the buffer that the next G2P writes: reading between stages changes nothing, and returns
    # the particles as the last G2P left them, all planes or some
    scene = _scene("cloth") if kind == "cloth" else _scene("sand")
    if kind == "predicted":
        scene.params.stress_at_predicted_F = 1
    outs = []
    for read in (False, True):
        with Solver(0) as s:
            sc = _load(scene, s)
            for _ in range(3):
                before = s.get_particles()
                for stage in (_lib.STAGE_SORT, _lib.STAGE_P2G, _lib.STAGE_GRID, _lib.STAGE_G2P):
                    if read:
                        p = s.get_particles()
                        for k in KEYS:
                            assert np.array_equal(p[k].view(np.uint32), before[k].view(np.uint32)), (k, stage)
                    s.stage(stage, sc.dt)
            outs.append(s.get_particles())
            some = np.empty((9, sc.n), np.float32)
            assert s.lib.mpm_get_particles(s.h, None, None, some.ctypes.data_as(ctypes.POINTER(ctypes.c_float)), None, None, None) == 0
            assert np.array_equal(some.view(np.uint32), outs[-1]["B"].view(np.uint32))
    for k in KEYS:
        assert np.array_equal(outs[0][k].view(np.uint32), outs[1][k].view(np.uint32)), k


@pytest.mark.parametrize("res", [(16, 16, 16), (17, 16, 16), (15, 16, 17), (64, 64, 64), (64, 64, 65), (63, 65, 64)])
@pytest.mark.parametrize("spread", ["everywhere", "ends"])
def test_scan_of_sparse_grids(res, spread):
    # scan blocks of 4096 cells: one, a last one of few cells, 64 (the most that one launch scans) and 65; particles
    # in every block or only in the first and last cells
    rng = np.random.default_rng(sum(res))
    n, cells = 5000, int(np.prod(res))
    key = rng.integers(0, cells, n) if spread == "everywhere" else np.where(rng.random(n) < 0.5, rng.integers(0, 40, n),
                                                                            cells - 1 - rng.integers(0, 40, n))
    c = np.stack([key % res[0], key // res[0] % res[1], key // (res[0] * res[1])])
    x = ((c + rng.uniform(0.1, 0.9, (3, n))) / np.array(res)[:, None]).astype(np.float32)
    with Solver(0) as s:
        s.set_grid((0, 0, 0), (1, 1, 1), res)
        s.set_params(scenes.sand_params())
        s.set_particles(x, np.ones(n, np.float32))
        for _ in range(2):
            s.stage(_lib.STAGE_SORT, 0.0)
            keys, ids, bins = s.get_sorted()
            order = np.lexsort((np.arange(n), key))
            assert np.array_equal(ids, order) and np.array_equal(keys, key[order])
            assert np.array_equal(bins, np.concatenate([[0], np.cumsum(np.bincount(key, minlength=cells))]))
            tiles = np.unique((c[2] // 4 * 100 + c[1] // 4) * 100 + c[0] // 4)
            assert s.stats()["n_active_tiles"] == len(tiles)
            for st in (_lib.STAGE_P2G, _lib.STAGE_GRID, _lib.STAGE_G2P):
                s.stage(st, 0.0)
            p = s.get_particles()
            assert np.array_equal(p["x"], x)


@pytest.mark.parametrize("steps", [(1, 5), (4, 3), (7, 8)])
def test_cloth_forces_formed_anew(steps):
    # a substep leaves the element forces of the next one; after a change of the parameters (here: the same
    # again) they are formed by a kernel of their own, with the same bits
    scene = _scene("cloth")
    outs = []
    for again in (False, True):
        with Solver(0) as s:
            sc = _load(scene, s)
            s.run(sc.dt, steps[0])
            if again:
                s.set_params(sc.params)
            s.run(sc.dt, steps[1])
            outs.append((s.get_mesh(), s.get_particles(), s.stats()["fp64_svd_count"]))
    assert outs[0][2] == outs[1][2]
    for a, b in zip(outs[0][:2], outs[1][:2]):
        for k in a:
            assert np.array_equal(a[k].view(np.uint32), b[k].view(np.uint32)), k
