"""GPU check of the P2G shape that an untuned context takes as its particles spread: a block flies apart from a few
tiles (16-wave rows) to more than the CUs (layers). The shape follows between two runs, and within mpm_solve; results
do not depend on it (the bar is equal bits against a fixed shape), and no run waits for the tile count.
"""
import time

import numpy as np
import pytest
import torch

from anisotropicelastoplasticity_amd import Solver, _lib, scenes

pytestmark = pytest.mark.gpu

KEYS = ("x", "v", "B", "F", "plastic")
FIXED = (8, 512, 4096, _lib.SORT_COUNTING, _lib.P2G_ROWS)


def _flying_apart(res=96):
    # 16 cells wide, velocities 72/s times the distance from the middle: 2.2 times as wide after 1/60 s
    lo, hi = (0.5 - 8.0 / 96,) * 3, (0.5 + 8.0 / 96,) * 3
    sc = scenes.small_scene(_lib.SNOW, 2, 0, _lib.FRICTION_STICKY, seed=4, res=(res,) * 3, cells=(16, 16, 16), lo=lo, hi=hi,
                            prims=[], dt=1e-4, E=1e3)
    sc.particles["v"] = (72.0 * (sc.particles["x"] - 0.5)).astype(np.float32)
    return sc


def _same(a, b, what):
    for k in KEYS:
        assert np.array_equal(a[k].view(np.uint32), b[k].view(np.uint32)), (what, k)


def _wide(t):
    return (t["p2g_pass"], t["p2g_ranks"], t["p2g_blocks"]) == (
        _lib.P2G_ROWS, 8, torch.cuda.get_device_properties(0).multi_processor_count)


def _advance(s, dt, how, n):
    if how == "run":
        s.run(dt, n)
    else:
        for _ in range(n):
            if how == "substep":
                s.substep(dt)
            else:
                for stage in (_lib.STAGE_SORT, _lib.STAGE_P2G, _lib.STAGE_GRID, _lib.STAGE_G2P):
                    s.stage(stage, dt)


@pytest.mark.parametrize("how", ["run", "substep", "stage"])
def test_shape_follows_runs(how):
    sc = _flying_apart()
    outs = []
    for fixed in (False, True):
        with Solver(0) as s:
            sc.load_into(s)
            if fixed:
                s.set_tuning(*FIXED)
            first = s.tuning()
            # the count that a call finds is that of an earlier one, up to some hundred substeps old
            for n in (200, 200, 200, 1):
                _advance(s, 0.4 * sc.dt, how, n)
                s.synchronize()
            print(how, fixed, first, s.tuning(), s.stats()["n_active_tiles"], flush=True)
            if not fixed:
                assert _wide(first)
                assert s.tuning()["p2g_pass"] == _lib.P2G_LAYERS
            assert s.stats()["status"] == 0
            outs.append(s.get_particles())
    _same(outs[0], outs[1], how)


def test_shape_follows_solve():
    sc = _flying_apart()
    outs = []
    for fixed in (False, True):
        with Solver(0) as s:
            sc.load_into(s)
            if fixed:
                s.set_tuning(*FIXED)
            first = s.tuning()
            s.solve(0.05, 0.0)
            print(fixed, first, s.tuning(), s.stats()["n_active_tiles"], s.clock(), flush=True)
            if not fixed:
                assert _wide(first)
                assert s.tuning()["p2g_pass"] == _lib.P2G_LAYERS
            assert s.clock()["frames"] == 1
            outs.append((s.get_particles(), s.clock()))
    assert outs[0][1] == outs[1][1]
    _same(outs[0][0], outs[1][0], "solve")


def test_new_grid():
    # particles kept, the grid replaced: the shape, and the state after some substeps, are those of a fresh context
    sc, fine = _flying_apart(), _flying_apart(res=192)
    outs = []
    for regrid in (False, True):
        with Solver(0) as s:
            (sc if regrid else fine).load_into(s)
            if regrid:
                s.set_grid(fine.gmin, fine.gmax, fine.res)
            shape = s.tuning()
            s.run(2e-5, 5)
            outs.append((shape, s.stats()["n_active_tiles"], s.get_particles()))
    print(outs[0][:2], outs[1][:2], flush=True)
    assert outs[0][:2] == outs[1][:2] and not _wide(outs[0][0])
    _same(outs[0][2], outs[1][2], "grid")


def test_run_does_not_wait():
    # a captured shape for a new dt must not wait for the substeps queued before it
    sc = scenes.small_scene(_lib.SNOW, 2, 0, _lib.FRICTION_STICKY, seed=4, res=(128,) * 3, cells=(64, 64, 32), lo=(0.25, 0.25, 0.3),
                            hi=(0.75, 0.75, 0.55), prims=[], dt=1e-5)
    with Solver(0) as s:
        sc.load_into(s)
        s.run(sc.dt, 4)
        s.synchronize()
        s.run(sc.dt, 300)
        t0 = time.perf_counter()
        s.run(0.5 * sc.dt, 4)
        t1 = time.perf_counter()
        s.synchronize()
        t2 = time.perf_counter()
    print("call %.1f ms, then wait %.1f ms" % (1e3 * (t1 - t0), 1e3 * (t2 - t1)), flush=True)
    assert t1 - t0 < 0.5 * (t2 - t0)
