"""Small clouds' Taubin passes in one launch, where workgroups wait for one another: several handles at once, and a wait
that runs out."""
import os
import subprocess
import threading
import time

import numpy as np
import pytest

from multigpuegtsmoothing_amd import datasets as D

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_launch_budget(tmp_path):
    exe = str(tmp_path / "budget_check")
    subprocess.run(["g++", "-std=c++17", "-pthread", "-I", os.path.join(ROOT, "multigpuegtsmoothing_amd", "csrc"),
                    os.path.join(ROOT, "tests", "native", "budget_check.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout.strip() == "0", r.stdout


@pytest.mark.gpu
def test_two_clouds_that_fill_the_gpu(egt_mod):
    """Two clouds whose tiles fill the GPU each, smoothed from two threads: results are those of each cloud alone, and
    the calls together take less than half the time of the waits that two launches holding each other's places out
    would run into (20 ms in each of 8 rounds; about 2 ms a call)."""
    E = egt_mod
    clouds = [D.torus(262_144, seed=710), D.sphere(262_144, seed=711)]
    rounds = 8

    def run(i, out, barrier):
        outs, tiles, spent = [], [], 0.0
        for _ in range(rounds):
            g = E.GridStructure(clouds[i], 1, 1e-6, 1024, 4)
            g.GRIDCUDAKNNSELF_COMPACT(8, 1e8)
            if barrier:
                barrier.wait()
            t0 = time.perf_counter()
            E.EGT_CUDA(g).PerformSmoothing(60, 0.5, -0.53, 0.65)
            spent += time.perf_counter() - t0
            tiles.append(g.stats()["taubin_tile"])
            outs.append(E.getOutputPoints(g))
            g.close()
        out[i] = outs, tiles, spent

    alone, together = {}, {}
    for i in range(2):
        run(i, alone, None)
        assert alone[i][1] == [256] * rounds
    barrier = threading.Barrier(2, timeout=30)
    threads = [threading.Thread(target=run, args=(i, together, barrier)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    print("tiles", together[0][1], together[1][1], "ms", together[0][2] * 1e3, together[1][2] * 1e3, flush=True)
    for i in range(2):
        assert set(together[i][1]) <= {256, 1024}
        for out in together[i][0]:
            for a, b in zip(alone[i][0][0], out):
                np.testing.assert_array_equal(a, b, err_msg=f"cloud {i}")
    assert min(together[0][2], together[1][2]) < rounds * 0.010


@pytest.mark.gpu
@pytest.mark.parametrize("regularized", [0, 1])
def test_wait_that_runs_out(egt_mod, oracle_mod, regularized):
    """A wait of no time at all: tiles give up, every workgroup leaves, and the call runs a launch per pass from
    untouched points. Later calls on the handle do so at once, until the option is set again."""
    E, O = egt_mod, oracle_mod
    pts, k = D.torus(60_001, seed=712), 16
    og = O.Grid(*pts)
    x, y, z = og.xs, og.ys, og.zs
    rows = og.knn(k)[0]
    g = E.GridStructure(pts, 1, 1e-6, 1024, 4)
    g.set_option(E.OPT_TAUBIN_REGULARIZED, regularized)
    g.GRIDCUDAKNNSELF_COMPACT(k, 1e8)
    tiles = []
    for wait in (0, None, 500):
        if wait is not None:
            g.set_option(E.OPT_TAUBIN_WAIT, wait)
        E.EGT_CUDA(g).PerformSmoothing(20, 0.5, -0.53, 0.65)
        tiles.append(g.stats()["taubin_tile"])
        rows = O.egg(x, y, z, rows, 0.65)
        x, y, z = O.taubin_f32(x, y, z, rows, 20, 0.5, -0.53, regularized=bool(regularized))
        for a, b in zip(E.getOutputPoints(g), og.output(x, y, z)):
            np.testing.assert_array_equal(a, b, err_msg=f"wait {wait}")
    assert tiles == [1024, 1024, 256]
    for bad in (-1, 1_000_001):
        with pytest.raises(E.EGTError):
            g.set_option(E.OPT_TAUBIN_WAIT, bad)
    g.close()


@pytest.mark.gpu
def test_wait_that_runs_out_for_some_tiles(egt_mod, oracle_mod):
    """Clouds of exactly one tile, which finish alone, of two tiles, which wait for one another for as many passes as
    they keep step, and a large one: tiles that are through, in mid-run and still waiting leave together, and no point
    of any cloud has moved before the passes run again."""
    E, O = egt_mod, oracle_mod
    sizes = [256] * 20 + [512] * 60 + [20_000] + [512] * 20 + [256] * 3
    clouds = [D.sphere(n, seed=750 + i) for i, n in enumerate(sizes)]
    b = E.BatchGrid(clouds)
    b.set_option(E.OPT_TAUBIN_WAIT, 0)
    b.knn(12)
    E.EGT_CUDA(b).PerformSmoothing(40, 0.5, -0.53, 0.65)
    assert b.stats()["taubin_tile"] == 1024
    out = [b.split(a) for a in E.getOutputPoints(b)]
    for c in (0, 19, 20, 21, 50, 79, 80, 81, 100, 103):
        ref = O.pipeline(*clouds[c], 12, 40, 0.5, -0.53, 0.65, normals=False)
        for ax in range(3):
            np.testing.assert_array_equal(out[ax][c], ref["output"][ax], err_msg=f"cloud {c}")
    b.close()
