"""Handles used from several threads at once: what one does never disturbs another's call."""
import threading

import numpy as np
import pytest

from multigpuegtsmoothing_amd import datasets as D

pytestmark = pytest.mark.gpu


def test_graph_replays_beside_growing_handles(egt_mod):
    """Two threads run the passes as graphs, two others search ever larger clouds on new handles, whose buffers grow (the
    device is synchronized before a buffer is given up). Every call succeeds, with the results of a run alone."""
    E = egt_mod
    clouds = [D.torus(40_000 + 9_001 * i, seed=720 + i) for i in range(2)]
    errors = []

    def smooth(i, rounds):
        outs = []
        for _ in range(rounds):
            g = E.GridStructure(clouds[i], 1, 1e-6, 1024, 4)
            g.set_option(E.OPT_TAUBIN_TILE, 1024)
            g.GRIDCUDAKNNSELF_COMPACT(16, 1e8)
            E.EGT_CUDA(g).PerformSmoothing(60, 0.5, -0.53, 0.65)
            assert g.stats()["taubin_tile"] == 1024
            outs.append(E.getOutputPoints(g))
            g.close()
        return outs

    alone = [smooth(i, 1)[0] for i in range(2)]
    together, stop = {}, threading.Event()

    def worker(i):
        try:
            together[i] = smooth(i, 25)
        except Exception as e:  # shown by the assertion below
            errors.append(e)

    def grower(i):
        try:
            n = 1_000
            while not stop.is_set():
                g = E.GridStructure(D.sphere(5_000, seed=730 + i), 1, 1e-6, 1024, 4)
                for k in (4, 16, 64):  # one handle's rows grow
                    g.GRIDCUDAKNNSELF_COMPACT(k, 1e8)
                    g.GRIDCUDAKNNCompact(D.sphere(n * k // 4, seed=740 + i), 4, 1e8)
                g.close()
                n = n % 16_000 + 1_000
        except Exception as e:
            errors.append(e)

    workers = [threading.Thread(target=worker, args=(i,)) for i in range(2)]
    growers = [threading.Thread(target=grower, args=(i,)) for i in range(2)]
    for t in workers + growers:
        t.start()
    for t in workers:
        t.join()
    stop.set()
    for t in growers:
        t.join()
    assert not errors, errors
    for i in range(2):
        for out in together[i]:
            for a, b in zip(alone[i], out):
                np.testing.assert_array_equal(a, b, err_msg=f"cloud {i}")
