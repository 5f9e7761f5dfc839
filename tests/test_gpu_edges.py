"""Sizes at the edges of the kernels' tiles and of the dispatch rules, against the host oracle (bit-exact)."""
import numpy as np
import pytest

from multigpuegtsmoothing_amd import datasets as D

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bucket", [1024, 1])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 2047, 2048, 2049, 4097])
def test_level_tables_at_tile_edges(egt_mod, oracle_mod, n, bucket):
    """The level tables are counted and ranked in tiles of 2048 positions; a coarse start level reads them all."""
    E, O = egt_mod, oracle_mod
    print("n", n, "bucket", bucket, flush=True)
    pts = D.mixture(n, seed=300 + n) if n > 16 else tuple(np.full(n, 0.25, np.float32) for _ in range(3))
    og = O.Grid(*pts, B=bucket)
    for level in (0, E.START_LEVEL_OCCUPANCY):
        g = E.GridStructure(pts, 1, 1e-6, bucket, 4)
        g.set_option(E.OPT_START_LEVEL, level)
        g.GRIDCUDAKNNSELF_COMPACT(8, 1e8)
        np.testing.assert_array_equal(g.GetKNNIndexes(), og.to_original(og.knn(8)[0]))
        g.close()


def test_batch_clouds_at_tile_edges(egt_mod, oracle_mod):
    """Clouds that begin at, before and after a 2048-position tile edge."""
    E, O = egt_mod, oracle_mod
    sizes = [2047, 1, 1, 2046, 2049, 64, 4096, 63]
    clouds = [D.sphere(n, seed=400 + i) for i, n in enumerate(sizes)]
    b = E.BatchGrid(clouds)
    b.set_option(E.OPT_START_LEVEL, E.START_LEVEL_OCCUPANCY)
    b.knn(12)
    for c, pts in enumerate(clouds):
        og = O.Grid(*pts)
        np.testing.assert_array_equal(b.GetKNNIndexes(c), og.to_original(og.knn(12)[0]), err_msg=f"cloud {c}")
    b.close()
