"""Search shapes and start levels that a caller names: each option value runs what it says, and the kernels that the
library does not choose on clouds of a test's size are compared with the oracle by naming them."""
import numpy as np
import pytest

from multigpuegtsmoothing_amd import datasets as D

pytestmark = pytest.mark.gpu


def _search(E, pts, k, **options):
    g = E.GridStructure(pts, 1, 1e-6, 1024, 4)
    for name, value in options.items():
        g.set_option(getattr(E, "OPT_" + name), value)
    g.GRIDCUDAKNNSELF_COMPACT(k, 1e8)
    rows, st = g.GetKNNIndexes(), g.stats()
    g.close()
    return rows, st


@pytest.mark.parametrize("shape", [0, 1, 2])
def test_named_start_level(egt_mod, oracle_mod, shape):
    """The own cell is reachable by name on a cloud of even density, where the library starts at the occupancy level,
    and no other option changes the start."""
    E, O = egt_mod, oracle_mod
    pts, k = D.sphere(20_000, seed=61), 24
    shapes = E.class_shapes_all(shape)
    own, s_own = _search(E, pts, k, KNN_CLASS_SHAPES=shapes, START_LEVEL=E.START_LEVEL_OWN_CELL)
    occ, s_occ = _search(E, pts, k, KNN_CLASS_SHAPES=shapes, START_LEVEL=E.START_LEVEL_OCCUPANCY)
    dflt, s_dflt = _search(E, pts, k, KNN_CLASS_SHAPES=shapes)
    cap, s_cap = _search(E, pts, k, KNN_CLASS_SHAPES=shapes, KNN_LONG_QUERY=0)
    print("cells a query: own", s_own["knn_cells"] / 20_000, "occupancy", s_occ["knn_cells"] / 20_000, flush=True)
    assert s_own["knn_cells"] > 2 * s_occ["knn_cells"]
    for st in (s_dflt, s_cap):
        assert (st["knn_cells"], st["knn_candidates"]) == (s_occ["knn_cells"], s_occ["knn_candidates"])
    og = O.Grid(*pts)
    want = og.to_original(og.knn(k)[0])
    for rows in (own, occ, dflt, cap):
        np.testing.assert_array_equal(rows, want)


@pytest.mark.parametrize("k", [8, 40, 64])
def test_named_lane_shape(egt_mod, oracle_mod, k):
    """A lane per query is reachable by name at every size: only that shape hands long queries on."""
    E, O = egt_mod, oracle_mod
    pts = D.sphere(5_000, seed=62)
    og = O.Grid(*pts)
    want = og.to_original(og.knn(k)[0])
    for shape in (0, 1, 2):
        rows, st = _search(E, pts, k, KNN_LONG_QUERY=1, KNN_CLASS_SHAPES=E.class_shapes_all(shape))
        assert (st["knn_long_queries"] > 0) == (shape != 2), shape
        np.testing.assert_array_equal(rows, want, err_msg=f"shape {shape}")
    # setting the cap asks for the lane shape, whatever its value
    rows, st = _search(E, pts, k, KNN_LONG_QUERY=2)
    assert st["knn_long_queries"] > 0
    np.testing.assert_array_equal(rows, want)


def test_tuned_start_level_replayed(egt_mod):
    """A level that the tuner chose, set on another handle, does the work of the handle it was tuned on."""
    E = egt_mod
    for pts, k in ((D.sphere(3_000, seed=63), 8), (D.mixture(30_000, seed=64), 8), (D.torus(40_000, seed=65), 40)):
        g = E.GridStructure(pts, 1, 1e-6, 1024, 4)
        level = g.autotune(k)[0]
        g.GRIDCUDAKNNSELF_COMPACT(k, 1e8)
        tuned = g.stats()
        g.close()
        print("level", level, flush=True)
        _, st = _search(E, pts, k, START_LEVEL=level if level else E.START_LEVEL_OWN_CELL)
        assert st["knn_cells"] == tuned["knn_cells"] and st["knn_candidates"] == tuned["knn_candidates"]
