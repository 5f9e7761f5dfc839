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


class _Named:
    """The package with every point-cloud handle made under the given options (a test of another file then runs in the
    shape that these name; a start level 0 in it means the own cell)."""

    def __init__(self, E, **options):
        def named(base):
            class Grid(base):
                def __init__(self, *args, **kwargs):
                    super().__init__(*args, **kwargs)
                    for name, value in options.items():
                        super().set_option(getattr(E, "OPT_" + name), value)

                def set_option(self, opt, value):
                    own = opt == E.OPT_START_LEVEL and value == 0
                    super().set_option(opt, E.START_LEVEL_OWN_CELL if own else value)

            return Grid

        self._E, self.GridStructure, self.BatchGrid = E, named(E.GridStructure), named(E.BatchGrid)

    def __getattr__(self, name):
        return getattr(self._E, name)


@pytest.mark.parametrize("k", [8, 16, 24])
@pytest.mark.parametrize("lanes", [0, 1, 64])
def test_query_shapes_at_300001(egt_mod, oracle_mod, k, lanes):
    """More queries than the library gives to a wave each at these k: its own choice is then a lane per query. A tenth of
    the queries outside the grid and a finite radius."""
    E, O = egt_mod, oracle_mod
    ref = D.sphere(20_000, seed=41)
    q = tuple(a.copy() for a in D.sphere(300_001, seed=42))
    q[0][::10] *= np.float32(1.3)
    print("k", k, "lanes", lanes, flush=True)
    g = E.GridStructure(ref, 1, 1e-6, 1024, 4)
    g.set_option(E.OPT_KNN_QUERY_LANES, lanes)
    g.GRIDCUDAKNNCompact(q, k, 0.05)
    got, st = g.GetKNNIndexesQuery(), g.stats()
    g.close()
    og = O.Grid(*ref)
    rows, _, inv, _ = og.knn_query(*q, k, thres=0.05)
    np.testing.assert_array_equal(got, og.ref_to_original(rows))
    assert st["query_invalid_rows"] == int(inv.sum())


@pytest.mark.parametrize("case", ["sphere_k16", "torus_k40", "sphere_k64", "mixture_k8", "torus_k1", "sphere_k33",
                                  "outside", "short", "device", "crowded0", "crowded-2"])
def test_lane_query_search(egt_mod, oracle_mod, case):
    """The query tests with a lane per query (so few queries go to a wave each by default)."""
    import test_gpu_query as Q

    E = _Named(egt_mod, KNN_QUERY_LANES=1)
    if case == "outside":
        Q.test_queries_outside_the_grid(E, oracle_mod)
    elif case == "short":
        Q.test_short_rows_duplicates_and_big_cells(E, oracle_mod)
    elif case == "device":
        Q.test_device_input_and_self_rows_untouched(E, oracle_mod)
    elif case.startswith("crowded"):
        Q.test_queries_crowded_cells(E, oracle_mod, int(case[7:]))
    else:
        Q.test_query_rows_bit_exact(E, oracle_mod, case)


def test_query_lanes_option(egt_mod):
    """The allocation-free search follows the named shape as well; other values are refused."""
    import torch
    from test_zz_no_alloc import _allocating, _noalloc

    E = egt_mod
    g = E.GridStructure(D.torus(60_000, seed=66), 1, 1e-6, 1024, 4)
    for nq, k in ((5_000, 40), (150_000, 8)):
        q = tuple(torch.from_numpy(a).cuda() for a in D.torus(nq, seed=67))
        want = _allocating(E, g, q, k)
        for lanes in (1, 64, 0):
            g.set_option(E.OPT_KNN_QUERY_LANES, lanes)
            np.testing.assert_array_equal(_noalloc(E, torch, g, q, k), want, err_msg=f"{nq} lanes {lanes}")
    for bad in (-1, 2, 65):
        with pytest.raises(E.EGTError):
            g.set_option(E.OPT_KNN_QUERY_LANES, bad)
    g.close()


LANE_TESTS = ([("test_knn_rows_bit_exact", (c, 1)) for c in ("sphere20k_k40", "torus30k_k16", "sphere5k_k64", "lattice_k18",
                                                             "dups_k8")]
              + [("test_lattice_rows_follow_bucket_count", (k,)) for k in (10, 18)]
              + [("test_knn_independent_of_start_level", (v, 1)) for v in ("occupancy", -3, -2, -1, 0, 2, 5, 9)]
              + [("test_knn_invalidation_rules", (1,)), ("test_duplicate_points_rows_bit_exact", (1,))]
              + [("test_knn_crowded_cells_sub_levels", (v, m, 1)) for v in (0, -1, -3) for m in (None, 3750)]
              + [("test_every_k_class_bit_exact", (k,)) for k in (1, 7, 9, 23, 31, 33, 47, 55, 63)])


@pytest.mark.parametrize("start", ["own", "default"])
@pytest.mark.parametrize("name,args", LANE_TESTS, ids=[f"{n[5:]}-{a}" for n, a in LANE_TESTS])
def test_lane_search(egt_mod, oracle_mod, name, args, start):
    """The self search tests with a lane per query (clouds of their sizes go to a wave per query by default), from the
    own cell, as the reference starts, and from the default level."""
    import test_gpu_parity as P

    options = {"START_LEVEL": egt_mod.START_LEVEL_OWN_CELL} if start == "own" else {}
    E = _Named(egt_mod, KNN_CLASS_SHAPES=egt_mod.class_shapes_all(0), **options)
    getattr(P, name)(E, oracle_mod, *args)


@pytest.mark.parametrize("start", ["own", "default"])
def test_lane_batch(egt_mod, oracle_mod, start):
    import test_gpu_batch as B

    options = {"START_LEVEL": egt_mod.START_LEVEL_OWN_CELL} if start == "own" else {}
    E = _Named(egt_mod, KNN_CLASS_SHAPES=egt_mod.class_shapes_all(0), **options)
    B.test_batch_matches_separate_oracle_runs(E, oracle_mod, 0, 1, None)


@pytest.mark.parametrize("n", [1, 64, 2048, 2049, 4097])
def test_own_cell_at_tile_edges(egt_mod, oracle_mod, n):
    import test_gpu_edges as T

    T.test_level_tables_at_tile_edges(_Named(egt_mod), oracle_mod, n, 1024)


@pytest.mark.parametrize("n,k,shape", [(99_968, 8, 2), (99_969, 8, 0), (120_000, 16, 2), (120_001, 16, 0),
                                       (299_968, 24, 2), (299_969, 24, 0), (99_968, 32, 2), (99_969, 32, 2),
                                       (299_968, 40, 2), (299_969, 40, 2), (99_969, 64, 2), (299_968, 64, 2)])
def test_both_sides_of_the_shape_limits(egt_mod, oracle_mod, n, k, shape):
    """The rule counts whole chunks of 64 queries. The largest size of the wave shape and the smallest of the lane shape
    at short lists, and of 1, 2 and 4 queries a wave at long ones: the search does the work of the named shape, and
    rows are the oracle's."""
    E, O = egt_mod, oracle_mod
    print("n", n, "k", k, flush=True)
    pts = D.torus(n, seed=31)
    rows, st = _search(E, pts, k)
    work = {}
    for s in (0, 2):
        named = _search(E, pts, k, KNN_CLASS_SHAPES=E.class_shapes_all(s))[1]
        work[s] = named["knn_cells"], named["knn_candidates"]
    print("cells, candidates: lane", work[0], "wave", work[2], flush=True)
    assert (st["knn_cells"], st["knn_candidates"]) == work[shape] != work[2 - shape]
    og = O.Grid(*pts)
    np.testing.assert_array_equal(rows, og.to_original(og.knn(k)[0]))


def test_taubin_graph_replays_match_launches(egt_mod):
    """The captured Taubin graphs against eager launches, by name (at this size the passes otherwise run in one launch):
    three smoothing calls of 60 iterations on one handle, two replays of the 25-iteration graph and one of the
    10-iteration graph each, with an eager search between the calls."""
    import test_gpu_parity as P

    E = egt_mod
    P.test_taubin_graph_replays_match_eager(_Named(E, TAUBIN_TILE=1024))
    g = E.GridStructure(D.sphere(30_000, seed=45), 1, 1e-6, 1024, 4)
    g.GRIDCUDAKNNSELF_COMPACT(16, 1e8)
    tiles = []
    for options in ((), ((E.OPT_TAUBIN_TILE, 1024),)):
        for o in options:
            g.set_option(*o)
        E.EGT_CUDA(g).PerformSmoothing(60, 0.5, -0.53, 0.65)
        tiles.append(g.stats()["taubin_tile"])
    g.close()
    assert tiles == [256, 1024]
