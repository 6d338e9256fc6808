"""Neighbour search on the device against the oracle (bit-exact sets).

The drop-in search evaluates the FP32 inclusion test of CompactNSearch's
default (float) build, strict d^2 < r^2 with ((dx dx + dy dy) + dz dz), self
excluded; the oracle evaluates the same test on the same FP32 positions, by
grid and by brute force (which agree, tests/test_oracle_ns.py). The time
step's own lists decide a pair within FP32 rounding of r^2 in FP64, as the
FP64 time step of the oracle does: they are compared with the oracle's FP64
search on the same (FP32) positions."""
import numpy as np
import pytest

from oracle import oracle
from splishsplash_amd import capi, scenes

pytestmark = pytest.mark.gpu


def csr_to_sets(off, idx):
    return [frozenset(idx[off[i]:off[i + 1]].tolist()) for i in range(len(off) - 1)]


def assert_same_csr(off_g, idx_g, off_o, idx_o):
    np.testing.assert_array_equal(np.diff(off_g.astype(np.int64)), np.diff(off_o.astype(np.int64)))
    for i in range(len(off_g) - 1):
        a = np.sort(idx_g[off_g[i]:off_g[i + 1]])
        b = np.sort(idx_o[off_o[i]:off_o[i + 1]])
        if not np.array_equal(a, b):
            raise AssertionError(f"point {i}: {a} vs {b}")


def radius_for(n, k=35.0):
    # ~k neighbours for n uniform points in the unit cube
    return float((k / (4.0 / 3.0 * np.pi * n)) ** (1 / 3))


@pytest.mark.parametrize("kind", ["uniform", "clustered"])
def test_drop_in_search_matches_oracle(kind):
    n = 60000
    x = scenes.uniform_points(n, seed=3) if kind == "uniform" else scenes.clustered_points(n, seed=3)
    x32 = np.ascontiguousarray(x, np.float32)
    r = radius_for(n)
    ns = capi.NeighborhoodSearch(r)
    i = ns.add_point_set(x32)
    ns.find_neighbors()
    off_g, idx_g = ns.neighbors_csr(i, i)
    off_o, idx_o = oracle.neighbors(x32, radius=np.float32(r))
    assert_same_csr(off_g, idx_g, off_o, idx_o)
    if kind == "uniform":
        assert 20 < np.diff(off_o).mean() < 60
    else:  # the clusters hold 80 % of the points in a small volume
        assert np.diff(off_o).mean() > 60


def test_drop_in_two_sets_activation_and_queries():
    rng = np.random.default_rng(9)
    fluid = np.ascontiguousarray(scenes.f32(rng.uniform(0.2, 0.8, (5000, 3))), np.float32)
    bnd = np.ascontiguousarray(scenes.box_wall_particles((0, 0, 0), (1, 1, 1), 0.05), np.float32)
    r = 0.1
    ns = capi.NeighborhoodSearch(r)
    f = ns.add_point_set(fluid, True, True, True)
    b = ns.add_point_set(bnd, False, False, True)  # Akinci: not searching, found
    assert ns.is_active(f, b) and ns.is_active(f, f)
    assert not ns.is_active(b, f) and not ns.is_active(b, b)
    ns.find_neighbors()
    off_g, idx_g = ns.neighbors_csr(f, b)
    off_o, idx_o = oracle.neighbors(fluid, bnd, radius=np.float32(r))
    assert_same_csr(off_g, idx_g, off_o, idx_o)
    # per-point accessors agree with the CSR view
    ps = ns.point_set(f)
    for k in (0, 17, 4999):
        lst = ps.neighbor_list(f, k)
        assert len(lst) == ps.n_neighbors(f, k)
        if len(lst):
            assert ps.neighbor(f, k, 0) == lst[0]
    # boundary-only activation (Simulation::updateBoundaryVolume pattern)
    ns.set_active(False)
    ns.set_active(b, True, True)
    ns.find_neighbors()
    off_g, idx_g = ns.neighbors_csr(b, b)
    off_o, idx_o = oracle.neighbors(bnd, radius=np.float32(r))
    assert_same_csr(off_g, idx_g, off_o, idx_o)
    # point query
    q = np.array([0.5, 0.5, 0.5])
    got = np.sort(ns.find_neighbors_point(q, f))
    d2 = ((fluid.astype(np.float32) - q.astype(np.float32)) ** 2).sum(1)
    assert set(got.tolist()) == set(np.nonzero(d2 < np.float32(r) * np.float32(r))[0].tolist())


def test_z_sort_and_sort_field():
    rng = np.random.default_rng(10)
    x = np.ascontiguousarray(scenes.f32(rng.uniform(0, 1, (3000, 3))), np.float32)
    ids = np.arange(len(x), dtype=np.uint32)
    ns = capi.NeighborhoodSearch(0.08)
    s = ns.add_point_set(x)
    ns.z_sort()
    ps = ns.point_set(s)
    x0 = x.copy()
    ps.sort_field(x)
    ps.sort_field(ids)
    np.testing.assert_array_equal(x, x0[ids])           # same permutation on both fields
    assert sorted(ids.tolist()) == list(range(len(x)))
    ns.find_neighbors()                                   # lists refer to the new order
    off_g, idx_g = ns.neighbors_csr(s, s)
    off_o, idx_o = oracle.neighbors(x, radius=np.float32(0.08))
    assert_same_csr(off_g, idx_g, off_o, idx_o)


def test_dfsph_internal_lists_match_oracle():
    sc = scenes.dam_break_small(per_side=30)
    g = capi.TimeStepDFSPH(sc["params"])
    g.set_fluid(sc["x"], sc["v"])
    g.add_boundary_particles(sc["boundary_x"])
    g.stage("neighborhood_search")
    x32 = np.ascontiguousarray(sc["x"], np.float32)
    off_g, idx_g = g.neighbors(boundary=False)
    x64 = x32.astype(np.float64)
    hs = 4.0 * sc["params"].particle_radius
    off_o, idx_o = oracle.neighbors(x64, radius=hs, dtype=np.float64)
    assert_same_csr(off_g, idx_g, off_o, idx_o)
    fluid_counts = np.diff(off_o)
    off_g, idx_g = g.neighbors(boundary=True)
    b64 = np.ascontiguousarray(sc["boundary_x"], np.float32).astype(np.float64)
    off_o, idx_o = oracle.neighbors(x64, b64, radius=hs, dtype=np.float64)
    assert_same_csr(off_g, idx_g, off_o, idx_o)
    cnt = g.get("fluid neighbor count")
    np.testing.assert_array_equal(cnt, fluid_counts)


def test_dfsph_lists_with_points_outside_the_grid():
    # Particles that leave the grid sit in its border cells; the lists trim
    # each row to the x reach of the query, and that trim must still find
    # every neighbour of a clamped point. Three blocks of the fluid are moved
    # beyond the grid (past +x, below -y, past +z), keeping their own
    # neighbourhoods, and the sets must equal the FP64 search.
    sc = scenes.dam_break_small(per_side=20)
    g = capi.TimeStepDFSPH(sc["params"])
    g.set_fluid(sc["x"], sc["v"])
    g.add_boundary_particles(sc["boundary_x"])
    g.stage("neighborhood_search")
    x = np.ascontiguousarray(g.get("position"), np.float32)
    order = np.argsort(x[:, 0] + 1e-3 * x[:, 1])
    for k, shift in enumerate(([5.0, 0.0, 0.0], [0.0, -3.0, 0.0], [0.0, 0.0, 4.0])):
        sel = order[400 * k:400 * k + 300]
        x[sel] += np.float32(shift)
    g.set("position", x)
    g.stage("neighborhood_search")
    off_g, idx_g = g.neighbors(boundary=False)
    hs = 4.0 * sc["params"].particle_radius
    off_o, idx_o = oracle.neighbors(x.astype(np.float64), radius=hs, dtype=np.float64)
    assert (np.diff(off_o) > 1).sum() > 0.9 * len(x)  # the moved blocks keep their neighbours
    assert_same_csr(off_g, idx_g, off_o, idx_o)


def test_microbench_uniform_literal_radius_small():
    # the microbenchmark's literal support radius 0.0375 at a reduced n
    n = 100000
    x = np.ascontiguousarray(scenes.uniform_points(n, seed=3), np.float32)
    ns = capi.NeighborhoodSearch(0.0375)
    s = ns.add_point_set(x)
    ns.find_neighbors()
    off_g, idx_g = ns.neighbors_csr(s, s)
    off_o, idx_o = oracle.neighbors(x, radius=np.float32(0.0375))
    assert_same_csr(off_g, idx_g, off_o, idx_o)


def test_dfsph_lists_beyond_the_lds_tile():
    # Clustered points with several hundred neighbours each: the time step's
    # lists take the path for capacities beyond the LDS tile; sets and the
    # FP32 densities still match the oracle.
    from splishsplash_amd.params import default_params
    x = np.ascontiguousarray(scenes.clustered_points(60000, seed=5, clusters=4, sigma=0.02), np.float32)
    h = 0.02
    prm = default_params(particle_radius=h / 4, boundary_handling_method=-1, viscosity_method=0)
    g = capi.TimeStepDFSPH(prm)
    g.set_fluid(x.astype(np.float64))
    g.stage("neighborhood_search")
    assert g.counters()["max_fluid_neighbors"] > 300
    off_g, idx_g = g.neighbors(boundary=False)
    off_o, idx_o = oracle.neighbors(x.astype(np.float64), radius=4.0 * prm.particle_radius, dtype=np.float64)
    assert_same_csr(off_g, idx_g, off_o, idx_o)
    g.stage("densities")
    o = oracle.OracleDFSPH(prm)
    o.set_fluid(x.astype(np.float64), np.zeros_like(x, np.float64))
    o.init()
    o.stage("neighborhood_search")
    o.stage("densities")
    ro = o.get("density")
    assert np.abs(g.get("density") - ro).max() / np.abs(ro).max() <= 1e-5


def test_empty_and_tiny_sets():
    ns = capi.NeighborhoodSearch(0.1)
    e = np.zeros((0, 3), np.float32)
    one = np.array([[0.5, 0.5, 0.5]], np.float32)
    a = ns.add_point_set(e)
    b = ns.add_point_set(one)
    ns.find_neighbors()
    assert ns.point_set(b).n_neighbors(b, 0) == 0
    assert ns.point_set(b).n_neighbors(a, 0) == 0
    assert ns.point_set(a).n_points() == 0


def expected_csr(x, radius, y=None):
    """The drop-in search's lists in its own order: (dz, dy) row, then cell
    along x, then point index (FP32 cell coordinates and inclusion test)."""
    src = x if y is None else y
    lo = np.minimum(x.min(0), src.min(0)).astype(np.float64)
    cs = radius * (1.0 + 1e-4)
    o, inv = (lo - cs).astype(np.float32), np.float32(1.0 / cs)
    cell = lambda p: np.floor((p - o) * inv).astype(np.int64)
    off, idx = oracle.neighbors(x, y, radius=np.float32(radius))
    i = np.repeat(np.arange(len(x)), np.diff(off.astype(np.int64)))
    d = cell(src)[idx] - cell(x)[i]
    order = np.lexsort((idx, d[:, 0], d[:, 1], d[:, 2], i))
    return off, idx[order]


@pytest.mark.parametrize("n,knot", [(1, 0), (63, 0), (65, 40), (700, 700), (5003, 900), (65536, 0), (65537, 0),
                                    (131071, 0), (131072, 0), (131109, 1500)])
def test_drop_in_lists_keep_their_order(n, knot):
    """Sizes around a wave, around the first query that a wave takes beside
    another and around the switch between a wave and a lane per query; `knot` points crowd into a corner of one cell, so that rows
    hold far more candidates than one window or hit word."""
    rng = np.random.default_rng(n)
    x = rng.uniform(0.0, 1.0, (n, 3)).astype(np.float32)
    r = max(radius_for(n, 20.0), 0.02) if n > 1 else 0.1
    x[rng.permutation(n)[:knot]] = (0.5 + rng.uniform(0.0, 0.6 * r, (knot, 3))).astype(np.float32)
    ns = capi.NeighborhoodSearch(r)
    i = ns.add_point_set(x)
    ns.find_neighbors()
    off, idx = ns.neighbors_csr(i, i)
    off_e, idx_e = expected_csr(x, r)
    np.testing.assert_array_equal(off, off_e)
    np.testing.assert_array_equal(idx, idx_e)


@pytest.mark.parametrize("n", [300, 140007])
def test_drop_in_lists_of_two_sets_keep_their_order(n):
    rng = np.random.default_rng(n)
    x = rng.uniform(0.0, 1.0, (n, 3)).astype(np.float32)
    y = scenes.box_wall_particles((-0.1, 0, 0), (1, 1, 1), 0.05).astype(np.float32)
    r = 0.06
    ns = capi.NeighborhoodSearch(r)
    # the queries' own set is not searched, so it is not in cell order
    a = ns.add_point_set(x, True, True, False)
    b = ns.add_point_set(y, False, False, True)
    ns.find_neighbors()
    off, idx = ns.neighbors_csr(a, b)
    off_e, idx_e = expected_csr(x, r, y)
    np.testing.assert_array_equal(off, off_e)
    np.testing.assert_array_equal(idx, idx_e)


@pytest.mark.parametrize("n", [2, 4094, 4096, 4098, 1024 * 4096, 1024 * 4096 + 2])
def test_list_offsets_at_the_limits_of_the_scans(n):
    # Pairs of points that see only each other: the offsets are a scan of n
    # ones, by one block up to 4,096 values, by two launches up to 4,096
    # tiles of 1,024, by three beyond.
    k = np.arange(n // 2)
    a = 0.1 * np.stack([k % 128, k // 128 % 128, k // 16384], 1)
    x = np.empty((n, 3), np.float32)
    x[0::2] = a
    x[1::2] = a + 0.01
    ns = capi.NeighborhoodSearch(0.05)
    ns.add_point_set(x)
    ns.find_neighbors()
    off, idx = ns.neighbors_csr(0, 0)
    np.testing.assert_array_equal(off, np.arange(n + 1))
    np.testing.assert_array_equal(idx, np.arange(n) ^ 1)
