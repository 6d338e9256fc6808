"""DFSPH stages on the device against the FP64 oracle from identical states.

Before every stage the oracle is given the device's current state (FP32
values, exact in FP64), both run the stage, and the stage's outputs are
compared normwise: max|gpu - oracle| / max|oracle| <= 1e-5 (FP32 bulk
arithmetic against the FP64 reference; the kernel-table index is decided in
FP64 near step boundaries so both read the same table entries)."""
import os

import numpy as np
import pytest
from scipy.spatial import cKDTree

from oracle import oracle
from splishsplash_amd import capi, learned, scenes
from splishsplash_amd.params import BOUNDARY_BENDER2019, BOUNDARY_NONE, VISCOSITY_STANDARD, VISCOSITY_WEILER2018, default_params

pytestmark = pytest.mark.gpu

TOL = 1e-5
STATE = ["position", "velocity", "acceleration", "density", "factor", "advected density", "p / rho^2",
         "p_v / rho^2", "pressure acceleration", "velocity difference"]

OUTPUTS = {
    "densities": ["density"],
    "dfsph_factor": ["factor"],
    "divergence_setup": ["advected density", "factor", "p_v / rho^2"],
    "divergence_iter": ["pressure acceleration", "p_v / rho^2"],
    "divergence_finish": ["velocity", "factor", "p_v / rho^2"],
    "clear_accel": ["acceleration"],
    "viscosity": ["acceleration"],
    "xsph": ["acceleration"],
    "update_velocity": ["velocity"],
    "pressure_setup": ["advected density", "factor", "p / rho^2"],
    "pressure_iter": ["pressure acceleration", "p / rho^2"],
    "pressure_finish": ["velocity", "p / rho^2"],
    "update_position": ["position"],
}


def rel(a, b):
    return float(np.abs(np.asarray(a, np.float64) - b).max() / max(np.abs(b).max(), 1e-30))


def sync_state(g, o, extra=()):
    for nm in STATE + list(extra):
        o.set(nm, g.get(nm).astype(np.float64))
    c = g.counters()
    o.set_time(c["time"], c["time_step_size"])


def make_pair(params, x, v, boundary_x=None, vm=None, spheres=(), meshes=()):
    g = capi.TimeStepDFSPH(params)
    g.set_fluid(x, v)
    o = oracle.OracleDFSPH(params)
    o.set_fluid(x, v)
    if boundary_x is not None:
        g.add_boundary_particles(boundary_x)
        o.add_boundary_particles(boundary_x)
    if vm is not None:
        g.set_volume_map_box(*vm)
        o.set_volume_map_box(*vm)
    for c, r in spheres:
        g.add_volume_map_sphere(c, r, 0.05)
        o.add_volume_map_sphere(c, r, 0.05)
    for verts, faces, res in meshes:
        g.add_volume_map_mesh(verts, faces, res)
        o.add_volume_map_mesh(verts, faces, res)
    o.init()
    g.init()
    return g, o


def perturbed_state(x, seed=0):
    rng = np.random.default_rng(seed)
    v = scenes.f32(rng.normal(0.0, 0.3, x.shape))
    p = scenes.f32(rng.uniform(0.0, 3e-4, len(x)))
    pv = scenes.f32(rng.uniform(0.0, 0.6, len(x)))
    return v, p, pv


def run_stage_sequence(g, o, seq, extra_state=(), tol=None):
    report = {}
    for st in seq:
        sync_state(g, o, extra_state)
        g.stage(st)
        o.stage(st)
        for nm in OUTPUTS.get(st, []):
            e = rel(g.get(nm), o.get(nm))
            report[(st, nm)] = e
            bound = (tol or {}).get(st, TOL)
            assert e <= bound, f"{st}: {nm} rel err {e:.3e}"
        if st == "cfl":
            hg, ho = g.counters()["time_step_size"], o.counters()["time_step_size"]
            assert hg == pytest.approx(ho, rel=1e-6)
        if st in ("divergence_iter", "pressure_iter"):
            k = "avg_divergence_err" if st == "divergence_iter" else "avg_density_err"
            eg, eo = g.counters()[k], o.counters()[k]
            assert eg == pytest.approx(eo, rel=1e-4, abs=1e-9 * max(1.0, abs(eo)))
            k = "avg_overpressure_err" + ("_v" if st == "divergence_iter" else "")
            eg, eo = g.counters()[k], o.counters()[k]
            assert eg == pytest.approx(eo, rel=1e-3, abs=1e-7 * max(1.0, abs(eo)))
    return report


STEP_SEQ = ["densities", "dfsph_factor", "divergence_setup", "divergence_iter", "divergence_iter",
            "divergence_finish", "clear_accel", "xsph", "cfl", "update_velocity", "pressure_setup",
            "pressure_iter", "pressure_iter", "pressure_finish", "update_position"]


def test_kernel_table_on_device():
    rng = np.random.default_rng(1)
    h = 0.1
    d = rng.normal(size=(20000, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    r = scenes.f32(d * rng.uniform(0, 1.02 * h, (20000, 1)))
    w, gw = capi.kernel_eval(h, r)
    wo, go = oracle.kernel_eval(h, r)
    assert rel(w, wo) <= 2e-6
    assert rel(gw, go) <= 2e-6


def test_akinci_stages_match_oracle():
    sc = scenes.dam_break_small(per_side=30)
    v, p, pv = perturbed_state(sc["x"], seed=1)
    g, o = make_pair(sc["params"], sc["x"], v, boundary_x=sc["boundary_x"])
    assert rel(g.get("boundary particle volume"), o.get_boundary_volumes(len(sc["boundary_x"]))) <= TOL
    g.set_time(0.0, 0.004)
    o.set_time(0.0, 0.004)
    g.stage("neighborhood_search")
    o.stage("neighborhood_search")
    g.set("p / rho^2", p)
    g.set("p_v / rho^2", pv)
    run_stage_sequence(g, o, STEP_SEQ)


@pytest.mark.parametrize("lanes", [2, 4])
def test_solver_sweeps_with_split_neighbour_sums(lanes):
    # The solver sweeps can split each particle's neighbour sum over 2 or 4
    # lanes (a different FP32 summation order); every stage output stays
    # within the same bound of the oracle, and whole steps still converge
    # like the oracle's.
    sc = scenes.dam_break_small(per_side=30)
    v, p, pv = perturbed_state(sc["x"], seed=3)
    g, o = make_pair(sc["params"], sc["x"], v, boundary_x=sc["boundary_x"])
    g.set_lanes_per_particle(lanes)
    g.set_time(0.0, 0.004)
    o.set_time(0.0, 0.004)
    g.stage("neighborhood_search")
    o.stage("neighborhood_search")
    g.set("p / rho^2", p)
    g.set("p_v / rho^2", pv)
    run_stage_sequence(g, o, STEP_SEQ)
    assert g.counters()["lanes_per_particle"] == lanes


@pytest.mark.parametrize("side", [3, 11, 26])
@pytest.mark.parametrize("kw", [{}, {"viscosity_method": 1, "viscosity": 0.05}, {"viscosity_method": 6}])
def test_shared_pairs_sum_as_one_lane(side, kw):
    # For small counts 16 lanes evaluate a particle's pairs and its sums
    # are taken in list order: bit for bit the fields of one lane per
    # particle, over whole steps with walls, XSPH and both viscosities. A
    # block of 27 particles has fewer neighbours than lanes; compressed to
    # 0.75 of its spacing a particle has more than one round of 64.
    sc = scenes.dam_break_small(per_side=side, **kw)
    x = (sc["x"] - 0.05) * (0.75 if side == 11 else 1.0)
    v, p, pv = perturbed_state(x, seed=side)
    sims = []
    for lanes in (0, 1):
        g = capi.TimeStepDFSPH(sc["params"])
        g.set_fluid(x, v)
        g.add_boundary_particles(sc["boundary_x"])
        g.set_lanes_per_particle(lanes)
        g.init()
        g.set("p / rho^2", p)
        g.set("p_v / rho^2", pv)
        g.step(1 if side == 11 else 3)  # (the compressed block bursts)
        sims.append(g)
    assert sims[0].counters()["lanes_per_particle"] == 16 and sims[1].counters()["lanes_per_particle"] == 1
    if side == 11:
        assert sims[0].get("fluid neighbor count").max() > 64
    for f in ("position", "velocity", "density", "factor", "p / rho^2", "p_v / rho^2", "pressure acceleration"):
        np.testing.assert_array_equal(sims[0].get(f), sims[1].get(f), err_msg=f)


@pytest.mark.parametrize("dims, n, lanes", [
    ((42, 40, 40), 65535, (1, 1)), ((42, 40, 40), 65536, (4, 4)), ((44, 44, 44), 83999, (4, 4)),
    ((44, 44, 44), 84000, (2, 4)), ((49, 49, 49), 111999, (2, 4)), ((49, 49, 49), 112000, (2, 2)),
    ((62, 62, 62), 235999, (2, 2)), ((62, 62, 62), 236000, (2, 1)), ((240, 100, 10), 240000, (2, 2))])
def test_lanes_of_large_scenes_follow_their_rule(dims, n, lanes):
    # The lanes fix the order of the sums, so they come from the count and
    # the lists alone and every handle with the same particles takes the
    # same: on both sides of each line, with packed lists and (the wide flat
    # block, 48,000 slots a layer of cells) with 32-bit ones.
    x = scenes.lattice_block(dims, 0.05, (0.0, 0.0, 0.0), jitter=0.001, seed=1)[:n]
    got = []
    for _ in range(3):
        g = capi.TimeStepDFSPH(default_params(boundary_handling_method=BOUNDARY_NONE))
        g.set_fluid(x)
        g.step(1)
        c = g.counters()
        got.append((c["lanes_per_particle"], c["lanes_per_particle_accel"], c["packed_lists"]))
    assert got == [(*lanes, int(dims[0] < 100))] * 3


def test_lanes_of_long_lists_follow_their_rule():
    # Four lanes from lists of 88 neighbours on, at any count: a block of
    # 240,000 particles with 1 to 88 more in one spot beside it.
    block = scenes.lattice_block((63, 63, 63), 0.05, (0.0, 0.0, 0.0), jitter=0.001, seed=1)[:240000]
    spot = np.float32([1.5, 1.5, -1.0]) + np.random.default_rng(8).uniform(-0.01, 0.01, (89, 3)).astype(np.float32)
    for k, lanes in ((1, (2, 1)), (88, (2, 1)), (89, (4, 4))):
        g = capi.TimeStepDFSPH(default_params(boundary_handling_method=BOUNDARY_NONE))
        g.set_fluid(scenes.f32(np.concatenate([block, spot[:k]])))
        g.stage("neighborhood_search")
        g.stage("densities")
        c = g.counters()
        assert g.get("fluid neighbor count").max() == max(32, k - 1)
        assert (c["lanes_per_particle"], c["lanes_per_particle_accel"]) == lanes


def tile_unions(x, h, lo):
    """Per 256 consecutive particles in cell order (rows of z and y, quarter
    cells along x, the grid's origin two supports and a cell below lo): how
    many particles are neighbours of one of them."""
    cell = h * (1 + 1e-4)
    c = np.floor((x - (np.asarray(lo) - 2 * h - cell)) / cell * [4, 1, 1]).astype(np.int64)
    order = np.lexsort((c[:, 0], c[:, 1], c[:, 2]))
    lists = cKDTree(x.astype(np.float64)).query_ball_point(x[order].astype(np.float64), h)
    return np.array([len({j for i, near in zip(order[b:b + 256], lists[b:b + 256]) for j in near if j != i})
                     for b in range(0, len(x), 256)])


@pytest.mark.parametrize("walls", ["akinci", "bender"])
@pytest.mark.parametrize("lanes", [1, 2])
def test_tiled_iterations_match_gathered_ones(walls, lanes):
    # Whole steps of a scene alone, whose iterations read neighbours from
    # tiles in LDS, against the same scene in a batched solve, which gathers
    # from the same packed lists: bit for bit. Compressed to 0.85 of its
    # spacing the long block has tiles that fit their share of LDS and tiles
    # that do not; 133,771 particles leave the last one ragged, and particles
    # strewn alone have no neighbours.
    sc = scenes.dam_break_small(boundary=walls, max_error=0.001, max_error_v=0.01, viscosity_method=VISCOSITY_STANDARD,
                                viscosity=0.01)
    block = scenes.lattice_block((88, 40, 38), 0.0425, (0.1, 0.1, 0.1), jitter=0.001, seed=1)
    alone = scenes.f32([[3.95, 2.2 + 0.05 * (k % 2), 0.1 + 0.15 * k] for k in range(11)])
    x = scenes.f32(np.concatenate([block, alone]))
    assert len(x) == 133771
    over = np.count_nonzero(tile_unions(x, 0.1, (0.0, 0.0, 0.0)) > 1856)
    assert 100 < over < 200  # of 523 tiles
    sims = []
    for batched in (False, True):
        g = learned.make_sim(dict(sc, x=x, v=np.zeros_like(x)))
        g.set_lanes_per_particle(lanes)
        g.enable_timing()
        capi.set_batch_mode("batched")
        try:
            if batched:
                capi.step_batch([g], 3)
            else:
                g.step(3)
        finally:
            capi.set_batch_mode("auto")
        sims.append(g)
    a, b = sims
    assert "tile_lists" in a.kernel_stats() and "tile_lists" not in b.kernel_stats()
    for f in ("position", "velocity", "p / rho^2", "p_v / rho^2", "pressure acceleration"):
        assert np.isfinite(a.get(f)).all()
        np.testing.assert_array_equal(a.get(f), b.get(f), err_msg=f)
    ca, cb = a.counters(), b.counters()
    for c in ("total_iterations", "total_iterations_v", "avg_density_err", "avg_divergence_err", "time"):
        assert ca[c] == cb[c], c


@pytest.mark.parametrize("mode", ["reference", "previous"])
def test_tiled_steps_match_gathered_ones_from_either_start(mode):
    # Whole steps from both starts, from tiles and, with 300 fixed particles
    # in one spot outside the walls whose row of candidates leaves no packed
    # lists, gathered: with one lane per particle the fluid's sums are the
    # same. Fixed iteration counts and time step: the spot has a share in the
    # mean errors, and nothing else.
    block = scenes.lattice_block((53, 50, 50), 0.05, (0.1, 0.1, 0.1), jitter=0.001, seed=1)
    spot = np.float32([3.2, 2.6, 4.2]) + np.random.default_rng(8).uniform(-0.01, 0.01, (300, 3)).astype(np.float32)
    params = default_params(cfl_method=0, time_step_size=0.001, min_iterations=24, max_iterations=24,
                            max_iterations_v=8, max_error_v=1e-9, xsph=0.01)
    v = perturbed_state(block, seed=11)[0]
    out = []
    for extra in (spot[:0], spot):
        g = capi.TimeStepDFSPH(params)
        g.set_fluid(scenes.f32(np.concatenate([block, extra])), scenes.f32(np.concatenate([v, 0 * extra])))
        g.add_boundary_particles(scenes.box_wall_particles((0.0, 0.0, 0.0), (4.0, 3.0, 2.7), 0.05))
        g.set_lanes_per_particle(1)
        g.enable_timing()
        g.init()
        for solver in learned.SOLVERS:
            g.set_warm_start_mode(solver, mode)
            g.set_warm_start_policy(solver, 0)
        g.set("state", np.concatenate([np.zeros(len(block)), np.full(len(extra), 2)]).astype(np.uint32))
        g.step(4)
        c = g.counters()
        assert ("tile_lists" in g.kernel_stats()) == (len(extra) == 0) == (c["packed_lists"] == 1)
        assert c["total_iterations"] == 4 * 24 and c["total_iterations_v"] == 4 * 8
        out.append({f: g.get(f)[:len(block)] for f in ("position", "velocity", "p / rho^2", "p_v / rho^2")})
    for f, a in out[0].items():
        assert np.isfinite(a).all()
        np.testing.assert_array_equal(a, out[1][f], err_msg=f)


def test_tiles_are_built_once_the_iterations_pay_for_them():
    # At 120,384 particles tiles pay from 20 iterations on one list. The
    # last solves' counts are 3 for a new handle, so they are built once the
    # lists have seen 40.
    x = scenes.lattice_block((76, 44, 36), 0.05, (0.1, 0.1, 0.1), jitter=0.001, seed=1)
    g = capi.TimeStepDFSPH(default_params(boundary_handling_method=BOUNDARY_NONE))
    g.set_fluid(x)
    g.enable_timing()
    for _ in range(2):
        g.stage("neighborhood_search")
        g.stage("densities")
        g.stage("dfsph_factor")
        g.stage("pressure_setup")
        for _ in range(40):
            g.stage("pressure_iter")
        assert "tile_lists" not in g.kernel_stats()
    g.stage("pressure_iter")
    assert g.kernel_stats()["tile_lists"][0] == 1


def test_tiles_that_are_mostly_overfull_wait():
    # At 0.8 of its spacing 324 of the block's 520 tiles outgrow their share
    # of LDS: after one solve the next 16 lists go without tiles.
    sc = scenes.dam_break_small(boundary="bender")
    x = scenes.lattice_block((95, 40, 35), 0.04, (0.1, 0.1, 0.1), jitter=0.001, seed=1)
    assert 300 < np.count_nonzero(tile_unions(x, 0.1, (0.0, 0.0, 0.0)) > 1856) < 350
    g = learned.make_sim(dict(sc, x=x, v=np.zeros_like(x)))
    g.enable_timing()
    for k in range(18):
        for stage in ("neighborhood_search", "volume_maps", "densities", "dfsph_factor", "pressure_solve"):
            g.stage(stage)
        assert g.kernel_stats()["tile_lists"][0] == (1 if k < 17 else 2)


def vm_scene(n=16, corner=0.06):
    x = scenes.lattice_block((n, n, n), 0.05, (corner, corner, corner), jitter=0.002, seed=5)
    # three particles inside the wall (projected back by the volume-map stage)
    x = np.concatenate([x, scenes.f32([[-0.01, 0.5, 0.5], [0.5, -0.004, 0.4], [0.3, 0.3, -0.02]])])
    lo, hi = (0.0, 0.0, 0.0), (2.0, 1.5, 1.5)
    res = scenes.volume_map_resolution(lo, hi, 0.1, 0.05)
    params = default_params(boundary_handling_method=BOUNDARY_BENDER2019, xsph=0.01, xsph_boundary=0.02,
                            cfl_factor=1.0, time_step_size=0.004)
    return x, params, (lo, hi, res)


def test_volume_map_stages_match_oracle():
    x, params, vm = vm_scene()
    v, p, pv = perturbed_state(x, seed=2)
    g, o = make_pair(params, x, v, vm=vm)
    g.stage("neighborhood_search")
    o.stage("neighborhood_search")
    sync_state(g, o)
    g.stage("volume_maps")
    o.stage("volume_maps")
    for nm in ("boundary volume", "boundary x", "position", "velocity"):
        e = rel(g.get(nm), o.get(nm))
        assert e <= TOL, f"volume_maps: {nm} rel err {e:.3e}"
    vb = o.get("boundary volume")
    assert (vb > 0).sum() > 500  # the wall is seen by the near-wall layers
    xg = g.get("position")
    assert (xg[-3:] != x[-3:]).any(axis=1).all()  # wall particles were projected
    g.set("p / rho^2", p)
    g.set("p_v / rho^2", pv)
    run_stage_sequence(g, o, STEP_SEQ, extra_state=("boundary volume", "boundary x"))


def test_volume_map_spheres_match_oracle():
    # Box wall plus two sphere obstacles cutting into the fluid block: the
    # particles inside a sphere are projected out of it, and near-surface
    # particles see up to three boundary objects (summed in object order).
    x, params, vm = vm_scene()
    spheres = [((0.45, 0.45, 0.45), 0.12), ((0.80, 0.35, 0.60), 0.15)]
    v, p, pv = perturbed_state(x, seed=4)
    g, o = make_pair(params, x, v, vm=vm, spheres=spheres)
    g.stage("neighborhood_search")
    o.stage("neighborhood_search")
    sync_state(g, o)
    g.stage("volume_maps")
    o.stage("volume_maps")
    names = ["position", "velocity"]
    for k in range(3):
        names += [f"boundary volume {k}", f"boundary x {k}"]
    for nm in names:
        e = rel(g.get(nm), o.get(nm))
        assert e <= TOL, f"volume_maps: {nm} rel err {e:.3e}"
    for k in (1, 2):
        assert (o.get(f"boundary volume {k}") > 0).sum() > 50
    inside = [np.linalg.norm(x - np.array(c), axis=1) < r for c, r in spheres]
    moved = (g.get("position") != x).any(axis=1)
    assert moved[inside[0] | inside[1]].all()
    g.set("p / rho^2", p)
    g.set("p_v / rho^2", pv)
    run_stage_sequence(g, o, STEP_SEQ, extra_state=tuple(names[2:]))


@pytest.mark.parametrize("lanes", [1, 2, 4])
def test_weiler_viscosity_matches_oracle(lanes):
    sc = scenes.dam_break_small(per_side=20)
    prm = sc["params"]
    prm.viscosity_method = VISCOSITY_WEILER2018
    prm.viscosity = 0.05
    prm.visco_max_error = 1e-5
    prm.visco_max_iter = 200
    rng = np.random.default_rng(3)
    v = scenes.f32(rng.normal(0.0, 0.5, sc["x"].shape))
    g, o = make_pair(prm, sc["x"], v, boundary_x=sc["boundary_x"])
    g.set_lanes_per_particle(lanes)
    g.set_time(0.0, 0.004)
    o.set_time(0.0, 0.004)
    for st in ("neighborhood_search", "densities"):
        g.stage(st)
        o.stage(st)
    g.set("velocity difference", scenes.f32(rng.normal(0.0, 0.01, v.shape)))
    sync_state(g, o)
    g.stage("clear_accel")
    o.stage("clear_accel")
    g.stage("viscosity")
    o.stage("viscosity")
    vn_g = g.get("velocity") + g.get("velocity difference")
    vn_o = o.get("velocity") + o.get("velocity difference")
    assert rel(vn_g, vn_o) <= 1e-4
    dv_o = o.get("velocity difference")
    assert np.abs(g.get("velocity difference") - dv_o).max() <= 1e-4 * np.abs(vn_o).max()
    ig, io = g.counters()["visco_iterations"], o.counters()["visco_iterations"]
    assert abs(ig - io) <= 2, (ig, io)
    assert io > 2


@pytest.mark.parametrize("lanes", [1, 2])
def test_full_step_matches_oracle_and_converges(lanes):
    sc = scenes.dam_break_small(per_side=20)
    g, o = make_pair(sc["params"], sc["x"], sc["v"], boundary_x=sc["boundary_x"])
    g.set_lanes_per_particle(lanes)
    eta = sc["params"].max_error * 0.01 * 1000.0
    for step in range(12):
        sync_state(g, o)
        g.step(1)
        o.step(1)
        cg, co = g.counters(), o.counters()
        # split sums change the FP32 summation order: a solve may end one
        # iteration earlier or later at the tolerance boundary
        assert abs(cg["iterations"] - co["iterations"]) <= (0 if lanes == 1 else 1), \
            (step, cg["iterations"], co["iterations"])
        assert cg["avg_density_err"] <= eta
        assert cg["time_step_size"] == pytest.approx(co["time_step_size"], rel=1e-6)
        for nm in ("position", "velocity"):
            e = rel(g.get(nm), o.get(nm))
            assert e <= 1e-4, f"step {step}: {nm} rel err {e:.3e}"
    assert cg["flags"] == 0


def test_dam_break_runs_stably():
    sc = scenes.dam_break_small(per_side=30)
    g = capi.TimeStepDFSPH(sc["params"])
    g.set_fluid(sc["x"], sc["v"])
    g.add_boundary_particles(sc["boundary_x"])
    eta = sc["params"].max_error * 0.01 * 1000.0
    for _ in range(40):
        g.step(1)
        c = g.counters()
        assert c["avg_density_err"] <= eta or c["iterations"] == 100
    x = g.get("position")
    assert np.isfinite(x).all() and c["flags"] == 0
    assert (x > -0.03).all() and (x[:, 0] < 4.03).all() and (x[:, 1] < 3.03).all() and (x[:, 2] < 2.03).all()
    assert x[:, 1].mean() < sc["x"][:, 1].mean()


def test_reset_zeroes_solver_fields_and_counters():
    # TimeStepDFSPH::reset: the solver fields and iteration counters return
    # to zero, positions, velocities and densities stay; the next step is the
    # oracle's step from that state.
    sc = scenes.dam_break_small(per_side=16)
    g, o = make_pair(sc["params"], sc["x"], sc["v"], boundary_x=sc["boundary_x"])
    g.step(60)  # past the start, where the lattice (0.8 rho0) is under-dense and p = 0
    x, v, rho = g.get("position"), g.get("velocity"), g.get("density")
    assert g.get("p / rho^2").max() > 0 and g.counters()["total_iterations"] > 0
    g.reset()
    for nm in ("p / rho^2", "p_v / rho^2", "factor", "advected density", "pressure acceleration"):
        assert not g.get(nm).any(), nm
    c = g.counters()
    assert c["iterations"] == 0 and c["iterations_v"] == 0 and c["total_iterations"] == 0 and c["steps"] == 0
    np.testing.assert_array_equal(g.get("position"), x)
    np.testing.assert_array_equal(g.get("velocity"), v)
    np.testing.assert_array_equal(g.get("density"), rho)
    for _ in range(2):
        sync_state(g, o)
        g.step(1)
        o.step(1)
        assert g.counters()["iterations"] == o.counters()["iterations"]
        for nm in ("position", "velocity"):
            assert rel(g.get(nm), o.get(nm)) <= 1e-4, nm


def test_emitted_particles_keep_state_and_join_the_step():
    # Emission (emitter + emittedParticles + resize): the existing particles
    # keep every field, the new ones get the next ids, their positions and
    # velocities and zero stiffness, and the following steps treat them like
    # any other particle (oracle from identical states).
    sc = scenes.dam_break_small(per_side=16)
    g, o = make_pair(sc["params"], sc["x"], sc["v"], boundary_x=sc["boundary_x"])
    g.step(60)
    assert g.get("p / rho^2").max() > 0
    keep = ("position", "velocity", "p / rho^2", "p_v / rho^2", "velocity difference")
    before = {nm: g.get(nm) for nm in keep}
    n = g.n
    s = np.arange(5, dtype=np.float32) * 0.05
    new = np.stack(np.meshgrid(s, s, s, indexing="ij"), -1).reshape(-1, 3) + np.float32([1.5, 1.2, 0.6])
    vnew = np.tile(np.float32([0.0, -1.0, 0.0]), (len(new), 1))
    for _ in range(3):  # the first emission grows the device arrays, the others use the headroom
        g.emit_particles(new, vnew)
        new = new + np.float32([0.3, 0.0, 0.0])
    assert g.n == n + 3 * 125
    for nm in keep:
        np.testing.assert_array_equal(g.get(nm)[:n], before[nm])
    assert not g.get("p / rho^2")[n:].any() and not g.get("p_v / rho^2")[n:].any()
    np.testing.assert_array_equal(g.get("velocity")[n:], np.tile(vnew, (3, 1)))
    o.set_fluid(g.get("position"), g.get("velocity"))
    for step in range(3):
        sync_state(g, o)
        g.step(1)
        o.step(1)
        assert g.counters()["iterations"] == o.counters()["iterations"], step
        for nm in ("position", "velocity"):
            assert rel(g.get(nm), o.get(nm)) <= 1e-4, (step, nm)
    # emission before the first step is the same as handing all particles
    # to set_fluid
    a = capi.TimeStepDFSPH(sc["params"])
    a.set_fluid(sc["x"][:-100], sc["v"][:-100])
    a.emit_particles(sc["x"][-100:], sc["v"][-100:])
    a.add_boundary_particles(sc["boundary_x"])
    b = capi.TimeStepDFSPH(sc["params"])
    b.set_fluid(sc["x"], sc["v"])
    b.add_boundary_particles(sc["boundary_x"])
    a.step(3)
    b.step(3)
    np.testing.assert_array_equal(a.get("position"), b.get("position"))


@pytest.mark.parametrize("bmode", ["akinci", "bender"])
def test_standard_viscosity_matches_oracle(bmode):
    # Viscosity_Standard (explicit, the method of the reference's own dam
    # break scenes) with fluid and boundary viscosity: the viscosity stage
    # and every other stage from identical states, then whole steps.
    if bmode == "akinci":
        sc = scenes.dam_break_small(per_side=20)
        x, prm = sc["x"] - np.float32(0.06), sc["params"]
        kw = dict(boundary_x=sc["boundary_x"])
        extra = ()
    else:
        x, prm, vm = vm_scene()
        kw = dict(vm=vm)
        extra = ("boundary volume", "boundary x")
    prm.viscosity_method = VISCOSITY_STANDARD
    prm.viscosity = 0.05
    prm.viscosity_boundary = 0.3
    v, p, pv = perturbed_state(x, seed=6)
    g, o = make_pair(prm, x, v, **kw)
    g.set_time(0.0, 0.004)
    o.set_time(0.0, 0.004)
    g.stage("neighborhood_search")
    o.stage("neighborhood_search")
    if bmode == "bender":
        sync_state(g, o)
        g.stage("volume_maps")
        o.stage("volume_maps")
    g.set("p / rho^2", p)
    g.set("p_v / rho^2", pv)
    seq = list(STEP_SEQ)
    seq.insert(seq.index("clear_accel") + 1, "viscosity")
    # With volume maps the boundary term samples four points on the tangent
    # plane of each boundary point; the device forms them in FP32, the
    # oracle in FP64, so a sample can fall on the other side of a kernel
    # table step (a 1e-4 change of that term), as for the Weiler2018 samples.
    run_stage_sequence(g, o, seq, extra_state=extra, tol={"viscosity": 1e-4} if bmode == "bender" else None)
    step_tol = 5e-4 if bmode == "bender" else 1e-4  # the sample-point effect above, through a whole step
    for step in range(4):
        sync_state(g, o, extra)
        g.step(1)
        o.step(1)
        assert g.counters()["iterations"] == o.counters()["iterations"], step
        for nm in ("position", "velocity"):
            assert rel(g.get(nm), o.get(nm)) <= step_tol, (step, nm)


def test_volume_map_mesh_matches_oracle():
    # A sphere obstacle given as a closed triangle mesh (528 facets): its
    # distance field comes from the triangles, its volume field from the
    # interpolated distance field. Next to the analytic box wall, every
    # stage matches the oracle's mesh map, and the facetted sphere stays
    # within the chord error of the analytic one.
    x, params, vm = vm_scene()
    verts, faces = scenes.read_obj(os.path.join(scenes.DATA, "unit_sphere.obj"))
    centre, radius = np.array([0.45, 0.45, 0.45]), 0.13
    verts = verts * radius + centre
    res = [19, 19, 19]
    v, p, pv = perturbed_state(x, seed=7)
    g, o = make_pair(params, x, v, vm=vm, meshes=[(verts, faces, res)])
    g.stage("neighborhood_search")
    o.stage("neighborhood_search")
    sync_state(g, o)
    g.stage("volume_maps")
    o.stage("volume_maps")
    names = ["position", "velocity"]
    for k in range(2):
        names += [f"boundary volume {k}", f"boundary x {k}"]
    for nm in names:
        e = rel(g.get(nm), o.get(nm))
        assert e <= TOL, f"volume_maps: {nm} rel err {e:.3e}"
    vb = o.get("boundary volume 1")
    assert (vb > 0).sum() > 50
    inside = np.linalg.norm(x - centre, axis=1) < radius * 0.97
    moved = (g.get("position") != x).any(axis=1)
    assert inside.sum() > 10 and moved[inside].all()
    g.set("p / rho^2", p)
    g.set("p_v / rho^2", pv)
    run_stage_sequence(g, o, STEP_SEQ, extra_state=tuple(names[2:]))


@pytest.mark.parametrize("visc", ["standard", "weiler"])
def test_density_map_stages_match_oracle(visc):
    # Koschier2017: the box wall and a sphere obstacle as density maps; the
    # sampling (boundary density, its gradient, the boundary point, particles
    # moved out of the wall) and every stage with the density-map terms
    # (density, factor, density change, pressure accelerations, a_ij p_j,
    # XSPH, standard or Weiler2018 boundary viscosity) from identical states
    from splishsplash_amd.params import BOUNDARY_KOSCHIER2017
    x, params, vm = vm_scene()
    params.boundary_handling_method = BOUNDARY_KOSCHIER2017
    if visc == "standard":
        params.viscosity_method = VISCOSITY_STANDARD
        params.viscosity = 0.01
        params.viscosity_boundary = 0.02
    else:
        params.viscosity_method = VISCOSITY_WEILER2018
        params.viscosity = 0.05
        params.viscosity_boundary = 0.05
        params.visco_max_error = 1e-5
        params.visco_max_iter = 200
    spheres = [((0.45, 0.45, 0.45), 0.12)]
    v, p, pv = perturbed_state(x, seed=6)
    g, o = make_pair(params, x, v, vm=vm, spheres=spheres)
    g.stage("neighborhood_search")
    o.stage("neighborhood_search")
    sync_state(g, o)
    g.stage("volume_maps")
    o.stage("volume_maps")
    names = ["position", "velocity"]
    for k in range(2):
        names += [f"boundary density {k}", f"boundary density gradient {k}", f"boundary x {k}"]
    for nm in names:
        e = rel(g.get(nm), o.get(nm))
        assert e <= TOL, f"volume_maps: {nm} rel err {e:.3e}"
    assert (o.get("boundary density 0") > 0).sum() > 500 and (o.get("boundary density 1") > 0).sum() > 20
    assert (g.get("position") != x).any(axis=1).sum() >= 3  # particles in the wall and the sphere moved out
    g.set("p / rho^2", p)
    g.set("p_v / rho^2", pv)
    seq = STEP_SEQ[:6] + ["clear_accel", "viscosity", "xsph"] + STEP_SEQ[8:]
    tol = {"viscosity": 1e-4} if visc == "weiler" else None
    run_stage_sequence(g, o, seq, extra_state=tuple(names[2:]), tol=tol)
