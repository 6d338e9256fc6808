"""Learned warm start on the device: sample recording, the residual-picked
first iteration, convergence to the configured tolerance, and the gain of a
network trained on the solver's own states over the reference's start."""
import numpy as np
import pytest

from splishsplash_amd import capi, learned, scenes

pytestmark = pytest.mark.gpu


def small_variant(seed, per_side=24, **kw):
    return scenes.dam_break_variant(seed, per_side=per_side, n_spheres=kw.pop("n_spheres", 0), **kw)


def test_sample_recording_counts_and_ranges():
    sc = small_variant(1)
    n = len(sc["x"])
    stride = 5
    sim = learned.make_sim(sc)
    # past the start, where the lattice (rho = 0.8 rho0) is under-dense and
    # no stiffness is stored yet
    sim.step(60)
    assert sim.get("p / rho^2").max() > 0
    sim.collect_training("pressure", stride, 1 << 20)
    sim.collect_training("divergence", stride, 1 << 20)
    sim.step(6)
    for s in learned.SOLVERS:
        x, t = sim.get_training(s)
        # one sample per stride-th particle and step (the offset rotates)
        assert 6 * (n // stride) <= len(x) <= 6 * (n // stride + 1), (s, len(x))
        assert np.isfinite(x).all() and np.isfinite(t).all()
        assert (t >= 0).all()
        assert ((x[:, 2] >= 0) & (x[:, 2] <= 1)).all()  # previous stiffness / step maximum
        assert (x[:, 6:] == 0).all()
        assert (x[:, 5] > 0).all()  # neighbour count / 40
    # the record is cleared by reading it, and capacity bounds it
    x, _ = sim.get_training("pressure")
    assert len(x) == 0
    sim.collect_training("pressure", 1, 100)
    sim.step(1)
    x, _ = sim.get_training("pressure")
    assert len(x) == 100


def test_untrained_network_still_converges():
    # Any prediction only changes the start: the solve must reach the same
    # tolerance on remaining compression and on overshoot, so even a random
    # network leaves the motion as it was (particles whose predicted start
    # is worse keep the reference's start).
    sc = small_variant(2)
    eta = sc["params"].max_error * 0.01 * sc["params"].density0
    th = {s: learned.init_theta(7) for s in learned.SOLVERS}
    sim = learned.make_sim(sc, th)
    for s in learned.SOLVERS:
        sim.set_warm_start_policy(s, 0)  # use the network in every solve
    ref = learned.make_sim(sc)
    for _ in range(40):
        sim.step(1)
        ref.step(1)
        c = sim.counters()
        assert (c["avg_density_err"] <= eta and c["avg_overpressure_err"] <= eta) or c["iterations"] == 100
    assert c["flags"] == 0
    assert np.isfinite(sim.get("position")).all()
    # same physics within the solver tolerance: mean height of the fluid
    yl, yr = sim.get("position")[:, 1].mean(), ref.get("position")[:, 1].mean()
    assert abs(yl - yr) < 0.01 * yr


@pytest.mark.parametrize("lanes", [1, 2, 4])
def test_zero_network_equals_plain_start(lanes):
    # At the first step every stored stiffness is 0, so the reference's start
    # and the prediction are both 0 and the first iteration keeps the
    # reference's start: the learned path must reproduce the plain one bit
    # for bit (same kernels' arithmetic, same iteration count), also with the
    # neighbour sums split over 2 or 4 lanes per particle.
    sc = small_variant(3)
    th0 = {s: np.zeros(capi.MLP_NPARAM, np.float32) for s in learned.SOLVERS}
    a = learned.make_sim(sc, th0)
    for s in learned.SOLVERS:
        a.set_warm_start_policy(s, 0)
    b = learned.make_sim(sc)
    a.set_lanes_per_particle(lanes)
    b.set_lanes_per_particle(lanes)
    a.step(1)
    b.step(1)
    assert a.counters()["learned_solves"] == 1
    for nm in ("position", "velocity", "p / rho^2"):
        np.testing.assert_array_equal(a.get(nm), b.get(nm))
    assert a.counters()["iterations"] == b.counters()["iterations"]


def test_trained_network_cuts_pressure_iterations():
    # Train on the solver states of three seeded variants, evaluate on a
    # held-out one: fewer pressure iterations at the same tolerance.
    data = [learned.collect(small_variant(s, per_side=28), steps=80, skip=30, stride=3) for s in (11, 12, 13)]
    th, loss = learned.train(learned.merge(data), steps=1500, batch=8192, lr=2e-3)
    assert all(np.isfinite(v) for v in loss.values())
    sc = small_variant(21, per_side=32)
    plain = learned.evaluate(sc, None, steps=60, warmup=30)
    lrn = learned.evaluate(sc, th, steps=60, warmup=30)
    eta = sc["params"].max_error * 0.01 * sc["params"].density0
    assert lrn["avg_density_err"] <= eta and lrn["flags"] == 0
    assert lrn["pressure_iterations"] < 0.9 * plain["pressure_iterations"], (plain, lrn)


def test_engagement_policy():
    # With the default policy the network is used only after a solve that
    # needed at least 4 (pressure) / 3 (divergence) iterations; a threshold
    # above the iteration cap never engages it.
    sc = small_variant(4)
    th = learned.load()
    a = learned.make_sim(sc, th)
    a.set_warm_start_policy("pressure", 1000)
    a.set_warm_start_policy("divergence", 1000)
    a.step(30)
    c = a.counters()
    assert c["learned_solves"] == 0 and c["learned_solves_v"] == 0
    b = learned.make_sim(sc, th)
    b.set_warm_start_policy("pressure", 0)
    b.step(30)
    assert b.counters()["learned_solves"] == 30


@pytest.mark.parametrize("lanes", [2, 4])
def test_learned_start_with_split_neighbour_sums(lanes):
    # The learned start followed by solver sweeps with 2 or 4 lanes per
    # particle: every solve reaches the tolerance, the network is used in
    # every solve, and the motion and iteration totals stay those of one
    # lane per particle.
    sc = small_variant(5)
    eta = sc["params"].max_error * 0.01 * sc["params"].density0
    th = learned.load()
    runs = {}
    for L in (1, lanes):
        sim = learned.make_sim(sc, th)
        sim.set_lanes_per_particle(L)
        for s in learned.SOLVERS:
            sim.set_warm_start_policy(s, 0)
        for _ in range(40):
            sim.step(1)
            c = sim.counters()
            assert (c["avg_density_err"] <= eta and c["avg_overpressure_err"] <= eta) or c["iterations"] == 100
        assert c["flags"] == 0 and c["learned_solves"] == 40 and c["lanes_per_particle"] == L
        runs[L] = (sim.get("position")[:, 1].mean(), c["total_iterations"])
    (y1, i1), (yl, il) = runs[1], runs[lanes]
    assert abs(yl - y1) < 0.005 * y1
    assert abs(il - i1) <= 0.1 * i1, runs


def test_packaged_networks_gain_on_heldout_variant():
    # The packaged networks (trained on 32 seeded variants) on a small
    # held-out variant: fewer pressure iterations, the tolerance met on both
    # sides, and the same motion as the reference's start.
    sc = scenes.dam_break_variant(4242, per_side=40, n_spheres=3)
    th = learned.load()
    eta = sc["params"].max_error * 0.01 * sc["params"].density0
    plain = learned.evaluate(sc, None, steps=80, warmup=80)
    lrn = learned.evaluate(sc, th, steps=80, warmup=80)
    assert lrn["flags"] == 0 and lrn["avg_density_err"] <= eta
    assert lrn["pressure_iterations"] < 0.8 * plain["pressure_iterations"], (plain, lrn)
    assert abs(lrn["sim_time"] - plain["sim_time"]) < 0.05 * plain["sim_time"]


def test_previous_stiffness_mode_converges_with_fewer_iterations():
    # Warm-start mode 1 (the previous step's full stiffness, no network):
    # same tolerance on both sides, fewer pressure iterations than the
    # reference's halved and clamped start, from identical states.
    sc = scenes.dam_break_variant(4243, per_side=40, n_spheres=2)
    r = learned.evaluate_snapshots(sc, {"plain": None, "previous": "previous"}, warmup=80, snapshots=8, every=5)
    assert r["previous"]["pressure_iterations"] < r["plain"]["pressure_iterations"], r
    eta = sc["params"].max_error * 0.01 * sc["params"].density0
    assert r["previous"]["avg_overpressure_err"] <= eta


@pytest.mark.parametrize("mode", ["threads", "graphs"])
def test_batch_first_steps_of_fresh_handles(mode):
    # Handles that have not tuned their lanes per particle take their first
    # step one at a time inside step_batch; the batch still advances every
    # scene by exactly the requested steps, as alone.
    scs = [scenes.ensemble_scene(s, nmin=5000, nmax=30000) for s in range(3)]
    alone = [learned.make_sim(sc) for sc in scs]
    batch = [learned.make_sim(sc) for sc in scs]
    for sim in alone:
        sim.step(4)
    capi.set_batch_mode(mode)
    try:
        capi.step_batch(batch, 4, threads=3)
    finally:
        capi.set_batch_mode("auto")
    for a, b in zip(alone, batch):
        np.testing.assert_array_equal(a.get("position"), b.get("position"))
        assert a.counters()["time"] == b.counters()["time"]
        assert a.counters()["total_iterations"] == b.counters()["total_iterations"]


@pytest.mark.parametrize("mode", ["batched", "graphs"])
def test_batch_follows_scenes_that_change_lanes(mode):
    # Up to 40,960 particles stepped together 16 lanes share a particle,
    # beyond one lane takes it: scenes that grow past that between two calls
    # on the same handles run at their new lanes. The FP64 error sums are
    # grouped by the blocks of a launch, so they too are those of the scene
    # alone only where the batch launches as many.
    sc = scenes.dam_break_variant(11, per_side=27, aspect=3.0, n_spheres=0)
    more = scenes.lattice_block((34, 27, 27), 0.05, (1.6, 0.1, 0.1))  # in the free part of the box
    alone, batch = learned.make_sim(sc), learned.make_sim(sc)
    capi.set_batch_mode(mode)
    try:
        for lanes in (16, 1):
            if lanes == 1:
                alone.emit_particles(more)
                batch.emit_particles(more)
            alone.step(3)
            capi.step_batch([batch], 3)
            assert alone.counters()["lanes_per_particle"] == batch.counters()["lanes_per_particle"] == lanes
            for f in ("position", "velocity", "p / rho^2"):
                np.testing.assert_array_equal(alone.get(f), batch.get(f), err_msg=f)
            ca, cb = alone.counters(), batch.counters()
            for c in ("total_iterations", "total_iterations_v", "avg_density_err", "avg_divergence_err", "time"):
                assert ca[c] == cb[c], c
    finally:
        capi.set_batch_mode("auto")


@pytest.mark.parametrize("mode", ["threads", "graphs"])
def test_batch_in_larger_company_keeps_the_fields(mode):
    # Each scene takes 16 lanes per particle alone; together they are more
    # than 40,960 particles and take one. Neighbour sums keep their order, so
    # fields and iteration counts stay (only FP64 totals are grouped
    # differently, in their last bits).
    scs = [scenes.dam_break_variant(20 + k, per_side=(26, 27, 28)[k], n_spheres=k) for k in range(3)]
    alone, batch = [learned.make_sim(sc) for sc in scs], [learned.make_sim(sc) for sc in scs]
    assert max(sim.n for sim in alone) <= 40960 < sum(sim.n for sim in alone)
    for sim in alone:
        sim.step(8)
    capi.set_batch_mode(mode)
    try:
        capi.step_batch(batch, 8)
    finally:
        capi.set_batch_mode("auto")
    for a, b in zip(alone, batch):
        ca, cb = a.counters(), b.counters()
        assert (ca["lanes_per_particle"], cb["lanes_per_particle"]) == (16, 1)
        for f in ("position", "velocity", "p / rho^2", "velocity difference"):
            np.testing.assert_array_equal(a.get(f), b.get(f), err_msg=f)
        assert ca["total_iterations"] == cb["total_iterations"]
        assert ca["total_iterations_v"] == cb["total_iterations_v"]
        assert ca["avg_density_err"] == pytest.approx(cb["avg_density_err"], rel=1e-12)


@pytest.mark.parametrize("mode", ["threads", "batched", "graphs", "auto"])
def test_batch_step_matches_scene_by_scene(mode):
    # Scenes stepped together give the same results as each stepped alone,
    # bit for bit: scene by scene on host threads, with the solves of all
    # scenes in batched launches, with those replayed from captured HIP
    # graphs (two lanes-per-particle groups; every step replays the graphs
    # of both solves, with the scenes' own work between the replays), and
    # in the default mode, whose first four steps alternate the two ways.
    scs = [scenes.ensemble_scene(s, nmin=5000, nmax=30000) for s in range(5)]
    alone = [learned.make_sim(sc) for sc in scs]
    batch = [learned.make_sim(sc) for sc in scs]
    for k, (a, b) in enumerate(zip(alone, batch)):
        lanes = 2 if k % 2 else 1
        a.set_lanes_per_particle(lanes)
        b.set_lanes_per_particle(lanes)
    for sim in alone:
        sim.step(6)
    capi.set_batch_mode(mode)
    try:
        capi.step_batch(batch, 3, threads=3)
        capi.step_batch(batch, 3, threads=3)  # a second call reuses the captured graphs
        if mode == "auto":
            assert capi.batch_choice() in ("threads", "graphs")
    finally:
        capi.set_batch_mode("auto")
    for a, b in zip(alone, batch):
        np.testing.assert_array_equal(a.get("position"), b.get("position"))
        np.testing.assert_array_equal(a.get("velocity"), b.get("velocity"))
        ca, cb = a.counters(), b.counters()
        assert ca["total_iterations"] == cb["total_iterations"]
        assert ca["total_iterations_v"] == cb["total_iterations_v"]
        assert ca["time"] == cb["time"]
    with pytest.raises(capi.SPHError):
        capi.step_batch([batch[0], batch[0]], 1)
