"""Whole-substep HIP graph replay against eager launches.

Every kernel of the substep is deterministic (integer atomics and max
reductions only), so a replayed graph must give bit-identical states and
statistics.  The graph is replayed several times with eager work and host
synchronisations in between, and every replay is compared."""
import ctypes as C

import numpy as np
import pytest

from gpu_common import Scene, block_scene

pytestmark = pytest.mark.gpu

sa = pytest.importorskip("sphpc_amd")


def _pair(tol, iters=4):
    s = 0.02
    sc = Scene(s, (2.0, 1.0, 1.0), iters=iters, tol=tol, k=0.5, c=0.01, vort_eps=0.01,
               vort_model=1, lambda_eps=600.0)
    pos, vel = block_scene((24, 20, 22), s, (0.1, 0.05, 0.1), jitter=0.01, seed=3,
                           vel_sigma=0.1, swirl=0.3)
    ctxs = []
    for graph in (False, True):
        c = sc.context(len(pos))
        dims, wmin, wmax = (32, 32, 32), (0.5, 0.0, 0.0), (1.3, 0.8, 0.8)
        ax = [wmin[i] + (np.arange(32) + 0.5) * 0.025 for i in range(3)]
        Z, Y, X = np.meshgrid(ax[2], ax[1], ax[0], indexing="ij")
        sdf = (np.sqrt((X - 0.9) ** 2 + (Y - 0.3) ** 2 + (Z - 0.2) ** 2) - 0.15).astype(np.float32)
        c.set_obstacle(sdf.ravel(), dims, 0.025, wmin, wmax)
        c.upload(pos, vel)
        c.set_graph(graph)
        ctxs.append(c)
    return sc, ctxs


def _same(a, b, step):
    pa, va = a.download()
    pb, vb = b.download()
    assert np.array_equal(pa, pb), step
    assert np.array_equal(va, vb), step
    sa_, sb = a.stats(), b.stats()
    assert sa_.iterations == sb.iterations, step
    assert sa_.converged == sb.converged, step
    assert sa_.max_density_error == sb.max_density_error, step
    assert sa_.neighbor_pairs == sb.neighbor_pairs, step
    assert sa_.substeps == sb.substeps, step


@pytest.mark.parametrize("tol", [0.0, 1e-3])
def test_graph_replay_bit_identical(tol):
    sc, (eager, graph) = _pair(tol)
    for step in range(6):
        eager.step(1)
        graph.step(1)
        graph.synchronize()
        _same(eager, graph, step)
        # eager work on the graph context between replays (FP64 block sums
        # are added atomically in any order: equal to rounding)
        ke_g, ke_e = graph.kinetic_energy(), eager.kinetic_energy()
        assert abs(ke_g - ke_e) <= 1e-12 * max(abs(ke_e), 1e-300)
    # a parameter change rebuilds the graph
    p = sc.gpu_params()
    p.solve_iterations = 6
    for c in (eager, graph):
        c.set_params(p)
    eager.step(3)
    graph.step(3)
    _same(eager, graph, "after set_params")


def test_graph_replay_with_warm_start():
    sc, (eager, graph) = _pair(1e-3, iters=10)
    net = sa.Mlp(seed=4)
    mean = np.array([1.0, 0.0, 0.01, 0.9, 0.0, 4.0, 0, 0, 0, 0, 0, 0], np.float32)
    std = np.array([0.3, 0.01, 0.01, 0.05, 0.01, 1.0, 1, 1, 1, 0.1, 0.1, 0.1], np.float32)
    net.set_normalization(mean, std, 0.005, 0.01)
    for c in (eager, graph):
        c.set_warm_start(net)
    for step in range(5):
        eager.step(1)
        graph.step(1)
        _same(eager, graph, step)
        assert np.array_equal(eager.field(sa.FIELD_LAMBDA_SUM), graph.field(sa.FIELD_LAMBDA_SUM))


def test_autotune_keeps_state_and_results():
    """The tuner restores the state it started from, and substeps with the
    tuned launch geometry are bit-identical to the default geometry."""
    sc, (ref, tuned) = _pair(1e-3)
    p0, v0 = tuned.download()
    t = tuned.autotune(2)
    p1, v1 = tuned.download()
    assert np.array_equal(p0, p1) and np.array_equal(v0, v1)
    assert all(b in (64, 128, 256) for b in t["block"].values())
    assert all(d in (8, 16, 32) for d in t["depth"].values())
    assert t["ms_per_substep_tuned"] > 0
    for step in range(3):
        ref.step(1)
        tuned.step(1)
        _same(ref, tuned, step)


def test_list_format_does_not_change_results():
    """Compact and wide neighbour lists give bit-identical substeps (same
    neighbours in the same order), eager and graph-replayed."""
    sc, (compact, wide) = _pair(1e-3)
    wide.set_tuning(wide_lists=True)
    assert wide.tuning()["wide_lists"] and not compact.tuning()["wide_lists"]
    for step in range(4):
        compact.step(1)
        wide.step(1)
        _same(compact, wide, step)
    ia, ca = compact.neighbors()
    ib, cb = wide.neighbors()
    assert np.array_equal(ca, cb) and np.array_equal(ia, ib)


def test_set_tuning_validates_and_round_trips():
    sc, (a, b) = _pair(0.0)
    a.set_tuning(block={"density_lambda": 64, "xsph": 128}, depth={"dp_update": 32},
                 split_collide=False, wide_lists=True)
    t = a.tuning()
    assert t["block"]["density_lambda"] == 64 and t["block"]["xsph"] == 128
    assert t["depth"]["dp_update"] == 32 and t["depth"]["density_lambda"] == 16
    assert t["wide_lists"] and not t["split_collide"]
    with pytest.raises(sa.SphError):
        a.set_tuning(block={"color": 96})
    with pytest.raises(sa.SphError):
        a.set_tuning(depth={"color": 12})
    for step in range(3):
        a.step(1)
        b.step(1)
        _same(a, b, step)


@pytest.mark.parametrize("depth,block,wide", [(8, 64, False), (32, 128, False), (8, 128, True),
                                              (32, 64, True)])
def test_launch_choices_do_not_change_results(depth, block, wide):
    """Every gather kernel at another depth (its own template instance) and
    block size, compact or wide lists: bit-identical to the defaults."""
    sc, (ref, other) = _pair(1e-3)
    names = [k for k in sa.kernel_names()
             if k in ("build_lists", "density_lambda", "dp_update", "color", "surface", "xsph",
                      "vorticity", "confine")]
    other.set_tuning(block={k: block for k in names}, depth={k: depth for k in names},
                     wide_lists=wide, split_collide=False)
    for step in range(3):
        ref.step(1)
        other.step(1)
        _same(ref, other, step)


@pytest.mark.parametrize("n,squeeze,wide,calls", [
    (1, 1.0, False, "fused"), (17, 1.0, False, "staged"), (1000, 0.85, False, "fused"),
    (1003, 0.85, True, "fused"), (4099, 0.85, True, "staged"), (32768, 1.0, False, "fused"),
    (32769, 1.0, False, "fused")])
def test_four_lanes_a_particle_equal_one(n, squeeze, wide, calls):
    """The gather kernels that small scenes take (four lanes a particle) give the
    bits of those with one lane, which an explicit depth asks for: both sides of
    the limit, part-filled waves, lists past 32 entries (lattice spacing times
    ``squeeze``), both list formats, the fused and the staged calls."""
    s, side = 0.02, int(np.ceil(np.cbrt(n) - 1e-9))
    sc = Scene(s, (2.0, 1.0, 1.0), iters=4, tol=1e-3 if calls == "fused" else 0.0, k=0.5, c=0.01,
               vort_eps=0.01, vort_model=1, lambda_eps=600.0)
    pos, vel = block_scene((side, side, side), s * squeeze, (0.1, 0.05, 0.1), jitter=0.05, seed=5,
                           vel_sigma=0.1, swirl=0.3)
    pos, vel = pos[:n], vel[:n]
    names = ("density_lambda", "density", "lambda", "dp", "dp_update", "color", "surface", "xsph",
             "vorticity", "confine")
    four, one = sc.context(n), sc.context(n)
    four.set_tuning(wide_lists=wide)
    one.set_tuning(depth={k: 16 for k in names}, wide_lists=wide)
    for c in (four, one):
        c.upload(pos, vel)
    for step in range(2):
        for c in (four, one):
            if calls == "fused":
                c.step(1)
                continue
            c.apply_gravity()
            c.predict_positions()
            c.find_all_neighbors()
            for it in range(3):
                c.compute_densities()
                c.compute_lambda()
                c.update_dps(it)
                c.update_position_stars()
            c.update_velocities()
            c.compute_surface_tension()
            c.apply_viscosity()
            c.compute_vorticity()
            c.apply_vorticity_confinement()
            c.update_positions()
        if squeeze < 1.0 and step == 0:  # the solver spreads them
            assert four.neighbors()[1].max() > 32
        _same(four, one, step)


@pytest.mark.parametrize("iters", [0, 1, 4])
@pytest.mark.parametrize("tol", [0.0, 1e-3, 10.0])
@pytest.mark.parametrize("depth", [0, 16])
def test_update_that_ends_the_substep_equals_separate_passes(iters, tol, depth):
    """Without velocity terms the last position update also makes the velocities
    and the results by id; with the obstacle push as its own pass (split) those are
    separate kernels.  Same bits, also where the loop ends within tolerance at once
    (10), in the middle or never, and without iterations."""
    sc, ctxs = _pair(tol, iters)
    p = sc.gpu_params()
    p.surface_tension = p.viscosity = p.vorticity = 0
    for c, split in zip(ctxs, (True, False)):
        c.set_params(p)
        c.set_tuning(split_collide=split, depth={"dp_update": depth})
    for step in range(3):
        for c in ctxs:
            c.step(1)
        _same(*ctxs, step)
        # no iteration, no density pass: the field holds nothing
        for f in (sa.FIELD_VELOCITY,) + ((sa.FIELD_DENSITY,) if iters else ()):
            assert np.array_equal(ctxs[0].field(f), ctxs[1].field(f)), (step, f)


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("passes,iters", [(6, 8), (130, 2)])
def test_density_stage_after_substeps_of_fewer_iterations(graph, passes, iters):
    """A density stage reports its own pass's maximum also where its slot (they go on
    counting over fused substeps, up to 128) holds an older and larger one: of a
    substep of more iterations than the later ones, or of earlier stages."""
    s = 0.02
    sc = Scene(s, (1.0, 1.0, 1.0), iters=iters, lambda_eps=600.0)
    dense, _ = block_scene((12, 12, 12), 0.8 * s, (0.1, 0.1, 0.1), jitter=0.01, seed=2)
    loose, _ = block_scene((12, 12, 12), 1.3 * s, (0.1, 0.1, 0.1), jitter=0.01, seed=2)
    with sc.context(len(dense)) as c:
        c.set_graph(graph)
        c.upload(dense)
        c.predict_positions()
        c.find_all_neighbors()
        for _ in range(passes):
            c.compute_densities()
        assert c.stats().max_density_error > 0.1
        c.step(3)
        c.upload(loose)
        p = sc.gpu_params()
        p.solve_iterations = 2
        c.set_params(p)
        c.step(3)
        for _ in range(2):
            c.compute_densities()
            assert c.stats().max_density_error == 0.0
            assert np.max(c.field(sa.FIELD_DENSITY)) < 1000.0
        c.step(1)
        assert c.stats().max_density_error == c.residuals()[-1]


GATHERS = ("density_lambda", "density", "lambda", "dp", "dp_update", "color", "surface", "xsph",
           "vorticity", "confine")


def _raw(ctx):
    t = sa.Tuning()
    sa.check(sa.lib().sph_get_tuning(ctx.handle, C.byref(t)))
    return t


def test_tuning_as_read_changes_nothing():
    """Kernels by rule stay by rule through a read and a write, through one that names
    another field or kernel, and in another context; naming a kernel takes it out (what
    is not named of it is 256 or 16), zeros put it back."""
    sc, (a, b) = _pair(0.0)
    rule = a.tuning()["by_rule"]
    assert set(GATHERS) <= set(rule) and "predict_hash" not in rule
    sa.check(sa.lib().sph_set_tuning(a.handle, C.byref(_raw(a))))
    assert a.tuning() == b.tuning()
    a.set_tuning(wide_lists=True, split_collide=True)
    assert a.tuning()["by_rule"] == rule
    a.set_tuning(block={"xsph": 64}, depth={"color": 8, "surface": 16})
    t = a.tuning()
    assert t["by_rule"] == [k for k in rule if k not in ("xsph", "color", "surface")]
    assert (t["block"]["xsph"], t["depth"]["xsph"]) == (64, 16)
    assert (t["block"]["color"], t["depth"]["color"]) == (256, 8)
    sa.check(sa.lib().sph_set_tuning(b.handle, C.byref(_raw(a))))
    assert b.tuning() == t
    a.set_tuning(block={"xsph": 0, "color": 0}, depth={"xsph": 0, "color": 0})
    assert a.tuning()["by_rule"] == [k for k in rule if k != "surface"]
    sa.check(sa.lib().sph_set_tuning(a.handle, C.byref(sa.Tuning())))
    assert a.tuning()["by_rule"] == rule
    a.autotune(1)
    sa.check(sa.lib().sph_set_tuning(b.handle, C.byref(_raw(a))))
    assert b.tuning() == a.tuning()
    for step in range(2):
        a.upload(*b.download())
        a.step(1)
        b.step(1)
        pa, va = a.download()
        pb, vb = b.download()
        assert np.array_equal(pa, pb) and np.array_equal(va, vb), step


@pytest.mark.parametrize("n,squeeze,wide,calls", [
    (1, 1.0, True, "staged"), (3, 1.0, False, "fused"), (15, 1.0, True, "fused"),
    (16, 1.0, False, "staged"), (65, 1.0, True, "staged"), (4099, 0.85, False, "staged"),
    (4099, 0.85, True, "fused"), (32768, 0.85, True, "fused")])
def test_four_lanes_by_rule_equal_one(n, squeeze, wide, calls):
    """More shapes of the comparison above, where the context of the default rule is known
    to be by rule also after the list format was chosen (one lane from 32,769 particles
    and for the kernels of the other context)."""
    with Scene(0.02, (1.0, 1.0, 1.0)).context(n) as c:
        c.set_tuning(wide_lists=wide)
        assert set(GATHERS) <= set(c.tuning()["by_rule"])
        c.set_tuning(depth={k: 16 for k in GATHERS})
        assert not set(GATHERS) & set(c.tuning()["by_rule"])
    test_four_lanes_a_particle_equal_one(n, squeeze, wide, calls)


@pytest.mark.parametrize("n", [1, 200, 4000])
def test_autotuner_keeps_nothing_slower_than_it_found(n):
    """The set it reports took no longer than the context's own launches, which stay if
    nothing was faster (small scenes, where times differ by chance alone), also where
    they were chosen before; kernels that did not run stay as they were."""
    sc = Scene(0.02, (1.0, 1.0, 1.0), iters=2, lambda_eps=600.0)
    side = int(np.ceil(np.cbrt(n) - 1e-9))
    pos = block_scene((side,) * 3, 0.02, (0.1, 0.1, 0.1))[0][:n]
    for chosen in ({}, {"dp_update": 8, "color": 32}):
        with sc.context(n) as c:
            c.upload(pos)
            for _ in range(3):
                c.set_tuning(depth=chosen)
                was = c.tuning()
                t = c.autotune(1)
                assert t["ms_per_substep_tuned"] <= t["ms_per_substep_default"]
                for k in ("color", "xsph", "dp"):
                    assert (t["block"][k], t["depth"][k]) == (was["block"][k], was["depth"][k])
                    assert (k in t["by_rule"]) == (k in was["by_rule"])
                if t["ms_per_substep_tuned"] == t["ms_per_substep_default"]:
                    for k in ("block", "depth", "by_rule", "split_collide", "wide_lists"):
                        assert t[k] == was[k]


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("block", [64, 128])
def test_list_build_does_not_depend_on_its_threads(block, wide):
    """Above 196,608 particles the list build takes the threads per block that are asked
    for; the lists are those of 256."""
    sc = Scene(0.02, (2.0, 2.0, 2.0))
    pos, vel = block_scene((59, 59, 59), 0.02 * 0.8, (0.0, 0.0, 0.0), jitter=0.05, seed=6)
    lists = []
    for b in (0, block):
        with sc.context(len(pos)) as c:
            c.set_tuning(block={"build_lists": b}, wide_lists=wide)
            c.upload(pos, vel)
            c.predict_positions()
            c.find_all_neighbors()
            lists.append(c.neighbors() + (c.stats().neighbor_pairs, c.stats().neighbor_overflow))
    (ids, cnt, pairs, lost), (ids2, cnt2, pairs2, lost2) = lists
    assert np.array_equal(cnt, cnt2) and (pairs, lost) == (pairs2, lost2) and pairs == cnt.sum()
    used = np.arange(sa.MAX_NEIGHBORS)[None, :] < cnt[:, None]
    shape = (len(pos), sa.MAX_NEIGHBORS)
    assert np.array_equal(ids.reshape(shape)[used], ids2.reshape(shape)[used])
