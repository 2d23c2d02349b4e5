"""The tile kernels over the launch shapes they accept and the grids they meet:
one to three quads per thread, tiles smaller and larger than the grid, odd and
even rows and columns, not square.  FP64 against the oracle's fast cycle, FP32
refinement against the one-launch-per-half-sweep kernels, bit for bit."""
import dataclasses

import numpy as np
import pytest

import oracle
from qdeqcycle_fdm_amd import config, lib

pytestmark = pytest.mark.gpu

PROD = dict(cycle=config.CYCLE_FAST, n_pre=1, n_post=3, n_coarse=0, relax=1.15)

# (tile x, tile y, thread rows): few quads, one per thread, two per thread,
# the rows raised to hold the tile, tiles taller and wider than the grids
SHAPES = [(2, 2, 4), (32, 34, 8), (32, 34, 4), (50, 50, 4), (6, 200, 16), (200, 6, 4)]


def _problem(ni, nk, levels):
    pb = config.make_reference_problem(ni, nk, 24000.0 / (ni - 1))
    return dataclasses.replace(pb, params=dataclasses.replace(pb.params, n_levels=levels))


def _perturbed(pb, seed):
    rng = np.random.default_rng(seed)
    U = pb.U0.copy()
    U[1:-1, 2:-2] += rng.normal(scale=0.5, size=(pb.params.nk, pb.params.ni - 2))
    return U


def _solve(pb, me, U, shape=None, **kw):
    with lib.Engine(pb, me, **{**PROD, "tol": 1e-300, "max_vcycles": 2, **kw}) as eng:
        if shape is None:
            eng.set_tiles(False)
        elif shape != "default":
            n = len(eng.tile_shapes())
            eng.set_tile_shapes([(shape, shape)] * n)
        V = U.copy()
        with pytest.raises(lib.QdeqError) as e:
            eng.ode_solve(V)
        assert e.value.status == lib.QDEQ_ERR_MG_NOT_CONVERGED
    return V


GRIDS = [(129, 129, 3), (130, 97, 3), (66, 131, 3), (129, 67, 3), (64, 64, 2), (63, 65, 2)]


@pytest.mark.parametrize("ni,nk,levels", GRIDS)
@pytest.mark.parametrize("n_pre,n_post", [(1, 3), (2, 2), (0, 1)])
def test_fp64_tiles_equal_oracle(ni, nk, levels, n_pre, n_post):
    pb = _problem(ni, nk, levels)
    me = oracle.mu_equi(pb.mu)
    U = _perturbed(pb, 21)
    p = pb.params
    mg = oracle.MG(ni, nk, p.dh, levels, me, relax=PROD["relax"])
    mg.set_cycle(n_pre, n_post, 0, True)
    ref = U.copy()
    mg.solve(ref, oracle.ORC_TOL_ABS, 1e-300, 2)
    for shape in SHAPES:
        got = _solve(pb, me, U, shape, n_pre=n_pre, n_post=n_post)
        np.testing.assert_array_equal(got, ref, err_msg=str(shape))


@pytest.mark.parametrize("ni,nk,levels", GRIDS)
def test_fp32_tiles_equal_untiled(ni, nk, levels):
    pb = _problem(ni, nk, levels)
    me = oracle.mu_equi(pb.mu)
    U = _perturbed(pb, 22)
    ref = _solve(pb, me, U, precision=config.PREC_FP32_IR)
    for shape in SHAPES + [(66, 66, 4), (250, 16, 4)]:  # three quads per thread
        got = _solve(pb, me, U, shape, precision=config.PREC_FP32_IR)
        np.testing.assert_array_equal(got, ref, err_msg=str(shape))


@pytest.mark.parametrize("ni,nk,levels", [(65, 65, 4), (130, 97, 3), (801, 481, 6), (1030, 67, 5),
                                          (67, 1030, 5)])
@pytest.mark.parametrize("precision", [config.PREC_FP64, config.PREC_FP32_IR])
def test_default_shapes_equal_untiled(ni, nk, levels, precision):
    pb = _problem(ni, nk, levels)
    me = oracle.mu_equi(pb.mu)
    U = _perturbed(pb, 23)
    ref = _solve(pb, me, U, precision=precision)
    got = _solve(pb, me, U, "default", precision=precision)
    np.testing.assert_array_equal(got, ref)


@pytest.mark.parametrize("ni,nk,levels", [(129, 129, 3), (130, 97, 3), (66, 131, 2), (41, 57, 1),
                                          (257, 65, 4), (100, 101, 2)])
@pytest.mark.parametrize("sweeps", [(32, 32, 32), (5, 8, 3), (0, 1, 1)])
def test_reference_cycle_on_tiles_equals_oracle(ni, nk, levels, sweeps):
    """The reference's V-cycle in passes of several sweeps: levels in tiles
    with a halo, whole levels in one tile, with and without the tail, odd and
    even numbers of passes."""
    pb = _problem(ni, nk, levels)
    me = oracle.mu_equi(pb.mu)
    U = _perturbed(pb, 23)
    p = pb.params
    mg = oracle.MG(ni, nk, p.dh, levels, me)
    mg.set_cycle(*sweeps, False)
    ref = U.copy()
    mg.solve(ref, oracle.ORC_TOL_ABS, 1e-300, 2)
    with lib.Engine(pb, me, tol=1e-300, max_vcycles=2, n_pre=sweeps[0], n_post=sweeps[1],
                    n_coarse=sweeps[2]) as eng:
        V = U.copy()
        with pytest.raises(lib.QdeqError) as e:
            eng.ode_solve(V)
        assert e.value.status == lib.QDEQ_ERR_MG_NOT_CONVERGED
    np.testing.assert_array_equal(V, ref)


@pytest.mark.parametrize("n,levels,cap", [(129, 4, 2), (257, 5, 3)])
def test_run_after_a_solve_that_fails_behind_a_queued_stage(n, levels, cap):
    """A stage solve that ends at the V-cycle cap, with the next stage queued
    behind it and its stop test handed to that stage's fault update, reports
    the cap; set up again, the context steps as a fresh one does."""
    pb = config.make_bp1_problem(n, basin=True, levels=levels, tol_mode=config.TOL_REL,
                                 tol=1e-10)
    me = oracle.mu_equi(pb.mu)
    kw = {**PROD, "ini_dt": 1e5, "max_vcycles": cap}
    runs = []
    for tries in (1, 3):
        with lib.Engine(pb, me, **kw) as eng:
            for _ in range(tries):
                eng.rk43_setup()
                with pytest.raises(lib.QdeqError) as e:
                    eng.rk43_step(60)
                assert e.value.status == lib.QDEQ_ERR_MG_NOT_CONVERGED
                st = eng.state()
            runs.append(st)
    a, b = runs
    for key in ("t", "vcycles", "solves"):
        assert a["info"][key] == b["info"][key], key
    np.testing.assert_array_equal(a["U"], b["U"])


@pytest.mark.parametrize("precision", [config.PREC_FP64, config.PREC_FP32_IR])
def test_untiled_solve_after_a_failed_run(precision):
    """The stop test that a failed run leaves due belongs to the tiles it ran
    on, also when the next solve runs without tiles."""
    pb = config.make_bp1_problem(129, basin=True, levels=4, tol_mode=config.TOL_REL, tol=1e-10)
    me = oracle.mu_equi(pb.mu)
    U = _perturbed(pb, 24)
    kw = {**PROD, "ini_dt": 1e5, "max_vcycles": 2, "precision": precision}
    ends = []
    for fail in (True, False):
        with lib.Engine(pb, me, **kw) as eng:
            if fail:
                eng.rk43_setup()
                with pytest.raises(lib.QdeqError):
                    eng.rk43_step(60)
            eng.set_tiles(False)
            V = U.copy()
            with pytest.raises(lib.QdeqError) as e:
                eng.ode_solve(V)
            assert e.value.status == lib.QDEQ_ERR_MG_NOT_CONVERGED
            ends.append(V)
    np.testing.assert_array_equal(ends[0], ends[1])


@pytest.mark.parametrize("ni,nk,levels", [(129, 129, 3), (130, 97, 3), (66, 131, 2), (41, 57, 1),
                                          (257, 65, 4), (100, 101, 2)])
@pytest.mark.parametrize("sweeps", [(20, 21, 32), (5, 8, 3), (0, 1, 1)])
def test_reference_cycle_fp32_on_tiles_equals_untiled(ni, nk, levels, sweeps):
    """The same passes for the FP32 correction of refinement (a first pass from
    zero, the last one added into the FP64 displacement), bit for bit against
    one launch per half-sweep."""
    pb = _problem(ni, nk, levels)
    me = oracle.mu_equi(pb.mu)
    U = _perturbed(pb, 25)
    kw = dict(cycle=config.CYCLE_REFERENCE, n_pre=sweeps[0], n_post=sweeps[1],
              n_coarse=sweeps[2], precision=config.PREC_FP32_IR)
    ends = []
    for tiled in (True, False):
        with lib.Engine(pb, me, tol=1e-300, max_vcycles=2, **kw) as eng:
            if not tiled:
                eng.set_tiles(False, 8, 2)
            V = U.copy()
            with pytest.raises(lib.QdeqError) as e:
                eng.ode_solve(V)
            assert e.value.status == lib.QDEQ_ERR_MG_NOT_CONVERGED
            ends.append(V)
    assert not np.array_equal(ends[0], U)
    np.testing.assert_array_equal(ends[0], ends[1])


# default, then each device-side decision switched off
SWITCHES = [{}, {"QDEQ_SPECULATE": "0"}, {"QDEQ_FOLD_STOP": "0"}, {"QDEQ_HOST_START": "1"},
            {"QDEQ_GRAPH_LAUNCH": "1"}]


@pytest.mark.parametrize("n,levels,sweeps", [(65, 3, (32, 32, 32)), (129, 4, (5, 8, 3))])
@pytest.mark.parametrize("precision,start", [(config.PREC_FP64, "plain"),
                                             (config.PREC_FP32_IR, "plain"),
                                             (config.PREC_FP64, "projection"),
                                             (config.PREC_FP32_IR, "projection"),
                                             (config.PREC_FP64, "learned"),
                                             (config.PREC_FP32_IR, "learned")])
def test_reference_cycle_runs_equal_without_device_decisions(n, levels, sweeps, precision, start,
                                                             monkeypatch):
    """RK43 steps on the reference's cycle, with each kind of start: bit for bit
    the same with stages launched ahead or not, stop tests in the kernel behind
    or on their own, starts chosen on the device or by the host, and as graphs."""
    pb = config.make_bp1_problem(n, basin=True, levels=levels, tol_mode=config.TOL_REL, tol=1e-10)
    me = oracle.mu_equi(pb.mu)
    names = {k for s in SWITCHES for k in s}
    g = None
    if start == "learned":  # zero weights: the previous solution and the remote edge's change
        g = lib.Guess(n, hidden=128, capacity=1)
        g.set_params(np.zeros(g.num_params, np.float32))
    runs = []
    for switch in SWITCHES:
        for k in names:
            monkeypatch.delenv(k, raising=False)
        for k, v in switch.items():
            monkeypatch.setenv(k, v)
        with lib.Engine(pb, me, precision=precision, n_pre=sweeps[0], n_post=sweeps[1],
                        n_coarse=sweeps[2], max_vcycles=200) as eng:
            eng.rk43_setup()
            if start == "projection":
                eng.projection_enable(6)
            if g is not None:
                eng.attach_guess(g, lib.GUESS_PREDICT)
            eng.rk43_step(25)
            eng.rk43_step(1)
            eng.rk43_step(15)
            runs.append((eng.state(), eng.launch_ahead_stats()["taken"], eng.folded_stop_tests(),
                         eng.projection_stats(), eng.guess_stats() if g is not None else None))
            if g is not None:
                eng.attach_guess(None, lib.GUESS_OFF)
    a, ahead, folded, proj, learned = runs[0]
    for switch, (b, b_ahead, b_folded, b_proj, b_learned) in zip(SWITCHES[1:], runs[1:]):
        for key in ("t", "dt", "vcycles", "solves", "attempts"):
            assert a["info"][key] == b["info"][key], (switch, key)
        for k in ("slip", "psi", "V", "U"):
            assert np.all(np.isfinite(b[k])), (switch, k)
            np.testing.assert_array_equal(a[k], b[k], err_msg=str((switch, k)))
        assert b_proj == proj and b_learned == learned, switch
        if "QDEQ_SPECULATE" in switch:
            assert b_ahead == 0
        if "QDEQ_FOLD_STOP" in switch:
            assert b_folded == 0
    # (a candidate start of FP32 refinement waits for the host)
    on_device = start == "plain" or (start == "projection" and precision == config.PREC_FP64)
    assert (ahead > 0) == on_device
    assert (folded > 0) == on_device
    if start == "projection":
        assert proj["used"] > 0
    if g is not None:
        assert learned["predicted"] > 0
        g.close()


@pytest.mark.parametrize("ni,nk,levels", [(129, 129, 3), (129, 1601, 7)])
def test_level0_up_tiles_taller_than_a_workgroup_holds(ni, nk, levels):
    """Without post-smoothing the shape checks accept up tiles of two or four
    columns and more rows than the quads of one workgroup: they run, cut, and
    are reported as they were given."""
    pb = _problem(ni, nk, levels)
    me = oracle.mu_equi(pb.mu)
    U = _perturbed(pb, 26)
    p = pb.params
    mg = oracle.MG(ni, nk, p.dh, levels, me, relax=PROD["relax"])
    mg.set_cycle(1, 0, 0, True)
    ref = U.copy()
    mg.solve(ref, oracle.ORC_TOL_ABS, 1e-300, 2)
    for up in [(2, 1360, 4), (2, 1362, 16), (2, 1600, 16), (4, 1020, 16), (4, 1060, 1)]:
        with lib.Engine(pb, me, **{**PROD, "n_post": 0, "tol": 1e-300, "max_vcycles": 2}) as eng:
            shapes = eng.tile_shapes()
            shapes[0] = (shapes[0][0], up)
            eng.set_tile_shapes(shapes)
            assert tuple(eng.tile_shapes()[0][1]) == up
            V = U.copy()
            with pytest.raises(lib.QdeqError) as e:
                eng.ode_solve(V)
            assert e.value.status == lib.QDEQ_ERR_MG_NOT_CONVERGED
        np.testing.assert_array_equal(V, ref, err_msg=str(up))
