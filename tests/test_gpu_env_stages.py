"""The envelope route's joined stage kernels over their range of splits: T = n1 n2 with
n1 = n2 and n2 = 2 n1, from the smallest grid to sequences past the held twiddles, with
and without the Raman response (on the smallest windows it wraps round the whole grid),
the in-stage absorber's second row, the modified noise, a Raman rate that varies along z
and the commit at a trial's head. One trial against the oracle's, within 1e-12; a march's
attempts by graph and by direct launches, to the bit."""

import dataclasses

import numpy as np
import pytest
from test_gpu_rk import norm_bound, oracle_trial, rel_l2

from solprop_amd.native import Workspace
from solprop_amd.problem import ScalarPath, Tableau, gnlse_problem

pytestmark = pytest.mark.gpu

SIZES = [(16, 1), (16, 2), (64, 1), (64, 2), (256, 1), (512, 1), (512, 2), (2048, 1), (2048, 2),
         (4096, 2), (16384, 2), (65536, 2), (262144, 1), (2097152, 1)]


def problem_of(n_t, ffac, option):
    kw = dict(n_t=n_t, ffac=ffac, window=n_t * 4e-15, fwhm=50e-15, soliton_order=2.0,
              noise_seed=7, noise_model="input", length=0.02, time_collar=0.2)
    if option == "no_raman":
        kw["raman_fraction"] = 0.0
    elif option == "absorber_noise":
        kw.update(absorber="in_stage", absorber_length=2e-3, noise_model="modified")
    problem = gnlse_problem(**kw)
    if option == "varying_rate":
        rate = problem.raman.rates[0]
        path = ScalarPath.chebyshev(lambda z: rate.value * (1.0 + 10.0 * z), 0.0, 0.02)
        problem.raman = dataclasses.replace(
            problem.raman, rates=(path, *problem.raman.rates[1:]))
    return problem


OPTIONS = ["raman", "no_raman", "absorber_noise", "varying_rate"]


# The largest grids run the Raman case alone.
@pytest.mark.parametrize("n_t, ffac, option", [(n, f, o) for n, f in SIZES for o in OPTIONS
                                               if n <= 65536 or o == "raman"])
def test_trial_over_the_splits(n_t, ffac, option):
    print("envelope trial", n_t, ffac, option, flush=True)
    problem = problem_of(n_t, ffac, option)
    if n_t <= 64:  # fewer samples than the pulse has: a rough field over the active bins
        rng = np.random.default_rng(n_t)
        size = np.abs(problem.field0).max() or 1.0
        problem.field0 = size * problem.active_mask * np.exp(
            2j * np.pi * rng.uniform(size=problem.field0.shape))
    dz = 1e-4
    advanced, norm, _ = oracle_trial(problem, dz)
    ws = Workspace(problem)
    probe = ws.probe(0.0, problem.field0)
    got = probe.trial(0.0, dz)
    field = probe.field()
    ws.close()
    assert rel_l2(field, advanced.reshape(field.shape)) < 1e-12
    y0 = problem.field0.reshape(field.shape)
    assert abs(got - norm) <= norm_bound(problem, advanced, y0)


# From 2^20 samples the kernels at the bins take two to four points a thread; 2^22 to 2^24
# split in sequences of 2048 and 4096 points, the longest. Two stages (Heun's pair) run
# every kernel and keep the oracle's time to seconds.
@pytest.mark.parametrize("n_t, ffac, option", [
    (2**20, 1, "absorber_noise"), (2**20, 4, "absorber_noise"), (2**20, 8, "raman"),
    (2**20, 16, "absorber_noise")])
def test_longest_sequences(n_t, ffac, option):
    print("envelope trial, two stages", n_t, ffac, option, flush=True)
    problem = problem_of(n_t, ffac, option)
    problem.tableau = Tableau(np.array([0.0, 1.0]), np.array([[0.0, 0.0], [1.0, 0.0]]),
                              np.array([0.5, 0.5]), np.array([-0.5, 0.5]), False)
    dz = 1e-4
    advanced, norm, _ = oracle_trial(problem, dz)
    ws = Workspace(problem)
    probe = ws.probe(0.0, problem.field0)
    got = probe.trial(0.0, dz)
    field = probe.field()
    ws.close()
    assert rel_l2(field, advanced.reshape(field.shape)) < 1e-12
    y0 = problem.field0.reshape(field.shape)
    assert abs(got - norm) <= norm_bound(problem, advanced, y0)


# A weak launch without noise: the embedded pair's solutions agree to 1e-9 .. 1e-7 of the
# tolerance, and their difference carries the rounding of the fields they are formed from.
# The oracle's own norm moves by 1e-7 .. 1e-6 of itself when the launch moves by one unit in
# the last place, so nothing closer can be asked of it: over six launches the device's root
# mean square difference from the oracle is held to three times that movement (the same
# arithmetic in another order rounds as much; six differences exceed thrice their standard
# deviation in root mean square once in 1e8).
@pytest.mark.parametrize("n_t", [512, 2048])
@pytest.mark.parametrize("order", [1.0, 1.5])
def test_weak_launch_norm_within_the_oracles_rounding(n_t, order):
    print("envelope weak launch", n_t, order, flush=True)
    problem = gnlse_problem(n_t=n_t, ffac=2, window=10e-12 * n_t / 8192, soliton_order=order,
                            noise_model="none")
    rng = np.random.default_rng(3)
    dz = 1e-4
    differences, movements = [], []
    ws = Workspace(problem)
    for _ in range(6):
        launch = problem.field0 * (1.0 + rng.uniform(-0.05, 0.05))
        problem_at = dataclasses.replace(problem, field0=launch)
        _, norm, _ = oracle_trial(problem_at, dz)
        differences.append(ws.probe(0.0, launch).trial(0.0, dz) - norm)
        for _ in range(3):
            moved = launch.copy()
            parts = moved.view(np.float64)
            parts *= 1.0 + np.finfo(np.float64).eps * rng.choice([-1, 0, 1], size=parts.shape)
            movements.append(
                oracle_trial(dataclasses.replace(problem, field0=moved), dz)[1] - norm)
    ws.close()
    assert 0.0 < norm < 1e-6
    assert np.sqrt(np.mean(np.square(differences))) <= 3.0 * np.sqrt(np.mean(np.square(movements)))


@pytest.mark.parametrize("option", ["raman", "absorber_noise", "varying_rate"])
def test_commits_at_the_head_by_graph_and_direct(option, monkeypatch):
    problem = problem_of(1024, 2, option)
    out = []
    for graph in ("1", "0"):
        monkeypatch.setenv("SOLPROP_MI355X_GRAPH", graph)
        ws = Workspace(problem)
        march = ws.march(0.0, problem.field0)
        rows = [march.advance(problem.z_end, work_limit=7).attempts for _ in range(3)]
        out.append((np.concatenate(rows), march.state()))
        ws.close()
    assert np.array_equal(out[0][0], out[1][0])
    assert np.array_equal(out[0][1], out[1][1])
