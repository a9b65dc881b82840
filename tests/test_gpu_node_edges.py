"""The fused node passes where their shapes end: node counts that leave waves and groups
partly filled, one to eight modes, one to six filter taps, a grid of few tiles. The whole
trial against the oracle's, under the tolerances of test_gpu_field (the fields cancel
nothing; the norm is an error estimate)."""

import pytest
from test_gpu_field import oracle_first_trial, rel_l2

from solprop_amd.native import Workspace
from solprop_amd.problem import capillary_problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("modes, nodes, n_t, rule", [
    (1, 9, 2048, "trapezoid"), (1, 12, 2048, "band"), (2, 31, 2048, "band"),
    (3, 33, 2048, "trapezoid"), (4, 61, 2048, "band"), (5, 32, 2048, "band"),
    (6, 97, 2048, "trapezoid"), (7, 40, 2048, "band"), (8, 64, 2048, "band"),
    (4, 128, 4096, "band")])
def test_trial_at_the_edges(modes, nodes, n_t, rule):
    print("node passes", modes, nodes, n_t, rule, flush=True)
    problem = capillary_problem(n_t=n_t, n_modes=modes, n_nodes=nodes, length=0.05,
                                integration=rule, band=(300e-9, 4e-6))
    dz = 2e-4
    advanced, norms = oracle_first_trial(problem, dz)
    ws = Workspace(problem)
    probe = ws.probe(0.0, problem.field0)
    got = probe.trial(0.0, dz)
    field = probe.field()
    ws.close()
    assert rel_l2(field, advanced.reshape(field.shape)) < 1e-11
    assert abs(got - norms[0]) / norms[0] < 1e-8
