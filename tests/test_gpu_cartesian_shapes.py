"""The Cartesian passes at the edges of their shapes: the shortest axes, one, two and three
register stages with every remainder, narrow and wide t workgroups, and operator tables
with a real part, which are stored whole."""

import dataclasses

import numpy as np
import pytest
from test_gpu_cartesian import device_replay, problem_of, rel

from oracle import cartesian as cart

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lossy", [False, True])
@pytest.mark.parametrize("grid", [(4, 4, 4), (8, 4, 16), (4, 16, 2048), (512, 4, 8),
                                  (16, 128, 64), (32, 32, 512), (128, 256, 8),
                                  # 64 and 32 sequences of 4 and 8 points, wide rows of 512
                                  # points, narrow ones of 1024, rows of 4096
                                  (64, 4, 256), (4, 256, 64), (8, 256, 32), (8, 64, 256),
                                  (64, 32, 512), (16, 8, 1024), (4, 4, 4096)])
def test_replay_at_the_edges_of_the_shapes(grid, lossy):
    print("Cartesian replay", grid, "lossy" if lossy else "lossless", flush=True)
    problem = problem_of(*grid)
    if lossy:
        # A loss of up to 40 per cent over the march and a prefactor turned by 0.1 rad.
        rate = np.linspace(0.0, 0.5 / problem.z_end, problem.phi_terms.size)
        problem = dataclasses.replace(
            problem, phi_terms=problem.phi_terms - rate.reshape(problem.phi_terms.shape),
            prefactor_terms=problem.prefactor_terms * np.exp(0.1j))
    expected, _, stiffness = cart.replay(problem, problem.field0)
    state, batch, h_rho = device_replay(problem)
    assert batch.done
    assert rel(state, expected) < 1e-12
    assert abs(h_rho - stiffness[-1]) <= 1e-10 * abs(stiffness[-1])
