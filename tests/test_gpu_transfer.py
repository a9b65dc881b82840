"""Large fields cross to the device and back bit for bit: sizes below, at and above the
pipelined copies' thresholds (8 MB; 32 MB for the slots at once; 64 MB to the device), and no
multiple of their chunk; often enough that slots are made for the middle sizes; two
workspaces at once."""

import threading

import numpy as np
import pytest

from solprop_amd.native import Workspace
from solprop_amd.problem import cartesian_problem, radial_problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(64, 64, 64), (128, 64, 64), (256, 256, 16), (64, 64, 512),
                                   (128, 64, 512)])
def test_cartesian_field_round_trip(shape):
    nx, ny, nt = shape
    problem = cartesian_problem(nx=nx, ny=ny, n_t=nt, spacing=96e-6 / nx, waist=20e-6, steps=2,
                                length=1e-6)
    rng = np.random.default_rng(3)
    ws = Workspace(problem)
    for _ in range(2 if nx * ny * nt > 2**21 else 10):
        field = rng.standard_normal(problem.field0.shape) + 1j * rng.standard_normal(
            problem.field0.shape)
        ws.load(0.0, field)
        assert np.array_equal(ws.state(), field)
    ws.close()


def test_two_workspaces_at_once():
    problem = radial_problem(n_t=4096, window=0.5e-12, n_r=331, length=0.02)
    rng = np.random.default_rng(5)
    fields = [rng.standard_normal((331, 2049)) + 1j * rng.standard_normal((331, 2049))
              for _ in range(2)]  # 10.9 MB, no multiple of a chunk
    spaces = [Workspace(problem) for _ in fields]
    out = [[], []]

    def turn(i):
        for _ in range(8):
            spaces[i].load(0.0, fields[i])
            out[i].append(spaces[i].state())

    threads = [threading.Thread(target=turn, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for ws in spaces:
        ws.close()
    assert all(np.array_equal(a, b) for states, b in zip(out, fields) for a in states)
