"""GPU: the surrogate's fused tile path at the edges of its padding, and the general
products of wider networks, against the FP64 oracle (``oracle/fno.py``).

Channels pad to 32 or 64, twice the modes to 64 or 128, bins to tiles of 64 and samples
to runs of 16. A batch splits each sample's tiles over some 512 workgroups forward and 256
backward: small ones give a workgroup one tile, the larger ones below a run of two to
eleven, whole or with a short last run, so that the buffers alternate and the spectral,
weight and bias sums are kept over tiles (`test_runs_of_tiles` holds the splits). The shapes
sit on and beside each of these edges. BF16 operands (unit roundoff 2^-9) pass
through two products a layer forward and three back, so a tensor's relative error is a
few 2^-9 sqrt(layers): the bounds are those of the other surrogate tests, 2 % and a cosine
of 0.9995, which one wrong row, column or sign in a small tensor breaks.
"""

import numpy as np
import pytest

from oracle import fno as oracle
from solprop_amd import surrogate
from test_gpu_fno import case, rel

pytestmark = pytest.mark.gpu

# (width, modes, layers, hidden, n, scan parameters, batch)
EDGES = [
    (1, 1, 1, 1, 4, 0, 1),
    (16, 8, 2, 32, 63, 1, 5),
    (31, 32, 2, 33, 64, 4, 17),
    (33, 33, 3, 127, 65, 8, 2),
    (48, 24, 4, 64, 500, 4, 16),
    (64, 64, 2, 128, 129, 4, 33),
    (64, 64, 4, 128, 2048, 4, 3),
    (64, 65, 2, 128, 256, 4, 3),
    (65, 16, 2, 64, 256, 4, 3),
    (32, 16, 2, 129, 256, 4, 3),
    # Runs of tiles: 4 and 8, 5 (2 at the end) and 11 (10), 3 (2, ragged bins) and 8, 3, 2.
    (16, 8, 2, 32, 2048, 4, 64),
    (48, 40, 2, 64, 2048, 4, 67),
    (33, 33, 2, 127, 500, 4, 130),
    (64, 64, 2, 128, 129, 4, 300),
    (32, 32, 1, 16, 65, 1, 520),
]


def tile_runs(n, batch, groups):
    """Tiles a workgroup and in a sample's last one (``fno_tile.hip`` ``tile_split``)."""
    tiles = -(-n // 64)
    per = -(-tiles // max(1, min(tiles, groups // batch)))
    return per, (tiles - 1) % per + 1


def test_runs_of_tiles():
    forward = {tile_runs(e[4], e[6], 512) for e in EDGES}
    backward = {tile_runs(e[4], e[6], 256) for e in EDGES}
    assert forward >= {(1, 1), (4, 4), (5, 2), (3, 2), (3, 3), (2, 2)}
    assert backward >= {(1, 1), (8, 8), (11, 10), (3, 3), (2, 2)}


@pytest.mark.parametrize("edge", EDGES, ids=lambda e: "-".join(map(str, e)))
def test_forward_and_gradient_at_the_edges(edge):
    width, modes, layers, hidden, n, n_params, batch = edge
    print("fno tiles", edge, flush=True)
    shape = surrogate.Shape(n_params=n_params, width=width, modes=modes, layers=layers,
                            hidden=hidden, n=n)
    o, flat, spectra, params, target = case(shape, batch, seed=3)
    net = surrogate.Network(shape, max_batch=batch + 3)
    net.set_parameters(flat)
    # A full batch first, so that a smaller one after it must not see its rows.
    full = np.resize(spectra, (batch + 3, n)), np.resize(params, (batch + 3, n_params))
    first = net.forward(*full)
    got = net.forward(spectra, params)
    loss, grad = net.gradient(spectra, params, target)
    again = net.gradient(spectra, params, target)
    net.close()
    assert loss == again[0] and np.array_equal(grad, again[1])
    x = surrogate.oracle_inputs(spectra, params)
    loss_ref, grad_ref, out_ref = oracle.loss_and_grad(o, flat.astype(np.float64), x, target)
    assert rel(got, out_ref) < 2e-2
    assert rel(first[:batch], out_ref) < 2e-2
    assert abs(loss - loss_ref) <= 2e-2 * loss_ref
    at = 0
    for name, shp in oracle.layout(o):
        size = int(np.prod(shp))
        g, r = grad[at:at + size].astype(np.float64), grad_ref[at:at + size]
        at += size
        norm = np.linalg.norm(r)
        if norm < 1e-9 * np.linalg.norm(grad_ref):
            continue  # a mode that the grid does not carry (the imaginary part at zero)
        assert rel(g, r) < 2e-2, (name, rel(g, r))
        assert g @ r / (np.linalg.norm(g) * norm) > 0.9995, name


@pytest.mark.parametrize("span", [1.0, 4.0, 12.0])
def test_head_slope_against_64_bits(span):
    """The head's units held at given pre-activations by their biases alone (all other
    weights zero): the biases' gradients are gelu's slopes there. Computed from tanhf the
    slope is within 5.6e-7 of 64 bits over |x| < 12 (3.6e-7 below 4); the bound adds the
    rounding of the sum over 64 equal bins, eight additions of at most half a unit each."""
    print("fno gelu slope", span, flush=True)
    shape = surrogate.Shape(n_params=1, width=8, modes=4, layers=1, hidden=128, n=64)
    o = oracle.Shape(in_ch=shape.in_ch, width=8, modes=4, layers=1, hidden=128, n=64)
    x = (span * np.linspace(-0.99, 0.99, 128)).astype(np.float32)
    weight = np.float32(2.0**-20)
    p = {name: np.zeros(size) for name, size in oracle.layout(o)}
    p["q1_b"], p["q2_w"], p["q2_b"] = x, np.full((1, 128), weight), np.full(1, 0.5)
    net = surrogate.Network(shape, max_batch=1)
    net.set_parameters(oracle.flatten(o, p).astype(np.float32))
    zero, params = np.zeros((1, 64), np.float32), np.zeros((1, 1), np.float32)
    out = net.forward(zero, params)
    assert np.all(out == out[0, 0])
    _, grad = net.gradient(zero, params, zero)
    net.close()
    got = oracle.unflatten(o, grad.astype(np.float64))["q1_b"] / (float(weight) * 2.0 * out[0, 0])
    v = x.astype(np.float64)
    c, a = np.sqrt(2.0 / np.pi), 0.044715
    s = 1.0 / (1.0 + np.exp(-2.0 * c * (v + a * v**3)))
    slope = s + 2.0 * v * s * (1.0 - s) * c * (1.0 + 3.0 * a * v**2)
    assert np.max(np.abs(got - slope)) <= 5.6e-7 + 8 * 2.0**-24
