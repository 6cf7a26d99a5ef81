"""Which batches of the sizing network go row by row: both sides of every line of the rule (weights of the later
layers, their reads over all rows, products of parameters and rows, short walks and wide outputs in a forward
pass), inputs split into few long sums, more inputs than a grid has rows, and the device memory that the partial
sums take. Against the float64 oracle.

Tolerance: all sums are FP32; a sum of K products is off by about sqrt(K) 2^-24 of its norm, so eight such steps
(products and sums of three layers, twice) stay below 8 sqrt(K) 2^-24 in the 2-norm, K the longest sum."""
import os
import sys

import numpy as np
import pytest
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle"))
import mlp_oracle as mo  # noqa: E402
from rapidgkc_amd import native  # noqa: E402

pytestmark = pytest.mark.gpu


def _off(a, b):
    return np.linalg.norm(np.asarray(a, dtype=np.float64) - b) / np.linalg.norm(b)


def _net(dims, B):
    """Biases ten deviations of a unit's products from zero, of either sign: no unit is near ReLU's corner, where a
    last bit would turn a whole gradient off."""
    rng = np.random.default_rng(sum(dims) + B)
    w = []
    for a, b, bias in zip(dims[:-1], dims[1:], (14.0, 140.0, 1.0)):
        w += [(rng.standard_normal(a * b) * np.sqrt(2.0 / a)).astype(np.float32),
              (bias * rng.choice([-1.0, 1.0], b)).astype(np.float32)]
    x = rng.standard_normal((B, dims[0])).astype(np.float32)
    t = rng.standard_normal((B, dims[3])).astype(np.float32)
    return np.concatenate(w), x, t


@pytest.mark.parametrize("dims,B", [
    ((40, 2048, 2040, 8), 3), ((40, 2048, 2048, 8), 3),             # 2^22 weights
    ((40, 1024, 1023, 1), 1024), ((40, 1024, 1024, 1), 1024),       # 2^30 reads
    ((1000, 2100, 100, 100), 900), ((1000, 2100, 100, 100), 1000),  # 2^31 products
    ((100, 100, 55, 50), 7), ((100, 100, 56, 50), 7),               # a walk of 256
    ((100, 100, 100, 1200), 7), ((100, 100, 100, 1201), 7),         # outputs of four walks
    ((20_000, 1024, 16, 16), 256),                                  # 64 splits of 320 inputs
    ((2_200_000, 4, 3, 2), 2),                                      # 68750 chunks of inputs
])
def test_mlp_dispatch(dims, B):
    print(f"[gpu] case mlp dispatch {dims} rows {B}", flush=True)
    w, x, t = _net(dims, B)
    w[dims[0] * dims[1]] = 14.0  # at least one unit of layer 1 and of layer 2 is on
    w[dims[0] * dims[1] + dims[1] + dims[1] * dims[2]] = 140.0
    ol, og, oy = mo.loss_and_grad(w, dims, x, t, None)
    tol = 8 * np.sqrt(max(*dims, B)) * 2.0 ** -24
    c = native.Counter(0)
    net = native.Mlp(c, *dims)
    net.set_params(w)
    free = torch.cuda.mem_get_info()[0]
    assert _off(net.forward(x), oy) < tol
    g, l = net.grad(x, t)
    assert _off(g, og) < tol and abs(l - ol) <= tol * ol
    # inputs, targets and activations, 64 MB of partial sums, and what the allocator rounds up
    need = 4 * B * (dims[0] + 2 * dims[1] + 2 * dims[2] + 3 * dims[3])
    assert free - torch.cuda.mem_get_info()[0] <= need + (64 << 20) + (32 << 20)
    net.close()
    c.close()
