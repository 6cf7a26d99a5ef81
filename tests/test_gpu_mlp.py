"""The sizing network's row-by-row path and its neighbours against the float64 oracle: one row, rows around
a workgroup's 64, the last batch that goes by rows and the first that does not, layer widths around the
waves' and workgroups', inputs that do not fill a chunk, masks with zeros and with nothing left, and
widths too large for the rows' LDS.

Tolerance: all sums are FP32 over at most 2563 terms, three layers deep; a sum of K products is off by
about sqrt(K) 2^-24 of its norm, so eight such steps (products and sums of three layers, twice) stay
below 8 sqrt(2563) 2^-24 = 2.4e-5 in the 2-norm."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle"))
import mlp_oracle as mo  # noqa: E402

pytestmark = pytest.mark.gpu
TOL = 8 * np.sqrt(2563) * 2.0 ** -24


def _off(a, b):
    n = np.linalg.norm(b)
    return np.linalg.norm(np.asarray(a, dtype=np.float64) - b) / n if n else np.linalg.norm(a)


@pytest.mark.parametrize("dims,B,mask", [
    ((2563, 128, 128, 1024), 16, None), ((2563, 128, 128, 1024), 1, "some"), ((2563, 128, 128, 1024), 65, "some"),
    ((5, 3, 2, 1), 3, None), ((33, 100, 7, 1025), 64, "some"), ((31, 1, 1, 2000), 2, None), ((32, 1030, 65, 10), 5, "none"),
    ((97, 64, 128, 127), 1024, None), ((97, 64, 128, 127), 1025, "some"), ((40, 9000, 8, 6500), 4, None),
])
def test_mlp_rows(dims, B, mask):
    from rapidgkc_amd import native
    print(f"[gpu] case mlp {dims} rows {B} mask {mask}", flush=True)
    rng = np.random.default_rng(sum(dims) + B)
    w = []
    for a, b in zip(dims[:-1], dims[1:]):
        w += [(rng.standard_normal(a * b) * np.sqrt(2.0 / a)).astype(np.float32), (0.1 * rng.standard_normal(b)).astype(np.float32)]
    w = np.concatenate(w)
    x = rng.standard_normal((B, dims[0])).astype(np.float32)
    t = rng.standard_normal((B, dims[3])).astype(np.float32)
    m = {None: None, "some": (rng.random((B, dims[3])) < 0.6).astype(np.float32),
         "none": np.zeros((B, dims[3]), dtype=np.float32)}[mask]
    c = native.Counter(0)
    net = native.Mlp(c, *dims)
    net.set_params(w)
    ol, og, oy = mo.loss_and_grad(w, dims, x, t, m)
    assert _off(net.forward(x), oy) < TOL
    for _ in range(2):
        g, l = net.grad(x, t, m)
        assert _off(g, og) < TOL and abs(l - ol) <= TOL * max(ol, 1e-30)
    net.close()
    c.close()
