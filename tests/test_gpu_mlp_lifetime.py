"""A network and its context end in either order, as the garbage collector may end them: calls on a network
whose context is gone report it, and the network can still be closed."""
import gc

import numpy as np
import pytest

from rapidgkc_amd import native

pytestmark = pytest.mark.gpu


def test_context_goes_first():
    c = native.Counter(0)
    a, b = native.Mlp(c, 8, 4, 4, 3), native.Mlp(c, 5, 4, 4, 2)
    x = np.ones((2, 8), dtype=np.float32)
    a.set_params(np.ones(a.n_params, dtype=np.float32))
    assert np.isfinite(a.forward(x)).all()
    b.close()
    print("[gpu] case network after its context", flush=True)
    c.close()
    for call in (lambda: a.forward(x), lambda: a.grad(x, np.ones((2, 3))), a.get_params,
                 lambda: a.train_step(x, np.ones((2, 3))), lambda: a.set_params(np.ones(a.n_params))):
        with pytest.raises(native.RgkcError) as e:
            call()
        assert e.value.code == -6
    a.close()


def test_collected_in_a_cycle():
    for _ in range(3):
        ring = [native.Counter(0)]
        ring += [native.Mlp(ring[0], 8, 4, 4, 3), ring]
        del ring
        gc.collect()
