"""A training batch in two launches (gradients; sums, Adam and packing) against
the separate gradient and Adam calls, bit for bit: groups of 16 samples full
and partly filled, more groups than one slice of the sum takes at once.  The
samples are all alike, so that the shuffle does not matter."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from positionbaseddynamicsold_amd import capi


@pytest.mark.parametrize("n", [1, 15, 16, 17, 255, 4096, 4097, 9000])
def test_training_step_equals_gradient_and_adam(n):
    print(f"training step over {n} samples", flush=True)
    rng = np.random.default_rng(n)
    X = np.repeat(rng.standard_normal((1, 22)), n, 0).astype(np.float32)
    Y = np.repeat(0.1 * rng.standard_normal((1, 3)), n, 0).astype(np.float32)
    with capi.Context() as a, capi.Context() as b:
        for c in (a, b):
            c.ws_init(5)
            c.ws_set_samples(X, Y)
            c.ws_train(0, 16, 1e-3, 0)  # standardises the samples
        for step in range(3):
            loss = a.ws_train(1, max(16, n), 1e-2, 7 + step)
            grad, want = b.ws_gradient(0, n)
            b.ws_adam_step(grad, 1e-2)
            assert np.float32(loss) == np.float32(want)
            assert np.array_equal(a.ws_params(), b.ws_params())
        for x, y in zip(a.ws_gradient(0, n), b.ws_gradient(0, n)):
            assert np.array_equal(x, y)
