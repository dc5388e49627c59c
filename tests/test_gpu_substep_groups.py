"""Contexts of single-tile cloths run several substeps in one launch, grouped so
that no launch is long: any number of substeps equals as many single ones."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from positionbaseddynamicsold_amd import capi

SIZES = [(9, 31), (32, 32), (17, 5), (2, 2), (40, 23)]


def stepped(calls, iterations, bend):
    with capi.Context() as ctx:
        for k, (rx, ry) in enumerate(SIZES):
            c = ctx.add_grid(rx, ry, 1.0, 0.8, jitter=1e-4, seed=k)
            ctx.set_constraint_option(c, capi.DISTANCE | (capi.BENDING if bend else 0), (1.0, 0.1, 1.0))
            ctx.set_pins(c, [0])
            ctx.set_params(c, sphere_on=k % 2, sphere_c=(0.5, -0.3, 0.4), sphere_r=0.25, damping=0.99)
        ctx.init()
        ctx.set_solver(iterations=iterations)
        for n in calls:
            ctx.step(n)
        assert all(ctx.info(c).whole for c in range(len(SIZES)))
        return *ctx.state_save(), [ctx.get(c, capi.STATE_P) for c in range(len(SIZES))], ctx.last_sweeps(0)


# groups of 64, of 30 and of one substep, with and without a remainder
@pytest.mark.parametrize("substeps,iterations", [(130, 4), (128, 5), (65, 68), (3, 2100)])
@pytest.mark.parametrize("bend", [False, True])
def test_grouped_substeps_equal_single_ones(substeps, iterations, bend):
    print(f"{substeps} substeps of {iterations} sweeps, bend={bend}", flush=True)
    x, v, p, sweeps = stepped([substeps], iterations, bend)
    X, V, P, _ = stepped([1] * substeps, iterations, bend)
    assert sweeps == iterations
    assert np.isfinite(x).all() and np.array_equal(x, X) and np.array_equal(v, V)
    assert all(np.array_equal(a, b) for a, b in zip(p, P))
