"""Bending prims with few or no distance prims: colours without distance
records, between colours that have some."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from positionbaseddynamicsold_amd import capi


@pytest.mark.parametrize("n", [5, 32, 90])
@pytest.mark.parametrize("pairs", ["none", "two", "star"])
def test_colours_without_distance_prims_equal_the_global_path(orc, n, pairs):
    pos, tris = orc.grid_mesh(n, n, 1.0, 1.0, jitter=1e-3, seed=1)
    # disjoint pairs have one colour; a star has one per pair, up to far beyond those of the bending prims
    pr = {"none": None, "two": [[0, 1], [2 * n, 2 * n + 1]], "star": [[0, k] for k in range(1, min(len(pos), 30))]}[pairs]
    x = []
    for path in (capi.PATH_AUTO, capi.PATH_GLOBAL):
        with capi.Context() as ctx:
            c = ctx.add_mesh(pos, tris)
            if pr:
                ctx.set_distance_pairs(c, np.array(pr, np.int32))
            ctx.set_constraint_option(c, capi.BENDING | (capi.DISTANCE if pr else 0), (1.0, 0.2, 1.0))
            ctx.set_pins(c, [0, n - 1])
            ctx.init()
            ctx.set_solver(iterations=6, path=path)
            ctx.step(4)
            x.append(ctx.get(c))
    assert np.isfinite(x[0]).all() and np.array_equal(x[0], x[1])
