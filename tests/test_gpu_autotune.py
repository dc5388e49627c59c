"""What the autotuner returns: settings that the launches really have, and none
that are slower than those at hand."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from positionbaseddynamicsold_amd import capi


def grids(sizes, bend, **kw):
    ctx = capi.Context()
    for n, m in sizes:
        c = ctx.add_grid(n, m, 1.0, 1.0, jitter=1e-4, seed=0)
        ctx.set_constraint_option(c, capi.DISTANCE | (capi.BENDING if bend else 0), (1.0, 0.1, 1.0))
        ctx.set_pins(c, [0])
    ctx.init()
    ctx.set_solver(**kw)
    ctx.step(2)
    return ctx


@pytest.mark.parametrize("asked", [0, 2])
def test_bending_grids_are_returned_the_one_sweep_they_run(asked):
    with grids([(90, 90)], True, tile_sweeps=asked) as ctx:
        p, _, ms, trials = ctx.autotune(2)
        print(f"{trials} candidates, {ms:.3f} ms: {p.tile_sweeps} sweeps, {p.block_threads} threads", flush=True)
        assert p.tile_sweeps == 1


def test_settings_at_hand_stay_where_no_candidate_is_as_fast():
    # thousands of tiny cloths: a wave each leaves room for many on a CU (3000
    # of them, 40 substeps: 2.6 ms with 64 threads, 5.8 with 256, the fewest of
    # the candidates)
    with grids([(8, 8)] * 3000, False, block_threads=64) as ctx:
        p, _, ms, trials = ctx.autotune(40)
        print(f"{trials} candidates, {ms:.4f} ms: {p.block_threads} threads", flush=True)
        assert p.block_threads == 64


@pytest.mark.parametrize("sizes,bend", [([(32, 32)] * 8, False), ([(120, 77), (30, 30)], False), ([(60, 50)], True)])
def test_states_and_results_are_unchanged(sizes, bend):
    with grids(sizes, bend) as a, grids(sizes, bend) as b:
        a.autotune(3)
        for _ in range(2):
            for x, y in zip(a.state_save(), b.state_save()):
                assert np.array_equal(x, y)
            a.step(7)
            b.step(7)
