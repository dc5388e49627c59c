"""Limits of the tile plan.  The largest tile: 160 KiB of LDS less 256 bytes hold
10,224 vertices."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from positionbaseddynamicsold_amd import capi

LARGEST = (160 * 1024 - 256) // 16


def stepped(pos, tris, path, bend):
    with capi.Context() as ctx:
        c = ctx.add_mesh(pos, tris)
        ctx.set_constraint_option(c, capi.DISTANCE | (capi.BENDING if bend else 0), (1.0, 0.1, 1.0))
        ctx.set_pins(c, [0, 141])
        ctx.init()
        ctx.set_solver(iterations=4, path=path)
        ctx.step(3)
        return ctx.info(c), ctx.get(c)


@pytest.mark.parametrize("bend", [False, True])
def test_a_mesh_of_the_largest_tile_is_one_tile(orc, bend):
    pos, tris = orc.grid_mesh(142, 72, 1.0, 0.5, jitter=1e-4, seed=0)
    assert len(pos) == LARGEST
    info, x = stepped(pos, tris, capi.PATH_AUTO, bend)
    assert (info.whole, info.ntiles, info.max_loaded) == (1, 1, LARGEST)
    assert np.array_equal(x, stepped(pos, tris, capi.PATH_GLOBAL, bend)[1])


def test_one_vertex_more_is_not(orc):
    pos, tris = orc.grid_mesh(142, 72, 1.0, 0.5, jitter=1e-4, seed=0)
    pos = np.concatenate([pos, [[1.01, 0.0, 0.5]]]).astype(np.float32)
    tris = np.concatenate([tris, [[LARGEST - 1, LARGEST, LARGEST - 1 - 142]]]).astype(np.int32)
    info, x = stepped(pos, tris, capi.PATH_AUTO, False)
    assert info.whole == 0 and 1 < info.ntiles and info.max_loaded <= LARGEST
    assert np.array_equal(x, stepped(pos, tris, capi.PATH_GLOBAL, False)[1])


# budgets too small for the cones of the four sweeps that a launch runs by default
@pytest.mark.parametrize("budget", [64, 100, 256, 512, 1024])
@pytest.mark.parametrize("before_init", [False, True])
def test_small_budgets_take_fewer_sweeps_per_launch(budget, before_init):
    x = []
    for path in (capi.PATH_AUTO, capi.PATH_GLOBAL):
        with capi.Context() as ctx:
            c = ctx.add_grid(46, 34, 1.0, 0.7, jitter=1e-4, seed=0)
            ctx.set_constraint_option(c, capi.DISTANCE, (1.0, 1.0, 1.0))
            ctx.set_pins(c, [0, 45])
            if before_init:
                ctx.set_solver(iterations=5, path=path, tile_max_verts=budget)
                ctx.init()
            else:
                ctx.init()
                ctx.set_solver(iterations=5, path=path, tile_max_verts=budget)
            ctx.step(3)
            assert path == capi.PATH_GLOBAL or ctx.info(c).max_loaded <= budget
            x.append(ctx.get(c))
            # a larger budget takes four again
            ctx.set_solver(iterations=5, path=path)
            ctx.step(3)
            x.append(ctx.get(c))
    assert np.array_equal(x[0], x[2]) and np.array_equal(x[1], x[3])


@pytest.mark.parametrize("mesh", [False, True])
def test_init_refuses_a_budget_that_no_plan_fits(orc, mesh):
    pos, tris = orc.grid_mesh(20, 20, 1.0, 1.0, jitter=1e-4, seed=0)
    with capi.Context() as ctx:
        c = ctx.add_mesh(pos, tris) if mesh else ctx.add_grid(20, 20, jitter=1e-4)
        ctx.set_constraint_option(c, capi.DISTANCE, (1.0, 1.0, 1.0))
        ctx.set_solver(iterations=4, tile_sweeps=4, tile_max_verts=64)
        with pytest.raises(capi.PbdError, match="tile budget") as e:
            ctx.init()
        assert e.value.code == capi.PBD_ERR_LIMIT
        ctx.set_solver(iterations=4, tile_max_verts=1024)
        ctx.init()
        ctx.step(1)
        assert np.isfinite(ctx.get(c)).all()


@pytest.mark.parametrize("form,whole", [(0, 0), (1, 0), (2, 1)])
def test_a_launch_that_decides_keeps_cloths_of_one_tile_whole(form, whole):
    # the tiles of a cloth wait for each other there
    with capi.Context() as ctx:
        for n in (60, 130):
            c = ctx.add_grid(n, n, 1.0, 1.0, jitter=1e-4, seed=n)
            ctx.set_constraint_option(c, capi.DISTANCE, (1.0, 1.0, 1.0))
            ctx.set_pins(c, [0])
        ctx.init()
        ctx.ws_init(0)
        ctx.ws_enable(True)
        ctx.set_solver(iterations=6, tile_sweeps=2, check_every=2, warm_iterations=2, per_chunk_launches=form)
        assert (ctx.info(0).whole, ctx.info(0).ntiles, ctx.info(1).whole) == (whole, 1, 0)
        ctx.step(2)
        assert np.isfinite(ctx.get(0)).all()
