"""The launch forms of the tile kernel against the per-colour launches over
global memory, bit for bit: records kept in registers (one and two per thread
and colour) or fetched phase by phase, several substeps in one launch, tiles
smaller than the budget.  Sizes lie at the edges of the forms' ranges."""
import numpy as np
import pytest

from positionbaseddynamicsold_amd import capi, scenes

pytestmark = pytest.mark.gpu


def context(rx, ry, stiffness, pins, sphere):
    ctx = capi.Context()
    cid = ctx.add_grid(rx, ry, 1.0, (ry - 1) / (rx - 1), jitter=1e-3, seed=rx * 1000 + ry)
    ctx.set_constraint_option(cid, capi.DISTANCE, (stiffness, 1.0, 1.0))
    if pins:
        ctx.set_pins(cid, [0, 1, rx - 1, rx * ry - 1])
    if sphere:
        ctx.set_params(cid, sphere_on=1, sphere_c=(0.5, -0.29, 0.5), sphere_r=0.3)
    ctx.init()
    return ctx, cid


# colours of up to 256, 512, 1024, 2048 and more records, one tile; several tiles
@pytest.mark.parametrize("rx,ry", [(2, 2), (5, 3), (22, 23), (23, 23), (32, 32), (46, 45), (64, 64), (65, 63), (100, 90),
                                   (131, 70)])
@pytest.mark.parametrize("stiffness,pins,sphere", [(1.0, True, False), (0.6, False, True)])
def test_forms_equal_global_launches(rx, ry, stiffness, pins, sphere):
    print(f"forms {rx}x{ry} s={stiffness} pins={pins} sphere={sphere}", flush=True)
    want = None
    for kw in (dict(path=capi.PATH_GLOBAL), dict(), dict(graph=1), dict(block_threads=256), dict(block_threads=1024),
               dict(tile_max_verts=1500, graph=1), dict(tile_sweeps=3, tile_max_verts=4000)):
        ctx, cid = context(rx, ry, stiffness, pins, sphere)
        with ctx:
            ctx.set_solver(dt=scenes.DT, iterations=7, **kw)
            if kw.get("path"):
                for _ in range(3):
                    ctx.step(1)
            else:
                ctx.step(2)
                ctx.step(1)
            got = ctx.get(cid), ctx.get(cid, capi.STATE_V), ctx.get(cid, capi.STATE_P)
            assert ctx.last_sweeps(cid) == 7
        if want is None:
            want = got
        for a, b in zip(want, got):
            assert np.array_equal(a, b), kw
