"""State read back in packed chunks: sizes around one chunk (43,520 vertices),
two and many chunks, each with x alone, v alone and both."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from positionbaseddynamicsold_amd import capi


@pytest.mark.parametrize("nv", [3, 4, 5, 43519, 43520, 43521, 87040, 87043, 400001])
def test_read_back_equals_what_was_loaded(nv):
    print(f"read back {nv} vertices", flush=True)
    rng = np.random.default_rng(nv)
    x, v = rng.standard_normal((2, nv, 3)).astype(np.float32)
    first = nv // 2 if nv > 5 else nv
    with capi.Context() as ctx:
        ids = []
        for n in (first, nv - first):
            if n:
                i = ctx.add_mesh(np.zeros((n, 3), np.float32), np.array([[0, 1, 2]], np.int32))
                ctx.set_constraint_option(i, 0)
                ids.append((i, n))
        ctx.init()
        ctx.state_load(x, v)
        for _ in range(2):
            a, b = ctx.state_save()
            assert np.array_equal(a, x) and np.array_equal(b, v)
        a[:], b[:] = 0, 0
        capi.check(ctx.lib.pbd_state_save(ctx.h, capi.fptr(a), None))
        capi.check(ctx.lib.pbd_state_save(ctx.h, None, capi.fptr(b)))
        capi.check(ctx.lib.pbd_state_save(ctx.h, None, None))
        assert np.array_equal(a, x) and np.array_equal(b, v)
        at = 0
        for i, n in ids:
            assert np.array_equal(ctx.get(i), x[at : at + n])
            assert np.array_equal(ctx.get(i, capi.STATE_V), v[at : at + n])
            at += n
