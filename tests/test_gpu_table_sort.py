"""The sorted broadphase table against numpy's stable sort of its own keys:
sizes at the edges of a sort tile (4096), one tile per row sum and beyond the
256 tiles that a workgroup sums itself; one to four digits; keys spread out,
few, all alike and outside the grid; both entry points, the second also with
arrays that are not 16-byte aligned."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from positionbaseddynamicsold_amd import capi
from test_zz_no_alloc import DeviceArrays


def triangles(nt, spread, seed):
    rng = np.random.default_rng(seed)
    nv = min(3 * nt, 100_003)
    pos = (spread * rng.standard_normal((nv, 3))).astype(np.float32)
    return pos, rng.integers(0, nv, (nt, 3)).astype(np.int32)


def check(keys, ids, raw, start, end):
    order = np.argsort(raw, kind="stable")
    assert np.array_equal(ids, order)
    assert np.array_equal(keys, raw[order])
    want = [np.full(len(start), -1, np.int32), np.full(len(end), -1, np.int32)]
    k = keys[keys >= 0]
    first = len(keys) - len(k)
    want[0][k[::-1]] = np.arange(len(keys) - 1, first - 1, -1)
    want[1][k] = np.arange(first, len(keys))
    assert np.array_equal(start, want[0]) and np.array_equal(end, want[1])


CASES = [(1, (1, 4)), (63, (1, 4)), (65, (1, 12)), (4095, (1, 12)), (4096, (1, 20)), (4097, (1, 20)), (8193, (0, 0)),
         (100_000, (1, 24)), (1 << 20, (1, 20)), (1 << 20, (1, 7)), ((1 << 20) + 4097, (1, 20))]


@pytest.mark.parametrize("nt,grid", CASES)
@pytest.mark.parametrize("spread", [0.0, 0.3, 20.0])
def test_table_is_the_stable_sort_of_its_keys(nt, grid, spread):
    print(f"table of {nt} triangles, grid {grid}, spread {spread}", flush=True)
    pos, tris = triangles(nt, spread, nt)
    d = capi.hash_desc(grid[0], (0.0, 0.0, 0.0), (12, 4, 12), (0.1, 0.1, 0.1), grid[1])
    with capi.Context() as ctx:
        ctx.sh_build(d, pos, tris)
        got = ctx.sh_get()
    check(*got)
    if nt > 1 << 20:
        return
    cells = len(got[3])
    dev = DeviceArrays()
    try:
        dpos, dtris = dev.upload(pos), dev.upload(tris)
        for shift in (0, 1):
            out = [dev.filled(n + shift) for n in (nt, nt, nt, cells, cells)]
            at = [C.c_void_p(p.value + 4 * shift) for p in out]
            assert capi.load().pbd_sh_build_noalloc(0, None, C.byref(d), dpos, len(pos), dtris, nt, *at) == capi.PBD_OK
            for p, want in zip(out, got):
                assert np.array_equal(dev.download(p, len(want) + shift)[shift:], want)
    finally:
        dev.free()
