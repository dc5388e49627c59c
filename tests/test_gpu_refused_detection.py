"""A detection that is refused leaves nothing of an earlier, smaller scene
behind: the getters would index the new scene's triangles and vertices with the
old scene's edges, pairs and contacts."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from positionbaseddynamicsold_amd import capi


def crossing_sheets(orc, n, gap):
    """Two n x n sheets, the upper one pushed through the lower one's plane."""
    a, ta = orc.grid_mesh(n, n, 1.0, 1.0, jitter=1e-3, seed=1)
    b, tb = orc.grid_mesh(n, n, 0.9, 0.9, jitter=1e-3, seed=2)
    x = np.concatenate([a, b + np.array([0.05, gap, 0.05], np.float32)]).astype(np.float32)
    p = x.copy()
    p[len(a):, 1] -= np.float32(2.0 * gap)
    return x, p, np.concatenate([ta, tb + len(a)]).astype(np.int32)


@pytest.mark.parametrize("first", ["centroid", "swept"])
def test_a_refused_detection_leaves_empty_lists(orc, first):
    th = 0.01
    desc = dict(cell=(0.1, 0.1, 0.1), table_bits=12)
    d, g = capi.hash_desc(1, **desc), orc.grid(1, **desc)
    x, p, tris = crossing_sheets(orc, 8, 0.015)
    X, P, big = crossing_sheets(orc, 24, 0.015)
    far = P.copy()
    far[-1] += np.float32(1e4)  # its box spans more cells than are allowed
    w = np.ones(len(X), np.float32)
    with capi.Context() as ctx:
        ctx.sh_build(d, x, tris)
        assert len(ctx.ccd_detect(d, x, p, tris, th, swept=first == "swept")[0]) > 0
        assert len(ctx.ccd_detect_ee(d, x, p, tris, th)[0]) > 0
        assert len(ctx.ccd_pairs()) > 0
        with pytest.raises(capi.PbdError, match="4096 cells") as e:
            ctx.ccd_detect(d, X, far, big, th, swept=True)
        assert e.value.code == capi.PBD_ERR_LIMIT
        assert len(ctx.ccd_pairs()) == 0 and len(ctx.ccd_ee_pairs()) == 0
        assert np.array_equal(ctx.ccd_resolve(far, w, th, 2), far)
        # the cell table is that of the scene at hand
        ctx._sh_nt = len(big)
        assert np.array_equal(ctx.sh_get()[2], orc.tri_keys(g, far, big)[0])
        # an edge detection on the refused scene has no vertex-face contacts to go with
        for a, b in zip(ctx.ccd_detect_ee(d, X, far, big, th), orc.ccd_detect_ee(g, X, far, big, th)):
            assert np.array_equal(a, b)
        assert len(ctx.ccd_pairs()) == 0
        # and the next detection is whole again
        arr, n = orc.ccd_detect(g, X, P, big, th)
        assert n > 0
        for a, b in zip(ctx.ccd_detect(d, X, P, big, th), orc.contacts_arrays(arr, n)):
            assert np.array_equal(a, b)
        assert np.array_equal(ctx.ccd_pairs(), orc.candidate_pairs(g, P, big))
