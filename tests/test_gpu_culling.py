"""Boxes and half-spaces may only rule out pairs that are no contacts.  Each
case here has faces that they apply to, contacts with such faces, and pairs
near them that are none; sizes from a centimetre up and far from the origin."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from positionbaseddynamicsold_amd import capi


def tumbling(move, shift, scale, seed):
    """Well-shaped triangles close together, each moved and turned."""
    rng = np.random.default_rng(seed)
    nt = 300
    a = rng.uniform(0, 2 * np.pi, (nt, 1)) + np.array([0.0, 2.1, 4.2]) + 0.3 * rng.standard_normal((nt, 3))
    u, v = np.linalg.qr(rng.standard_normal((nt, 3, 3)))[0][:, :2].transpose(1, 0, 2)
    corner = rng.uniform(0, 0.2, (nt, 1, 3)) + 0.03 * (np.cos(a)[..., None] * u[:, None] + np.sin(a)[..., None] * v[:, None])
    x = ((corner.reshape(-1, 3) + shift) * scale).astype(np.float32)
    p = x + scale * move * (rng.standard_normal((nt, 1, 3)) + 0.1 * rng.standard_normal((nt, 3, 3))).reshape(-1, 3)
    return x, p.astype(np.float32), np.arange(3 * nt, dtype=np.int32).reshape(nt, 3)


def may_be_culled(x, p, tris, th):
    """The faces that boxes may rule pairs out of: a good shape over the whole
    step, and a thickness that is not tiny beside the edges."""
    X, P = x[tris].astype(np.float64), p[tris].astype(np.float64)
    e1, e2 = X[:, 1] - X[:, 0], X[:, 2] - X[:, 0]
    d1, d2 = P[:, 1] - P[:, 0] - e1, P[:, 2] - P[:, 0] - e2
    length = lambda v: np.linalg.norm(v, axis=1)  # noqa: E731
    l1, l2, m1, m2 = length(e1), length(e2), length(d1), length(d2)
    longest = np.maximum(np.maximum(l1, l2), length(e2 - e1)) + m1 + m2
    area = length(np.cross(e1, e2)) - (l1 * m2 + l2 * m1 + m1 * m2)
    return (area >= 0.05 * longest**2) & (th >= 4e-3 * longest)


@pytest.mark.parametrize("swept", [False, True])
@pytest.mark.parametrize("th", [4e-4, 2e-3, 0.01])
@pytest.mark.parametrize("move", [0.0, 0.003, 0.02])
@pytest.mark.parametrize("shift,scale", [(0.0, 1.0), (200.0, 1.0), (0.0, 0.1), (0.0, 50.0)])
def test_every_contact_is_kept(orc, swept, th, move, shift, scale):
    print(f"culling swept={swept} th={th} move={move} shift={shift} scale={scale}", flush=True)
    x, p, tris = tumbling(move, shift, scale, 7)
    t = np.float32(th * scale)
    cull = may_be_culled(x, p, tris, t)
    desc = dict(cell=(0.25 * scale,) * 3, table_bits=9)
    arr, n = orc.ccd_detect_swept(x, p, tris, t) if swept else orc.ccd_detect(orc.grid(1, **desc), x, p, tris, t)
    want = orc.contacts_arrays(arr, n)
    assert n > 0 and cull[want[0][:, 1]].sum() > 0 and cull.sum() > 100
    with capi.Context() as ctx:
        got = ctx.ccd_detect(capi.hash_desc(1, **desc), x, p, tris, t, swept=swept)
        assert len(ctx.ccd_pairs()) > 2 * n
        for a, b in zip(got, want):
            assert np.array_equal(a, b)
