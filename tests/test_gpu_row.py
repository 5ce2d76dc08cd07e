"""The one-pass row reductions (gm_reductions) against numpy on the fields
and positions the context holds, at grids on both sides of the kernel's
splits: one plane a thread and several, 16 rows of epsilon* and one more,
more columns than workgroups.

The operations per point are the same; sums are reordered (at most 2.2e6
terms of one sign in partial sums: 1e-12 relative), exp, sin, cos, sqrt and
the quotients may differ by a few last bits (1e-13 relative for maxima)."""
import numpy as np
import pytest

from conftest import small_braid

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def g(require_gpu):
    import glemur_amd
    return glemur_amd


def norm(a):
    return np.sqrt((a * a).sum(-1))


@pytest.mark.parametrize("prec", ["F64", "F32K"])
@pytest.mark.parametrize("shape", [(2, 2, 2), (17, 5, 16), (16, 16, 17), (31, 67, 260), (300, 300, 30), (1100, 1000, 2)])
def test_row_reductions(g, prec, shape):
    p = small_braid(*shape)
    for k in ("redB2", "redJMax", "redJxB_B2Max", "redConvex", "redWedgeMin", "redErrB_1ez", "redErrXb_XbAn",
              "redEpsilonStar"):
        setattr(p, k, True)
    p.ar, p.az, p.phi1 = 1.3, 3.0, 0.6
    nx, ny, nz = shape
    B0, xb = g.init_state(p)
    x = xb.reshape(nz + 2, ny + 2, nx + 2, 3).copy()
    r = np.random.default_rng(3)
    x[1:-1, 1:-1, 1:-1] += r.uniform(-0.1, 0.1, (nz, ny, nx, 3)) * (p.dx, p.dy, p.dz)
    with g.Context(p, getattr(g, "PREC_" + prec)) as c:
        c.upload(B0, x.reshape(-1), 0.0, 0.01)
        c.fields()
        res = c.reductions()
        x, B = (c.download(f).reshape(nz + 2, ny + 2, nx + 2, 3) for f in (g.FIELD_XB, g.FIELD_B))
        J = c.download(g.FIELD_J).reshape(nz, ny, nx, 3)
        det = c.download(g.FIELD_DETJAC).reshape(nz + 2, ny + 2, nx + 2)
        wedge, convex = (c.download(f) for f in (g.FIELD_WEDGEMIN, g.FIELD_CONVEXITY))
    inner = (slice(1, -1),) * 3
    x, B, det = x[inner], B[inner], det[inner]
    b2 = (B * B).sum(-1)
    w = np.ones((nz, ny, nx))
    for axis in range(3):
        for side in (0, -1):
            np.moveaxis(w, axis, 0)[side] *= 0.5
    jxb, den = norm(np.cross(J, B)), norm(J) * np.sqrt(b2)
    want = {"B2": (b2 * det * w).sum() * p.dx * p.dy * p.dz, "JMax": norm(J).max(), "JxB_B2Max": (jxb / b2).max(),
            "JxBMax_JBMax": jxb.max() / den.max(), "wedgeMin": wedge.min(), "convex": convex.min()}
    lat = [np.arange(n) * h + o for n, h, o in ((nx, p.dx, p.Ox), (ny, p.dy, p.Oy), (nz, p.dz, p.Oz))]
    X, Y, Z = lat[0][None, None, :], lat[1][None, :, None], lat[2][:, None, None]
    f = np.exp(-(X * X + Y * Y) / p.ar ** 2 - Z * Z / p.az ** 2) * p.phi1
    d = [x[..., 0] - np.cos(f) * X - np.sin(f) * Y, x[..., 1] + np.sin(f) * X - np.cos(f) * Y, x[..., 2] - Z]
    want["errXb_XbAn"] = np.sqrt(sum((q * q).sum() for q in d) / b2.size)
    want["errB_1ez"] = np.sqrt(((B - (0, 0, 1)) ** 2).sum() / b2.size)
    col = (slice(None), ny // 2, nx // 2)
    a, z = ((J * B).sum(-1) / b2)[col], x[..., 2][col]
    with np.errstate(divide="ignore", invalid="ignore"):
        q = np.abs((a[:, None] - a[None]) / (z[:, None] - z[None]))
    want["epsilonStar"] = np.sqrt(2.0) * np.nanmax(np.where(z[:, None] == z[None], 0, q))
    sums = ("B2", "errB_1ez", "errXb_XbAn", "epsilonStar")
    for k, v in want.items():
        assert abs(getattr(res, k) - v) <= (1e-12 if k in sums else 1e-13) * abs(v), (k, getattr(res, k), v)
