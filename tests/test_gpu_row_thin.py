"""Row reductions of grids with fewer columns than a workgroup has threads,
where groups of threads share the planes: against numpy on the fields the
context holds, and no slower than a compact grid of as many points.

The operations per point are the same; sums are reordered (at most 1.2e6
terms of one sign: 1e-12 relative), quotients and roots may differ by a few
last bits (1e-13 relative for maxima)."""
import time

import numpy as np
import pytest

from conftest import small_braid

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def g(require_gpu):
    import glemur_amd
    return glemur_amd


ROW = {k: True for k in ("redB2", "redJMax", "redJxB_B2Max", "redConvex", "redWedgeMin", "redErrB_1ez", "redErrXb_XbAn")}


# one plane a group and several, a last group without planes, groups of one
# and of nearly all threads
@pytest.mark.parametrize("prec", ["F64", "F32K"])
@pytest.mark.parametrize("shape", [(2, 2, 50), (2, 3, 700), (5, 17, 33), (16, 8, 9001), (3, 85, 40)])
def test_thin_grids(g, prec, shape):
    nx, ny, nz = shape
    p = small_braid(*shape, **ROW)
    B0, xb = g.init_state(p)
    x = xb.reshape(nz + 2, ny + 2, nx + 2, 3).copy()
    r = np.random.default_rng(5)
    x[1:-1, 1:-1, 1:-1] += r.uniform(-0.1, 0.1, (nz, ny, nx, 3)) * (p.dx, p.dy, p.dz)
    with g.Context(p, getattr(g, "PREC_" + prec)) as c:
        c.upload(B0, x.reshape(-1), 0.0, 0.01)
        c.fields()
        res = c.reductions()
        B = c.download(g.FIELD_B).reshape(nz + 2, ny + 2, nx + 2, 3)[1:-1, 1:-1, 1:-1]
        J = c.download(g.FIELD_J).reshape(nz, ny, nx, 3)
        det = c.download(g.FIELD_DETJAC).reshape(nz + 2, ny + 2, nx + 2)[1:-1, 1:-1, 1:-1]
        wedge, convex = (c.download(f) for f in (g.FIELD_WEDGEMIN, g.FIELD_CONVEXITY))
    b2 = (B * B).sum(-1)
    w = np.ones((nz, ny, nx))
    for axis in range(3):
        for side in (0, -1):
            np.moveaxis(w, axis, 0)[side] *= 0.5
    norm = lambda a: np.sqrt((a * a).sum(-1))
    assert wedge.size == nx * ny * nz
    want = {"JMax": norm(J).max(), "JxB_B2Max": (norm(np.cross(J, B)) / b2).max(), "wedgeMin": wedge.min(),
            "convex": convex.min()}
    for k, v in want.items():
        assert abs(getattr(res, k) - v) <= 1e-13 * abs(v), k
    sums = {"B2": (b2 * det * w).sum() * p.dx * p.dy * p.dz,
            "errB_1ez": np.sqrt(((B - (0, 0, 1)) ** 2).sum() / b2.size)}
    for k, v in sums.items():
        assert abs(getattr(res, k) - v) <= 1e-12 * abs(v), k


def test_thin_grid_takes_no_longer(g):
    """2 x 2 x 50000 points against 58 x 58 x 60 (as many): the same work, so
    at most 1.5 times as long (a thread a column took 6.7 times)."""
    t = []
    for shape in ((58, 58, 60), (2, 2, 50000)):
        p = small_braid(*shape, **ROW)
        B0, xb = g.init_state(p)
        with g.Context(p, g.PREC_F64) as c:
            c.upload(B0, xb, 0.0, 0.01)
            c.fields()
            c.reductions()
            ts = []
            for _ in range(30):
                t0 = time.perf_counter()
                c.reductions()
                ts.append(time.perf_counter() - t0)
            t.append(min(ts))
    print("us a row", [round(v * 1e6, 1) for v in t])
    assert t[1] <= 1.5 * t[0]
