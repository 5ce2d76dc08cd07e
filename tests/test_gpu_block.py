"""Stage kernels that compute blocks of points at once (small grids) against
the marching kernels.

Every point takes the same floating-point operations in the same order in
both, so positions (hi and lo words), t, dt, error maxima, decisions and the
criteria agree bit for bit; the energy is the same sum in another order
(1e-12 relative: at most 10^5 terms of one sign, rounded once each).  The
marching run is the one whose tiles the caller sets."""
import numpy as np
import pytest

from conftest import evolved_state, small_braid

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def g(require_gpu):
    import glemur_amd
    return glemur_amd


P = {"pressure": True, "beta": 0.05}
# grids smaller than a block, one point past one, long thin ones in each
# direction, and one of several blocks a CU; every variant of the kernels
CASES = [
    ((2, 2, 2), {}), ((3, 2, 5), P), ((9, 8, 8), {}), ((17, 16, 33), {"epsilonProf": True}),
    ((61, 3, 4), {}), ((3, 61, 4), P), ((4, 3, 90), {"zUpdate": False}),
    ((24, 19, 31), {"xPeri": True}), ((24, 19, 31), {"yPeri": True, **P}), ((13, 18, 16), {"zPeri": True}),
    ((15, 14, 17), {"xPeri": True, "yPeri": True, "zPeri": True, "epsilonProf": True, **P}),
    ((21, 18, 20), {"initDist": b"initShearX", "initShearA": 0.05, "initShearB": 0.02, **P}),
    ((52, 47, 60), {}),
]


@pytest.mark.parametrize("prec", ["F64", "F32K"])
@pytest.mark.parametrize("shape,kw", CASES)
def test_blocks_equal_the_march(g, prec, shape, kw):
    p = small_braid(*shape, **kw)
    p.nCycle = 10 ** 6
    B0, xb = evolved_state(p, 2)
    res = []
    for tile in (None, (6, 5, 4)):
        with g.Context(p, getattr(g, "PREC_" + prec)) as c:
            if tile:
                c.set_tile(*tile)
            c.upload(B0, xb, 0.0, 0.01)
            c.run(max_attempts=6, batch=3, use_graph=tile is None)
            res.append((c.download(g.FIELD_XB), c.download(g.FIELD_XB_LO), c.time(), c.step_log(6)))
    a, b = res
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1]) and a[2] == b[2]
    assert len(a[3]) == len(b[3]) == 6
    for r, q in zip(a[3], b[3]):
        assert (r.maxDelta, r.dt_used, r.accepted, r.ratio, r.ratio_pt, r.jxb_b2, r.jmax) == \
               (q.maxDelta, q.dt_used, q.accepted, q.ratio, q.ratio_pt, q.jxb_b2, q.jmax)
        assert abs(r.energy - q.energy) <= 1e-12 * abs(q.energy)
