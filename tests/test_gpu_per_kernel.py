"""A whole attempt of the per-kernel path (gm_step, with B of faces and inner
points in one launch, the current within the slope's launch and the stage
positions alternating between buffers) against the entry points called one by
one: the same operations in the same order, so every field agrees bit for
bit.  Grids at and beside the 256 points of a workgroup, every kind of
boundary."""
import numpy as np
import pytest

from conftest import evolved_state, small_braid

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def g(require_gpu):
    import glemur_amd
    return glemur_amd


P = {"pressure": True, "beta": 0.05}


@pytest.mark.parametrize("shape,kw", [((2, 2, 2), {}), ((16, 16, 17), P), ((17, 19, 23), {"xPeri": True, **P}),
                                      ((9, 8, 31), {"yPeri": True, "zPeri": True}),
                                      ((13, 12, 11), {"xPeri": True, "yPeri": True, "zPeri": True, **P})])
def test_step_equals_single_calls(g, shape, kw):
    p = small_braid(*shape, inertia=True, nu=0.6, **kw)
    B0, xb = evolved_state(p, 2)
    uu = np.random.default_rng(4).normal(size=3 * p.ninner) * 1e-3
    dt = 1e-3
    with g.Context(p, g.PREC_F64) as a, g.Context(p, g.PREC_F64) as b:
        for c in (a, b):
            c.upload(B0, xb, 0.0, dt)
            c.upload_velocity(uu)
        for n in range(6):
            a.b_jacb0()
            a.set_bbound()
            a.set_peri_B()
            a.current()
            if p.pressure:
                a.gradp()
            a.rk_kk(n, dt)
        md = a.rk_xnewstar()
        stage = a.download(g.FIELD_XB)
        a.accept()
        s = b.step()
        assert s.accepted and s.maxDelta == md
        for f in (g.FIELD_XB, g.FIELD_B, g.FIELD_J, g.FIELD_KK, g.FIELD_UU, g.FIELD_DETJAC):
            assert np.array_equal(a.download(f), b.download(f)), f
    # a rejected attempt leaves the positions of the last stage
    p.maxError = md / 2
    with g.Context(p, g.PREC_F64) as b:
        b.upload(B0, xb, 0.0, dt)
        b.upload_velocity(uu)
        assert not b.step().accepted
        assert np.array_equal(b.download(g.FIELD_XB), stage)
