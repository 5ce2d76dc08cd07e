"""Limits of a run: n_cycle <= 0 takes params.nCycle, and with that at zero
or below no accepted step is left, so the run ends with its first attempt
(as an ensemble's does); single steps have no limits."""
import pytest

from conftest import small_braid

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def g(require_gpu):
    import glemur_amd
    return glemur_amd


@pytest.mark.parametrize("ncycle", [0, -3])
@pytest.mark.parametrize("prec,kw", [("F64", {}), ("F32K", {}), ("F64", {"inertia": True, "nu": 0.6})])
def test_no_cycles_left(g, prec, kw, ncycle):
    p = small_braid(**kw)
    p.nCycle = ncycle
    B0, xb = g.init_state(p)
    with g.Context(p, getattr(g, "PREC_" + prec)) as c:
        c.upload(B0, xb, 0.0, 0.01)
        for n in (1, 2):
            st = c.run(max_attempts=6, batch=2, use_graph=n == 2)
            assert st.n_attempt == n and st.stopped
        c.step()
        assert c.run(max_attempts=6).n_attempt == 4
    if not kw:
        with g.Batch([p], getattr(g, "PREC_" + prec)) as b:
            b.members[0].upload(B0, xb, 0.0, 0.01)
            assert [b.run(max_attempts=6, batch=2)[0].n_attempt for _ in range(2)] == [1, 2]
