"""GPU test that the pressure hierarchy follows the context's current options,
not those of its first solve: solves to 1e-9 and below without the limiter take
the halved box levels, the others the matched ones, whatever was set before.
Both contexts build from the same matrix, so a context that was switched and a
fresh one do the same arithmetic and are compared bit for bit."""
import numpy as np
import pytest

from minicombust_app_amd import mcflow as mc
from tests.helpers import assert_bits

pytestmark = pytest.mark.gpu


def _solve(g):
    n = np.arange(g.N)
    g.set(mc.ARR_AU, np.concatenate([10.0 + 3.0 * np.exp(-0.2 * (n % 18)) + 0.01 * np.sin(n), np.zeros(6)]))
    g.pressure_assemble()
    b = np.random.default_rng(9).standard_normal(g.N)
    x, st = g.solve_pressure(b - b.mean())
    assert st.converged
    return x.copy(), st.iterations


@pytest.mark.parametrize("psolve,graph", [(mc.PSOLVE_FP64, 0), (mc.PSOLVE_MIXED, 0), (mc.PSOLVE_FP64, 1)])
@pytest.mark.parametrize("before,after", [
    (dict(p_rtol=1e-8), dict(p_rtol=1e-10)),
    (dict(p_rtol=1e-10), dict(p_rtol=1e-8)),
    (dict(p_rtol=1e-10, limit_grad=0), dict(p_rtol=1e-10, limit_grad=1)),
    (dict(p_rtol=1e-10, limit_grad=1), dict(p_rtol=1e-10, limit_grad=0)),
])
def test_hierarchy_follows_the_options(before, after, psolve, graph):
    print("hierarchy %s -> %s psolve=%d graph=%d" % (before, after, psolve, graph), flush=True)
    with mc.Context(9, mode=mc.MODE_SIMPLE, psolve=psolve, pcg_graph=graph, **after) as g:
        want, its = _solve(g)
    with mc.Context(9, mode=mc.MODE_SIMPLE, psolve=psolve, pcg_graph=graph, **before) as g:
        _solve(g)
        g.set_options(**after)
        got, n = _solve(g)
        assert n == its
        assert_bits(got, want, "pressure correction after the options changed")
        assert g.stats()["amg_setups"] == 2


def test_hierarchy_kept_while_the_choice_stands():
    print("hierarchy kept", flush=True)
    with mc.Context(9, mode=mc.MODE_SIMPLE, p_rtol=1e-8) as g:
        _solve(g)
        for kw in (dict(p_rtol=1e-7), dict(limit_grad=1), dict(p_rtol=1e-10), dict(p_rtol=1e-8, limit_grad=0)):
            g.set_options(**kw)   # never both a tight tolerance and no limiter
            _solve(g)
        g.set_options(p_rtol=1e-10)
        g.set_options(p_rtol=1e-8)   # and back before the next solve
        _solve(g)
        assert g.stats()["amg_setups"] == 1
