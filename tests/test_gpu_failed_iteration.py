"""GPU test of the state an iteration leaves when one of its solves does not
converge: on the generated box, whose assembly kernels leave out stores that a
later stage overwrites, the arrays are the failed stage's own, as the general
kernels store them (a context whose geometry was set, here to the values it
holds, runs those).

A solve is made to fail by an iteration limit it cannot meet, a scalar's by a
NaN in a boundary slot of its field, which only that field's gradient reads.
There the right-hand side is left out: the general kernels multiply every
component of a neighbour's gradient, the box kernels those along the normal, so
a NaN reaches fewer of their cells."""
import numpy as np
import pytest

from minicombust_app_amd import mcflow as mc

pytestmark = pytest.mark.gpu

ARRAYS = [mc.ARR_AU, mc.ARR_AV, mc.ARR_SV, mc.ARR_SW, mc.ARR_FF0, mc.ARR_FF1, mc.ARR_MFLUX, mc.ARR_A_VALS,
          mc.ARR_PA_VALS, mc.ARR_PB]


def _same(x, y):
    return np.array_equal(x.view(np.uint64), y.view(np.uint64))


@pytest.mark.parametrize("mode", [mc.MODE_SIMPLE, mc.MODE_COMPAT])
# (at m = 2 every cell is a wall cell, whose ED row has no gradient, and the
# pressure solve is the dense one, which meets any tolerance in one iteration)
@pytest.mark.parametrize("stage,m", [("momentum", 2), ("momentum", 5), ("momentum", 12), ("pressure", 5),
                                     ("pressure", 12), ("TE", 2), ("TE", 5), ("TE", 12), ("ED", 5), ("ED", 12),
                                     ("TEM", 2), ("TEM", 5), ("TEM", 12)])
def test_arrays_after_a_failed_solve(stage, m, mode):
    print("failed %s m=%d mode=%d" % (stage, m, mode), flush=True)
    nan = stage in ("TE", "ED", "TEM")
    what = "scalar" if nan else stage
    # the compatible form solves the pressure system in its first iteration only
    good = 0 if stage == "pressure" and mode == mc.MODE_COMPAT else 2
    with mc.Context(m, mode=mode) as a, mc.Context(m, mode=mode) as b:
        b.set(mc.ARR_CELL_DENSITY, b.get(mc.ARR_CELL_DENSITY))
        rng = np.random.default_rng(m)
        for f in (mc.U, mc.V, mc.W, mc.P, mc.TE, mc.ED, mc.TEM):
            v = a.phi(f) * (1.0 + 0.1 * rng.standard_normal(a.N + 6)) + 1e-3 * rng.random(a.N + 6)
            for c in (a, b):
                c.set(mc.ARR_PHI + f, v)
        for c in (a, b):
            for it in range(good):
                c.simple_iteration(it)
            if stage == "momentum":
                c.set(mc.ARR_PHI + mc.U, 50.0 * rng.standard_normal(c.N + 6) if c is a else a.phi(mc.U))
                c.set_options(mom_maxit=1, mom_rtol=1e-15)
            elif stage == "pressure":
                c.set_options(p_maxit=1, p_rtol=1e-14)
            else:
                f = {"TE": mc.TE, "ED": mc.ED, "TEM": mc.TEM}[stage]
                v = c.phi(f)
                v[c.N:] = np.nan
                c.set(mc.ARR_PHI + f, v)
        for c in (a, b):
            with pytest.raises(mc.MCError, match=what):
                c.simple_iteration(good)
        for i in ARRAYS + ([] if nan else [mc.ARR_SU]):
            x, y = a.get(i), b.get(i)
            assert _same(x, y), (i, int((x != y).sum()), np.abs(x - y).max())
