"""GPU tests of passes that replace plainer ones bit for bit, each with the form
that runs asserted, so that a fallback cannot pass in its place.

Regular matched levels (boxes of even sides under a momentum diagonal that
varies along x only) against their index arrays; the V-cycle's one-workgroup
tails against per-pass launches, over the storages and sweep counts they take;
reductions finished by their consumer against the finishing kernels; the box
assembly kernels against the general ones under the options the default test
leaves out."""
import numpy as np
import pytest

from minicombust_app_amd import mcflow as mc
from tests.helpers import assert_bits

pytestmark = pytest.mark.gpu

FIELDS = [mc.U, mc.V, mc.W, mc.P, mc.TE, mc.ED, mc.TEM, mc.FUL, mc.PRO, mc.VARF, mc.VARP]
ARRAYS = [mc.ARR_AU, mc.ARR_AV, mc.ARR_SU, mc.ARR_SV, mc.ARR_SW, mc.ARR_FF0, mc.ARR_FF1, mc.ARR_MFLUX, mc.ARR_A_VALS,
          mc.ARR_PA_VALS, mc.ARR_PB]


def _context(m, psolve, **kw):
    g = mc.Context(m, mode=mc.MODE_SIMPLE, psolve=psolve, p_rtol=1e-8, **kw)
    x = np.arange(g.N) % (2 * m)
    g.set(mc.ARR_AU, np.concatenate([10.0 + 3.0 * np.exp(-0.2 * x), np.zeros(6)]))
    g.pressure_assemble()
    b = np.random.default_rng(m).standard_normal(g.N)
    return g, b - b.mean()


# m: levels that are halved boxes; at 52 and 64 the second passes 32,768 rows
REGULAR = {8: 1, 10: 1, 12: 1, 16: 2, 18: 1, 20: 2, 32: 3, 36: 2, 52: 2, 64: 4}


@pytest.mark.parametrize("psolve,half", [(mc.PSOLVE_FP64, 1), (mc.PSOLVE_MIXED, 1), (mc.PSOLVE_MIXED, 0)])
@pytest.mark.parametrize("m", sorted(REGULAR))
def test_regular_transfers_same_bits(m, psolve, half):
    print("regular transfers m=%d psolve=%d half=%d" % (m, psolve, half), flush=True)
    g, b = _context(m, psolve, amg_half=half, amg_tail=0)
    with g:
        g.plain_passes(mc.PLAIN_TRANSFERS)
        want, st0 = g.solve_pressure(b)
        levels = [g.amg_level(l) for l in range(g.forms()["amg_levels"])]
        assert sum(k == mc.LEVEL_REGULAR for _, _, k in levels) == REGULAR[m], levels
        g.plain_passes(0)
        got, st1 = g.solve_pressure(b)
        assert st0.converged and st1.iterations == st0.iterations
        assert_bits(got, want, "pressure correction, coordinates vs index arrays")


# diagonal storage (one, two and four rows a thread), a mixture, CSR
TAILS = [(10, mc.TAIL_DIA), (14, mc.TAIL_DIA), (20, mc.TAIL_DIA), (24, mc.TAIL_DIA), (32, mc.TAIL_DIA),
         (18, mc.TAIL_MIXED), (36, mc.TAIL_MIXED), (11, mc.TAIL_CSR), (19, mc.TAIL_CSR), (33, mc.TAIL_CSR)]


@pytest.mark.parametrize("psolve", [mc.PSOLVE_FP64, mc.PSOLVE_MIXED])
@pytest.mark.parametrize("m,form,nu", [(m, f, 3) for m, f in TAILS] +
                         [(m, f, nu) for m, f in [(20, mc.TAIL_DIA), (18, mc.TAIL_MIXED), (33, mc.TAIL_CSR)]
                          for nu in (1, 2, 4, 5)])
def test_matched_tail_same_bits(m, form, nu, psolve):
    print("matched tail m=%d form=%d nu=%d psolve=%d" % (m, form, nu, psolve), flush=True)
    key = "tail32" if psolve == mc.PSOLVE_MIXED else "tail64"
    g, b = _context(m, psolve, amg_tail=0, amg_nu=nu)
    with g:
        want, st0 = g.solve_pressure(b)
        assert g.forms()[key] == mc.TAIL_NONE
        g.set_options(amg_tail=1)
        got, st1 = g.solve_pressure(b)
        assert g.forms()[key] == form
        assert st0.converged and st1.iterations == st0.iterations
        assert_bits(got, want, "pressure correction, tail vs per-pass launches")


def _same_runs(a, b, iterations):
    for it in range(iterations):
        for c in (a, b):
            c.simple_iteration(it)
        for i in [mc.ARR_PHI + f for f in FIELDS] + [mc.ARR_GRAD + f for f in FIELDS] + ARRAYS:
            assert_bits(a.get(i), b.get(i), "array %d after iteration %d" % (i, it))


@pytest.mark.parametrize("mode,psolve", [(mc.MODE_SIMPLE, mc.PSOLVE_FP64), (mc.MODE_SIMPLE, mc.PSOLVE_MIXED),
                                         (mc.MODE_COMPAT, mc.PSOLVE_FP64)])
@pytest.mark.parametrize("m", [1, 2, 5, 12, 40])
def test_folded_finishes_same_bits(m, mode, psolve):
    print("folded finishes m=%d mode=%d psolve=%d" % (m, mode, psolve), flush=True)
    with mc.Context(m, mode=mode, psolve=psolve) as a, mc.Context(m, mode=mode, psolve=psolve) as b:
        b.plain_passes(mc.PLAIN_FINISH)
        _same_runs(a, b, 3)
        sa, sb = a.stats(), b.stats()
        assert [sa[k] for k in ("mom_iters", "scalar_iters", "p_iters")] == [sb[k] for k in
                                                                            ("mom_iters", "scalar_iters", "p_iters")]


@pytest.mark.parametrize("kw", [dict(psolve=mc.PSOLVE_MIXED), dict(psolve=mc.PSOLVE_MIXED, amg_half=0),
                                dict(solve_scalars=0), dict(limit_grad=1),
                                dict(psolve=mc.PSOLVE_MIXED, p_rtol=1e-10), dict(warm_start=0)],
                         ids=lambda kw: "-".join("%s%g" % i for i in kw.items()))
@pytest.mark.parametrize("m", [2, 5, 12, 33])
def test_box_assembly_under_options(m, kw):
    print("box assembly m=%d %s" % (m, kw), flush=True)
    with mc.Context(m, mode=mc.MODE_SIMPLE, **kw) as a, mc.Context(m, mode=mc.MODE_SIMPLE, **kw) as b:
        b.set(mc.ARR_CELL_DENSITY, b.get(mc.ARR_CELL_DENSITY))
        assert a.forms()["box_tables"] == 1 and b.forms()["box_tables"] == 0
        rng = np.random.default_rng(m)
        for f in FIELDS:
            v = a.phi(f) * (1.0 + 0.1 * rng.standard_normal(a.N + 6)) + 1e-3 * rng.random(a.N + 6)
            for c in (a, b):
                c.set(mc.ARR_PHI + f, v)
        _same_runs(a, b, 3)


@pytest.mark.parametrize("m", [2, 3, 5, 12, 20, 33, 64])
def test_generated_boxes_use_the_tables(m):
    print("box tables m=%d" % m, flush=True)
    with mc.Context(m) as g:
        assert g.forms()["box_tables"] == 1


def test_refused_geometry_leaves_the_tables_in_use():
    """A geometry array set with a wrong count is refused and changes nothing."""
    print("refused geometry", flush=True)
    with mc.Context(5) as g:
        v = g.get(mc.ARR_CELL_DENSITY)
        for n in (0, g.N - 1, g.N + 1):
            assert g.L.mc_array_set(g.h, mc.ARR_CELL_DENSITY, v.ctypes.data, n) != mc.MC_OK
        assert g.L.mc_array_set(g.h, mc.ARR_CELL_DENSITY, None, g.N) != mc.MC_OK
        assert g.forms()["box_tables"] == 1
        g.set(mc.ARR_CELL_DENSITY, v)
        assert g.forms()["box_tables"] == 0
