"""GPU test of the generated box's assembly kernels (closed-form neighbours,
geometry from per-axis tables) against the general ones: setting a geometry
array, here to the values it holds, puts a context on the general kernels.
Both form the same sums in the same order, so everything is compared bit for
bit.  Modifiers: the smallest box, rows shorter and longer than a wavefront,
rows that end in the middle of a brick, several y chunks."""
import numpy as np
import pytest

from minicombust_app_amd import mcflow as mc

pytestmark = pytest.mark.gpu

FIELDS = [mc.U, mc.V, mc.W, mc.P, mc.TE, mc.ED, mc.TEM, mc.FUL, mc.PRO, mc.VARF, mc.VARP]
ARRAYS = [mc.ARR_AU, mc.ARR_AV, mc.ARR_SU, mc.ARR_SV, mc.ARR_SW, mc.ARR_FF0, mc.ARR_FF1, mc.ARR_MFLUX,
          mc.ARR_A_VALS, mc.ARR_PA_VALS, mc.ARR_PB]


def same(a, b, arrays, where):
    for i in arrays:
        x, y = a.get(i), b.get(i)
        assert np.array_equal(x.view(np.uint64), y.view(np.uint64)), (where, i, np.abs(x - y).max())


@pytest.mark.parametrize("mode", [mc.MODE_SIMPLE, mc.MODE_COMPAT])
@pytest.mark.parametrize("m", [2, 3, 5, 12, 33])
def test_box_assembly_same_bits(m, mode):
    print("box assembly m=%d mode=%d" % (m, mode), flush=True)
    with mc.Context(m, mode=mode) as a, mc.Context(m, mode=mode) as b:
        b.set(mc.ARR_CELL_DENSITY, b.get(mc.ARR_CELL_DENSITY))
        rng = np.random.default_rng(m)
        for f in FIELDS:
            v = a.phi(f) * (1.0 + 0.1 * rng.standard_normal(a.N + 6)) + 1e-3 * rng.random(a.N + 6)
            a.set(mc.ARR_PHI + f, v)
            b.set(mc.ARR_PHI + f, v)
        state = [mc.ARR_PHI + f for f in FIELDS] + [mc.ARR_GRAD + f for f in FIELDS] + ARRAYS
        for c in (a, b):
            c.get_phi_gradients()
            c.set_up_field()
            c.momentum_assemble()
        # the pressure system is first written by the iteration's assembly
        same(a, b, [i for i in state if i not in (mc.ARR_PA_VALS, mc.ARR_PB)], "momentum")
        for it in range(3):
            for c in (a, b):
                c.simple_iteration(it)
            same(a, b, state, "iteration %d" % it)
