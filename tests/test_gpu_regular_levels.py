"""GPU test of the matched pressure hierarchy on boxes of even sides, whose
levels are halved boxes and take transfers without index arrays: from boxes
with one smoothed level to sizes where the second level passes 32,768 rows.

The transfers reproduce the index-array passes' bits, so the PCG's iteration
counts are the ones those passes gave; the residual is formed by numpy from the
library's matrix and stays within 1 % of the tolerance (the recursion leaves the
true residual by rounding, about 1e-15 an iteration)."""
import numpy as np
import pytest
import scipy.sparse as sp

from minicombust_app_amd import mcflow as mc

pytestmark = pytest.mark.gpu

ITERATIONS = {2: (1, 2), 4: (1, 2), 8: (10, 11), 12: (11, 12), 16: (14, 15), 20: (16, 17), 32: (18, 19), 52: (19, 21)}


@pytest.mark.parametrize("psolve", [mc.PSOLVE_FP64, mc.PSOLVE_MIXED])
@pytest.mark.parametrize("m", sorted(ITERATIONS))
def test_regular_levels(m, psolve):
    print("regular levels m=%d psolve=%d" % (m, psolve), flush=True)
    with mc.Context(m, mode=mc.MODE_SIMPLE, psolve=psolve, p_rtol=1e-8) as g:
        x = np.arange(g.N) % (2 * m)
        g.set(mc.ARR_AU, np.concatenate([10.0 + 3.0 * np.exp(-0.2 * x) + 0.01 * np.sin(np.arange(g.N)), np.zeros(6)]))
        g.pressure_assemble()
        b = np.random.default_rng(m).standard_normal(g.N)
        b -= b.mean()
        A = sp.csr_matrix((g.get(mc.ARR_PA_VALS), g.get(mc.ARR_COL), g.get(mc.ARR_ROW_PTR)), shape=(g.N, g.N))
        sol, st = g.solve_pressure(b)
        assert st.converged
        assert st.iterations == ITERATIONS[m][0 if psolve == mc.PSOLVE_FP64 else 1]
        r = b - A @ sol[:g.N]
        assert np.linalg.norm(r - r.mean()) <= 1.01e-8 * np.linalg.norm(b)
