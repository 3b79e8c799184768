"""GPU test of the Krylov reductions over their grids' range: one block, a few,
and both sides of the count up to which a reduction is finished by the kernel
that needs it (512 blocks of 256 rows: modifier 40 has 500, 41 has 539).

The three momentum systems are solved to 1e-10 from zero and from the current
field and the residual is formed by numpy from the library's matrix; BiCGStab's
recursive residual leaves the true one by rounding (about 1e-15 per iteration,
a few tens of iterations), so 1 % on top of the tolerance holds it."""
import numpy as np
import pytest
import scipy.sparse as sp

from minicombust_app_amd import mcflow as mc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("warm", [0, 1])
@pytest.mark.parametrize("m", [1, 2, 5, 11, 40, 41])
def test_momentum_residual(m, warm):
    print("momentum residual m=%d warm=%d" % (m, warm), flush=True)
    with mc.Context(m, mode=mc.MODE_SIMPLE, mom_rtol=1e-10, warm_start=warm) as g:
        rng = np.random.default_rng(m)
        for f in (mc.U, mc.V, mc.W):
            g.set(mc.ARR_PHI + f, g.phi(f) + rng.standard_normal(g.N + 6))
        g.get_phi_gradients()
        g.set_up_field()
        g.momentum_assemble()
        A = sp.csr_matrix((g.get(mc.ARR_A_VALS), g.get(mc.ARR_COL), g.get(mc.ARR_ROW_PTR)), shape=(g.N, g.N))
        rhs = [g.get(a)[:g.N].copy() for a in (mc.ARR_SU, mc.ARR_SV, mc.ARR_SW)]
        st = g.momentum_solve()
        assert st.converged
        for f, b in zip((mc.U, mc.V, mc.W), rhs):
            r = b - A @ g.phi(f)[:g.N]
            assert np.linalg.norm(r) <= 1.01e-10 * np.linalg.norm(b), (f, np.linalg.norm(r) / np.linalg.norm(b))
