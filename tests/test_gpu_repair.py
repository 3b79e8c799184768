"""GPU test of the TE / ED non-negativity repair around the list length up to
which one workgroup does it in LDS (4096 cells) and at its smallest lists,
against the in-order sweep in numpy: same bits, and the number of cells."""
import numpy as np
import pytest

from minicombust_app_amd import mcflow as mc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,count", [(1, 0), (1, 2), (2, 16), (5, 1), (5, 250), (16, 4095), (16, 4096), (16, 4097),
                                     (16, 8192), (21, 1023), (21, 1025)])
def test_repair_counts(m, count):
    print("repair m=%d count=%d" % (m, count), flush=True)
    with mc.Context(m) as g:
        rng = np.random.default_rng(100 * m + count)
        v = rng.random(g.N + 6) + 1e-3
        neg = rng.choice(g.N, count, replace=False)
        v[neg] *= -1.0
        nbr = g.get(mc.ARR_CELL_NEIGHBOURS).reshape(g.N, 6)
        want = v.copy()
        for c in np.sort(neg):
            s, k = 0.0, 0
            for nb in nbr[c]:
                if nb < g.N:
                    s += want[nb] if nb < c else v[nb]
                    k += 1
            want[c] = max(s / k, 1e-12)
        before = g.stats()["clip_cells"]
        g.set(mc.ARR_PHI + mc.TE, v)
        g.repair_nonneg(mc.TE)
        assert np.array_equal(g.phi(mc.TE), want)
        assert g.stats()["clip_cells"] - before == count
