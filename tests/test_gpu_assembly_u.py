"""b = b0 - K u of hex8 at nonzero displacements, with and without K, bit for
bit: the oracle's element products s u (elmt07_mec isw 2) subtracted colour by
colour, as the reference's coloured loop does.  1 to 6 elements a side, so
colours of one element, of fewer than a workgroup's and of more."""
import numpy as np
import pytest

from elastic_amd import mesh as M
from oracle import binding as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 3, 6])
def test_hex8_residual_at_displacements(n):
    from elastic_amd.system import System

    m = M.hex8_cube(n, jitter=0.15, seed=n, E=1.7, nu=0.23)
    u = np.random.default_rng(n).standard_normal((m.nnode, 3))
    s = System(m)
    ad0, al0 = s.values()
    b = s.assemble(u).copy()
    ad1, al1 = s.values()
    assert np.array_equal(ad0, ad1) and np.array_equal(al0, al1)
    ncol, color = O.colormsh(m)
    order, _ = O.setcolor(color, ncol)
    ref = s.b0.copy()
    for el in order - 1:
        nodes = m.ix[el, :8] - 1
        rc, _, p = O.element(7, 2, m.e[0], np.zeros(7, np.int32), m.x[nodes].ravel(),
                             u[nodes].ravel(), 3, 24)
        assert rc == 0
        eq = s.idn[nodes].ravel()
        ref[eq[eq > 0] - 1] -= p[eq > 0]
    assert np.array_equal(b, ref)
    b2 = s.b0.copy()
    s._assemble(2, 0, 1, np.ascontiguousarray(u), b2)  # the residual alone
    assert np.array_equal(b2, ref)
    s.ctx.close()
