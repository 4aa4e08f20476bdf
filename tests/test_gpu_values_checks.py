"""Checks that go with new values: the first zero on the diagonal of an
assembled K, found on the device."""
import numpy as np
import pytest

from elastic_amd import mesh as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("first", [0, 4, 17, None])
def test_assembled_zero_diagonal(first):
    """elements from `first` on have no stiffness: the first equation that only
    they touch is named, before and after a K without zeros"""
    from elastic_amd.solver import ElasticError
    from elastic_amd.system import System

    m = M.hex8_cube(3, jitter=0.1, seed=2)
    m.e, m.ie = np.concatenate([m.e, m.e]), np.concatenate([m.ie, m.ie])
    m.e[1, 0] = 0.0
    if first is not None:
        m.ix[first:, 8] = 2
    s = System(m)
    for _ in range(2):
        s.assemble()
        ad, _ = s.values()
        zero = np.flatnonzero(ad == 0.0)
        assert (len(zero) > 0) == (first is not None)
        if len(zero):
            with pytest.raises(ElasticError, match="at equation %d$" % (zero[0] + 1)):
                s.solve()
        else:
            x, st = s.solve()
            assert st["status"] == 0
    s.ctx.close()
