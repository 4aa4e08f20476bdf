"""Checks that go with new values: the first zero on the diagonal of an
assembled K (found on the device), and a pattern of the last one's sizes but
other contents in the solver call (compared while the values go up)."""
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


def test_solver_call_with_another_pattern_of_the_same_sizes():
    from elastic_amd.solver import solv

    def dense(cols, ad, al):
        A = np.diag(ad)
        for r, c in enumerate(cols, 1):
            A[r, c] = A[c, r] = al[r - 1]
        return A

    rng = np.random.default_rng(1)
    for cols in ((0, 1, 2), (0, 0, 1), (0, 1, 2), (0, 1, 0)):
        ia, ja = np.array([1, 1, 2, 3, 4], np.int32), np.array(cols, np.int32) + 1
        ad, al, b = 4.0 + rng.random(4), rng.random(3), rng.random(4)
        m, x = np.zeros(4), np.zeros(4)
        solv(4, 3, ia, ja, ad, al, m, b, x, tol=1e-13)
        ref = np.linalg.solve(dense(cols, ad, al), b)
        # condition below 4, stop at 1e-13
        assert np.linalg.norm(x - ref) <= 1e-11 * np.linalg.norm(ref)
        assert np.array_equal(m, 1.0 / ad)
