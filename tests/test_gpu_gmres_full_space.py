"""GMRES cycles as long as the space and longer: the basis then spans the whole
space, so what the first pass of Gram-Schmidt leaves of w lies in it too, w.w -
h2.h2 cancels and the norm is formed again from w, in every step from the neq-th
on.  The cycle's solution is the system's: x against a dense solve, within the
rounding of a system whose condition number is below 1e4 (1e-12; 1e-10 here)."""
import numpy as np
import pytest

from elastic_amd import mesh as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("resident", [1, 0])
@pytest.mark.parametrize("kind,n,opts,more", [
    ("hex8", 1, {}, 0), ("hex8", 1, {}, 21), ("hex8", 2, {"tile_blocks": 32}, 0),
    ("hex8", 2, {"tile_blocks": 32}, 4), ("hex8", 2, {"tile_blocks": 32}, 20),
    ("quad4", 3, {"tile_blocks": 32}, 30),
])
def test_cycles_beyond_the_dimension(kind, n, opts, more, resident):
    from elastic_amd.solver import GMRES
    from elastic_amd.system import System

    s = System(M.hex8_cube(n, jitter=0.15, seed=n + 1) if kind == "hex8" else M.quad4_square(n))
    for k, v in dict(opts, resident=resident).items():
        s.ctx.set_option(k, v)
    ad, al = s.values()
    A = np.diag(ad)
    row = np.repeat(np.arange(s.neq), np.diff(s.ia))
    A[row, s.ja - 1] = A[s.ja - 1, row] = al
    exact = np.linalg.solve(A, s.b)
    for cycles in (1, 3):
        print("gmres full space", kind, n, more, resident, cycles, flush=True)
        got = [s.solve(solver=GMRES, tol=1e-300, maxit=cycles, ngram=s.neq + more, allow_maxit=True)
               for _ in range(2)]
        assert np.array_equal(got[0][0], got[1][0])
        assert np.linalg.norm(got[0][0] - exact) <= 1e-10 * np.linalg.norm(exact)
    s.ctx.close()
