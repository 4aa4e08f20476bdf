"""GMRES's passes over the Krylov basis at the sizes where their workgroup shape
changes (rows per lane and groups of wavefronts per workgroup, 16,384 / 32,768 /
65,536 / 524,288 equations) and at cycle lengths around four and sixteen basis
vectors.  After one cycle of k steps x is the minimiser of ||M (b - A x)|| over
the Krylov space, whatever the orthogonalization; it is compared with an
Arnoldi process (modified Gram-Schmidt, least squares) in numpy on the same
products.  Both carry rounding of a few eps times the condition of the k-step
least-squares problem (below 1e4 for these k), so 1e-9 relative L2 holds with
room."""
import numpy as np
import pytest

from elastic_amd import mesh as M

pytestmark = pytest.mark.gpu


def _one_cycle(ctx, b, apply_m, k):
    g = apply_m(b)
    beta = np.linalg.norm(g)
    G, H = [g / beta], np.zeros((k + 1, k))
    for i in range(k):
        w = apply_m(ctx.spmv(G[i]))
        for _ in range(2):
            for j in range(i + 1):
                h = w @ G[j]
                H[j, i] += h
                w = w - h * G[j]
        H[i + 1, i] = np.linalg.norm(w)
        G.append(w / H[i + 1, i])
    rhs = np.zeros(k + 1)
    rhs[0] = beta
    y = np.linalg.lstsq(H, rhs, rcond=None)[0]
    return sum(y[j] * G[j] for j in range(k))


@pytest.mark.parametrize("n,k,precond", [(5, 1, 2), (5, 3, 6), (16, 4, 2), (17, 5, 6), (20, 17, 2),
                                         (26, 16, 2), (30, 19, 6), (56, 6, 2)])
def test_one_cycle_is_the_krylov_minimiser(n, k, precond):
    from elastic_amd.solver import GMRES
    from elastic_amd.system import System

    print("gmres basis", n, k, precond, flush=True)
    s = System(M.hex8_cube(n, jitter=0.15, seed=n))
    ad, _ = s.values()
    x, st = s.ctx.solve(s.b, solver=GMRES, precond=precond, tol=1e-30, maxit=1, ngram=k,
                        allow_maxit=True)
    assert st["iters"] == k and st["outer"] == 1
    if precond == 2:
        def apply_m(v):
            return v / ad
    else:  # 3x3 blocks of consecutive equations: c11 c22 c33 c21 c31 c32
        c = s.ctx.get_bdiag().reshape(-1, 6)
        full = np.stack([c[:, [0, 3, 4]], c[:, [3, 1, 5]], c[:, [4, 5, 2]]], 1)

        def apply_m(v):
            return np.einsum("nij,nj->ni", full, v.reshape(-1, 3)).ravel()
    ref = _one_cycle(s.ctx, s.b, apply_m, k)
    assert np.linalg.norm(x - ref) <= 1e-9 * np.linalg.norm(ref)
    s.ctx.close()
