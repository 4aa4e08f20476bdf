"""The J2 kernel works on groups of seven elements of a colour: meshes whose
colours have 1 to 27 elements (one group with room, exactly full, one over),
free and restrained dofs, against sums of B^T C B and B^T sigma formed per
element in numpy from the state the kernel integrated.  All terms of a sum are
FP64 and few (8 points x 9 products x at most 8 elements), so 1e-12 of the
largest entry bounds the order of the sums."""
import numpy as np
import pytest

from elastic_amd import mesh as M

pytestmark = pytest.mark.gpu

SIGN = np.array([[1, 1, 1], [-1, 1, 1], [-1, -1, 1], [1, -1, 1],
                 [1, 1, -1], [-1, 1, -1], [-1, -1, -1], [1, -1, -1]], float)


def _points(m, p):
    """(B, det, sigma, C) of every element and Gauss point by radial return"""
    E, nu, sy, H = m.e[0, 0], m.e[0, 1], p.sy, p.H
    mu, kap = E / (2 * (1 + nu)), E / (3 * (1 - 2 * nu))
    one, half = np.array([1, 1, 1, 0, 0, 0.0]), np.array([1, 1, 1, .5, .5, .5])
    Pd = np.diag(half) - np.outer(one, one) / 3
    cells = m.ix[:, :8] - 1
    for e, c in enumerate(cells):
        for at in 0.577350269189626 * SIGN:
            f = 1 + SIGN * at
            dn = .125 * np.stack([SIGN[:, 0] * f[:, 1] * f[:, 2], SIGN[:, 1] * f[:, 0] * f[:, 2],
                                  SIGN[:, 2] * f[:, 0] * f[:, 1]])
            J = dn @ m.x[c]
            g = np.linalg.solve(J, dn)
            B = np.zeros((6, 8, 3))
            for k in range(3):
                B[k, :, k] = g[k]
            for row, (a, b) in zip((3, 4, 5), ((0, 1), (1, 2), (2, 0))):
                B[row, :, a], B[row, :, b] = g[b], g[a]
            B = B.reshape(6, 24)
            C = kap * np.outer(one, one) + 2 * mu * Pd
            sig = C @ (B @ p.u()[c].ravel())
            s = sig - sig[:3].mean() * one
            sn = np.sqrt((s * s) @ (1 / half))
            fy = sn - np.sqrt(2 / 3) * sy
            if fy > 0:
                dg = fy / (2 * mu + 2 * H / 3)
                n = s / sn
                th = 1 - 2 * mu * dg / sn
                thb = 1 / (1 + H / (3 * mu)) - (1 - th)
                sig = sig - 2 * mu * dg * n
                C = kap * np.outer(one, one) + 2 * mu * th * Pd - 2 * mu * thb * np.outer(n, n)
            yield e, B, np.linalg.det(J), sig, C


@pytest.mark.parametrize("n", [2, 3, 4, 5, 6])
def test_tangent_and_residual(n):
    from elastic_amd.plasticity import PlasticPath

    m, ubar = M.hex8_block_pull(n, stretch=5e-3, nu=0.3)
    p = PlasticPath(m, ubar, sy=2e-3, H=0.05)
    p.increment(0.6)
    p.assemble(True)
    r, neq = p.residual(), p.sys.neq
    eq = p.sys.idn[m.ix[:, :8] - 1].reshape(len(m.ix), -1)
    K, f = np.zeros((neq + 1, neq + 1)), np.zeros(neq + 1)
    for e, B, det, sig, C in _points(m, p):
        np.add.at(K, np.ix_(eq[e], eq[e]), det * (B.T @ C @ B))
        np.add.at(f, eq[e], det * (B.T @ sig))
    assert np.abs(r + f[1:]).max() <= 1e-12 * np.abs(f).max()
    A = np.stack([p.ctx.spmv(np.eye(neq)[k]) for k in range(neq)], 1)
    assert np.abs(A - K[1:, 1:]).max() <= 1e-12 * np.abs(K).max()
    first = p.assemble(False), p.residual()
    assert np.array_equal(first[1], r)  # the residual alone: the same bits
