"""The work that users of this library have it do, as cases that can be timed.

A case is a dict of plain values.  `prepare(case, seed)` builds what a user's
program holds before the call (contexts with their systems on the GPU, right
hand sides), `run(state)` makes one pass through the public entry points, and
`exact(case, seed)` gives the same outputs from plain torch and numpy in 64
bits.  Sizes follow the library's workloads: hex8 cubes of 20^3 to 100^3
elements, tet4 cubes split in six, plane-strain squares of 32 to 512 elements
a side, and J2 load paths on hex8 cubes.

Paths ("path" of a case):

  solve     System.solve: b and x on the host, the system resident; PCG (FP64
            or mixed precision, Jacobi or 3x3 block Jacobi), BiCGSTAB, GMRES
  solv      the drop-in for the Fortran program's solver call: pattern, values
            and right hand side from host arrays at every call
  batch     a batch of requests: submitted, iterated together, x read back
  assemble  K and b = b0 - K u on the GPU for given displacements, then the
            nodal stresses of the same displacements
  j2        a Newton iterate of a plastic load path: return map, tangent and
            residual, then the tangent's product with the correction
  product   the product on caller-held device arrays, nothing allocated
"""
from __future__ import annotations

import math

import numpy as np
import torch

from elastic_amd import _lib, mesh
from elastic_amd.plasticity import PlasticPath
from elastic_amd.serving import Batch
from elastic_amd.solver import BDIAG3, BICGSTAB, DIAG, FP64, GMRES, MIXED, PCG, Context, solv
from elastic_amd.system import System

SOLVERS = {"pcg": PCG, "bicgstab": BICGSTAB, "gmres": GMRES}
TOL = 1e-11      # the solver interface's own default
MAXIT = 20000
EXACT_NEQ = 800_000  # beyond this many equations in all the plain solve takes too long


# -------------------------------------------------------------------- the list
def listed():
    return [
        # the smallest 3-D solve in use: one small part, latency and launches
        dict(name="pcg_hex8_20", path="solve", element="hex8", n=20, nu=0.3, solver="pcg",
             precision=FP64, precond=DIAG),
        # the headline: a large part solved once, in mixed precision
        dict(name="pcg_hex8_100_mixed", path="solve", element="hex8", n=100, nu=0.3, solver="pcg",
             precision=MIXED, precond=DIAG),
        # tetrahedra with strongly varying stiffness, block Jacobi, mixed
        dict(name="pcg_tet4_41_mixed", path="solve", element="tet4", n=41, nu=0.45, solver="pcg",
             precision=MIXED, precond=BDIAG3),
        # a plane-strain section of ordinary size, plain FP64
        dict(name="pcg_quad4_141", path="solve", element="quad4", n=141, nu=0.3, solver="pcg",
             precision=FP64, precond=DIAG),
        # the other two Krylov methods of the solver call
        dict(name="bicgstab_hex8_24", path="solve", element="hex8", n=24, nu=0.3, solver="bicgstab",
             precision=FP64, precond=DIAG),
        dict(name="gmres_hex8_17", path="solve", element="hex8", n=17, nu=0.3, solver="gmres",
             precision=FP64, precond=DIAG),
        # the Fortran program's call: every solve brings its values from the host
        dict(name="solv_hex8_43", path="solv", element="hex8", n=43, nu=0.3, solver="pcg",
             precision=FP64, precond=DIAG),
        # serving: plane-strain requests of mixed sizes, quad4 and tria3 in turn
        dict(name="batch_plane_16", path="batch", element="plane", n=160, nu=0.3, count=16,
             precision=FP64, precond=BDIAG3),
        # load paths of one 3-D part solved together in mixed precision
        dict(name="batch_hex8_33_mixed", path="batch", element="hex8", n=33, nu=0.3, count=6,
             precision=MIXED, precond=DIAG),
        # stiffness, residual and nodal stresses at given displacements
        dict(name="assemble_hex8_50", path="assemble", element="hex8", n=50, nu=0.3),
        # one Newton iterate of a plastic load path
        dict(name="j2_hex8_36", path="j2", element="hex8", n=36, nu=0.3),
        # the allocation-free product, for loops under graph capture
        dict(name="product_hex8_28", path="product", element="hex8", n=28, nu=0.3),
    ]


def _between(rng, lo, hi):
    """An integer between lo and hi, even over the logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    return dict(_draw(rng), nu=round(rng.uniform(0.2, 0.4), 4))


def _draw(rng):
    path = rng.choice(["solve", "solve", "solve", "solve", "solv", "batch", "assemble", "j2",
                       "product"])
    if path == "solve":
        element = rng.choice(["hex8", "hex8", "tet4", "quad4", "tria3"])
        solver = rng.choice(["pcg", "pcg", "pcg", "bicgstab", "gmres"])
        if element in ("quad4", "tria3"):  # plane sections are solved by FP64 PCG
            return dict(path=path, element=element, n=_between(rng, 32, 256), solver="pcg",
                        precision=FP64, precond=DIAG)
        if solver != "pcg":
            return dict(path=path, element="hex8",
                        n=_between(rng, 8, 30 if solver == "bicgstab" else 21), solver=solver,
                        precision=FP64, precond=DIAG)
        return dict(path=path, element=element,
                    n=_between(rng, 12, 72 if element == "hex8" else 48), solver="pcg",
                    precision=rng.choice([FP64, MIXED]), precond=rng.choice([DIAG, BDIAG3]))
    if path == "solv":
        return dict(path=path, element="hex8", n=_between(rng, 12, 56), solver="pcg",
                    precision=FP64, precond=DIAG)
    if path == "batch":
        if rng.random() < 0.5:
            return dict(path=path, element="plane", n=_between(rng, 48, 200),
                        count=rng.randint(3, 24), precision=FP64, precond=BDIAG3)
        return dict(path=path, element="hex8", n=_between(rng, 12, 40), count=rng.randint(2, 8),
                    precision=rng.choice([FP64, MIXED]), precond=DIAG)
    top = {"assemble": 64, "j2": 48, "product": 50}[path]
    return dict(path=path, element="hex8", n=_between(rng, 10, top))


# ------------------------------------------------------------------ the inputs
def _mesh(element, n, nu, rng):
    """A part of the given element, size and Poisson's ratio: jittered nodes
    (3-D), Young's modulus and traction from rng."""
    seed = int(rng.integers(1 << 30))
    E = float(10.0 ** rng.uniform(-0.3, 0.3))
    t = rng.uniform(-1.0, 1.0, 3)
    if element == "hex8":
        return mesh.hex8_cube(n, jitter=0.15, seed=seed, E=E, nu=nu, traction=1e-3 * t)
    if element == "tet4":
        return mesh.tet4_cube(n, jitter=0.2, seed=seed, nu=nu, traction=1e-3 * t)
    make = mesh.quad4_square if element == "quad4" else mesh.tria3_square
    return make(n, E=E, nu=nu, traction=t[:2])


def _batch_parts(case):
    """(element, size) of every part of a batch: copies of one 3-D size, or
    plane sections with sides from n/5 to n, quad4 and tria3 in turn."""
    n, count = case["n"], case["count"]
    if case["element"] != "plane":
        return [(case["element"], n)] * count
    return [("tria3" if k % 2 else "quad4",
             max(8, int(round(n * (0.2 + 0.8 * k / max(1, count - 1)))))) for k in range(count)]


def _displacements(m, rng):
    """A smooth displacement field on the free dofs, of the size a load gives."""
    c = 1e-3 * rng.uniform(-1.0, 1.0, (m.ndf, 4))
    x = m.x
    u = np.stack([c[d, 0] * x[:, 0] + c[d, 1] * x[:, 1] * x[:, -1]
                  + c[d, 2] * np.sin(2.0 * x[:, 0] + c[d, 3]) for d in range(m.ndf)], axis=1)
    u[m.id != 0] = 0.0
    return np.ascontiguousarray(u)


def _plastic_path(case, rng):
    """A load path partway through its first increment: displacements after one
    linear solve, part of the Gauss points beyond yield."""
    m, ubar = mesh.hex8_block_pull(case["n"], stretch=float(rng.uniform(4e-3, 6e-3)),
                                   nu=case["nu"])
    p = PlasticPath(m, ubar, sy=float(rng.uniform(1e-3, 4e-3)), H=0.05)
    p.increment(0.6)
    p.assemble(True)
    p.ctx.solve_resident(precision=FP64, tol=TOL, maxit=MAXIT)
    p.correct()
    return p


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    path = case["path"]
    if path == "batch":
        systems = [System(_mesh(*part, case["nu"], rng)) for part in _batch_parts(case)]
        for s in systems:
            if case["precond"] == BDIAG3:
                s.ctx.set_option("batch_precond", BDIAG3)
            s.ctx.upload_rhs(s.b)
        return dict(case=case, systems=systems,
                    batch=Batch(0, max_slots=max(2, len(systems)), iters_per_step=16))
    if path == "j2":
        p = _plastic_path(case, rng)
        return dict(case=case, j2=p, du=p.ctx.download_x())
    s = System(_mesh(case["element"], case["n"], case["nu"], rng))
    state = dict(case=case, system=s)
    if path == "assemble":
        state["u"] = _displacements(s.mesh, rng)
    elif path == "solv":
        ad, al = s.values()
        state.update(ia=s.ia, ja=s.ja, ad=ad, al=al, b=s.b, m=np.zeros(s.neq), x=np.zeros(s.neq))
    elif path == "product":
        ad, al = s.values()
        x = rng.standard_normal(s.neq)
        state.update({k: torch.from_numpy(v).cuda() for k, v in
                      dict(ia=s.ia, ja=s.ja, ad=ad, al=al, x=x, y=np.zeros(s.neq)).items()})
        state["entry"] = _lib.lib().elastic_spmv_csrc_noalloc
    return state


# --------------------------------------------------------------------- one pass
def run(state):
    case = state["case"]
    path = case["path"]
    if path == "solve":
        x, _ = state["system"].solve(solver=SOLVERS[case["solver"]], precond=case["precond"],
                                     precision=case["precision"], tol=TOL, maxit=MAXIT, ngram=50)
        return x
    if path == "solv":
        st = state
        solv(len(st["b"]), len(st["ja"]), st["ia"], st["ja"], st["ad"], st["al"], st["m"],
             st["b"], st["x"], tol=TOL, maxit=MAXIT, precision=case["precision"],
             precond=case["precond"])
        return dict(m=st["m"], x=st["x"])
    if path == "batch":
        b, systems = state["batch"], state["systems"]
        for k, s in enumerate(systems):
            b.submit(s.ctx, precision=case["precision"], tol=TOL, maxit=MAXIT, tag=k)
        done = 0
        while done < len(systems):
            b.step()
            done += len(b.poll())
        return [s.ctx.download_x() for s in systems]
    if path == "assemble":
        s, u = state["system"], state["u"]
        return dict(b=s.assemble(u), tx=s.stress(u))
    if path == "j2":
        p = state["j2"]
        rnorm = p.assemble(True)
        return dict(rnorm=rnorm, r=p.residual(), kdu=p.ctx.spmv(state["du"]))
    a = state
    rc = a["entry"](a["ad"].numel(), a["al"].numel(), a["ia"].data_ptr(), a["ja"].data_ptr(),
                    a["ad"].data_ptr(), a["al"].data_ptr(), a["x"].data_ptr(), a["y"].data_ptr(),
                    torch.cuda.current_stream().cuda_stream)
    if rc != _lib.OK:
        raise _lib.ElasticError(rc, "elastic_spmv_csrc_noalloc")
    return a["y"]


# ---------------------------------------------------------------- work of a pass
# lower neighbours of a node (node blocks of the stored triangle), dofs per
# node, elements per cell, and PCG iterations per element of the side: to
# TOL with Jacobi, as the workloads need them
ELEMENTS = {"hex8": (13, 3, 1, 14.0), "tet4": (7, 3, 6, 75.0), "quad4": (4, 2, 1, 12.0),
            "tria3": (3, 2, 2, 14.0)}


def _system_work(element, n):
    """(equations, stored values of the triangle, index bytes) of a part."""
    blocks, ndf, _, _ = ELEMENTS[element]
    nodes = n * (n + 1) ** (2 if ndf == 3 else 1)
    return ndf * nodes, nodes * (blocks * ndf * ndf + ndf * (ndf + 1) // 2), 4 * nodes * blocks


def _solve_work(element, n, solver, precision):
    """One iteration reads every stored value once and the method's vectors;
    GMRES(50) also its basis, twice 25 vectors on average."""
    neq, values, index = _system_work(element, n)
    iters = ELEMENTS[element][3] * n
    size = 4 if precision == MIXED else 8
    products, vectors = {"pcg": (1, 7), "bicgstab": (1, 12), "gmres": (1, 56)}[solver]
    if solver == "gmres":
        iters *= 3
    per = products * (values * size + index) + vectors * neq * size
    return iters * per, iters * (products * 4.0 * values + 2.0 * vectors * neq)


def work(case):
    n, path, element = case["n"], case["path"], case["element"]
    if path == "batch":
        parts = [_solve_work(*part, "pcg", case["precision"]) for part in _batch_parts(case)]
        return dict(bytes=sum(p[0] for p in parts), flops=sum(p[1] for p in parts))
    if path in ("solve", "solv"):
        nbytes, flops = _solve_work(element, n, case["solver"], case["precision"])
        if path == "solv":  # the values cross from the host once
            nbytes += 8 * _system_work(element, n)[1]
        return dict(bytes=nbytes, flops=flops)
    neq, values, index = _system_work(element, n)
    cells = n ** 3
    if path == "assemble":  # coordinates, u, connectivity in; K, b, stresses out
        return dict(bytes=8 * values + 8 * neq * 6 + 4 * 9 * cells, flops=24000.0 * cells)
    if path == "j2":  # the same, the plastic state in and out, one product
        return dict(bytes=2 * 8 * values + 8 * neq * 6 + 4 * 9 * cells + 2 * 8 * 56 * cells,
                    flops=60000.0 * cells + 4.0 * values)
    # CSRC arrays, x and y once each
    return dict(bytes=12 * 9 * 13 * (neq // 3) + 8 * 4 * neq, flops=4.0 * values)


# ------------------------------------------------------------- 64-bit references
def _symmetric(ia, ja, ad, al):
    """The full matrix of a CSRC triple as a torch CSR tensor on the GPU."""
    n = len(ad)
    row = torch.from_numpy(np.repeat(np.arange(n), np.diff(ia))).cuda()
    col = torch.from_numpy(ja.astype(np.int64) - 1).cuda()
    d = torch.arange(n, device="cuda")
    v, vd = torch.from_numpy(al).cuda(), torch.from_numpy(ad).cuda()
    idx = torch.stack([torch.cat([row, col, d]), torch.cat([col, row, d])])
    return torch.sparse_coo_tensor(idx, torch.cat([v, v, vd]), (n, n)).coalesce().to_sparse_csr()


def _solve_plain(ia, ja, ad, al, b):
    """Conjugate gradients in torch, FP64, until the residual stops mattering."""
    A, m = _symmetric(ia, ja, ad, al), 1.0 / torch.from_numpy(ad).cuda()
    r = torch.from_numpy(np.array(b)).cuda()
    x, p = torch.zeros_like(r), m * r
    rz = torch.dot(r, p)
    stop = 1e-30 * float(rz)
    for k in range(40000):
        q = A @ p
        alpha = rz / torch.dot(p, q)
        x += alpha * p
        r -= alpha * q
        z = m * r
        new = torch.dot(r, z)
        p = z + (new / rz) * p
        rz = new
        if k % 50 == 0 and float(rz) < stop:
            break
    return x.cpu().numpy()


_SIGN = np.array([[1, 1, 1], [-1, 1, 1], [-1, -1, 1], [1, -1, 1],
                  [1, 1, -1], [-1, 1, -1], [-1, -1, -1], [1, -1, -1]], float)


def _hex_b(xe, at):
    """(strain matrix (cells, 6, 24), determinant) of trilinear hexahedra at a
    natural point; strains xx yy zz xy yz zx."""
    f = 1.0 + _SIGN * at
    dn = 0.125 * np.stack([_SIGN[:, 0] * f[:, 1] * f[:, 2], _SIGN[:, 1] * f[:, 0] * f[:, 2],
                           _SIGN[:, 2] * f[:, 0] * f[:, 1]])
    jac = np.einsum("dn,enj->edj", dn, xe)
    g = np.linalg.solve(jac, np.broadcast_to(dn, (len(xe), 3, 8)))
    B = np.zeros((len(xe), 6, 8, 3))
    for k in range(3):
        B[:, k, :, k] = g[:, k]
    for row, (a, b) in zip((3, 4, 5), ((0, 1), (1, 2), (2, 0))):
        B[:, row, :, a], B[:, row, :, b] = g[:, b], g[:, a]
    return B.reshape(len(xe), 6, 24), np.linalg.det(jac)


def _elastic(E, nu):
    lam, mu = E * nu / ((1 + nu) * (1 - 2 * nu)), E / (2 * (1 + nu))
    C = np.zeros((6, 6))
    C[:3, :3] = lam
    C[np.arange(6), np.arange(6)] += [2 * mu] * 3 + [mu] * 3
    return C


def _to_equations(fe, cells, idn, neq):
    """Element vectors added to the equations of their free dofs."""
    eq = idn[cells].reshape(len(cells), -1)
    return np.bincount(eq.ravel(), fe.ravel(), minlength=neq + 1)[1:]


def _gauss():
    g = 0.577350269189626
    return [g * s for s in _SIGN]


def _exact_assemble(state):
    s, u = state["system"], state["u"]
    m = s.mesh
    cells, C = m.ix[:, :8] - 1, _elastic(m.e[0, 0], m.e[0, 1])
    xe, ue = m.x[cells], u[cells].reshape(len(cells), 24)
    fe = 0.0
    for at in _gauss():
        B, det = _hex_b(xe, at)
        sig = np.einsum("eij,ej->ei", B, ue) @ C
        fe = fe + np.einsum("eij,ei,e->ej", B, sig, det)
    total = np.zeros((m.nnode, 6))
    for a in range(8):
        B, _ = _hex_b(xe, _SIGN[a])
        np.add.at(total, cells[:, a], np.einsum("eij,ej->ei", B, ue) @ C)
    count = np.bincount(cells.ravel(), minlength=m.nnode)
    return dict(b=s.b0 - _to_equations(fe, cells, s.idn, s.neq), tx=total / count[:, None])


def _exact_j2(state):
    """Radial return with linear hardening from a virgin state, its tangent
    applied to the correction."""
    p, m = state["j2"], state["j2"].mesh
    E, nu, H = m.e[0, 0], m.e[0, 1], p.H
    mu, kappa, C = E / (2 * (1 + nu)), E / (3 * (1 - 2 * nu)), _elastic(E, nu)
    half = np.array([1, 1, 1, 0.5, 0.5, 0.5])
    one = np.array([1, 1, 1, 0, 0, 0], float)
    free = p.sys.idn > 0
    du = np.zeros((m.nnode, 3))
    du[free] = state["du"][p.sys.idn[free] - 1]
    cells = m.ix[:, :8] - 1
    xe, ue, de = m.x[cells], p.u()[cells].reshape(-1, 24), du[cells].reshape(-1, 24)
    fe, ke = 0.0, 0.0
    for at in _gauss():
        B, det = _hex_b(xe, at)
        st = np.einsum("eij,ej->ei", B, ue) @ C
        d = np.einsum("eij,ej->ei", B, de)
        s = st - st[:, :3].mean(1, keepdims=True) * one
        sn = np.sqrt((s * s) @ (1 / half))
        f = sn - np.sqrt(2 / 3) * p.sy
        dg = np.maximum(f, 0.0) / (2 * mu + 2 * H / 3)
        nrm = s / np.where(sn > 0, sn, 1.0)[:, None]
        th = 1 - 2 * mu * dg / np.where(sn > 0, sn, 1.0)
        thb = np.where(f > 0, 1 / (1 + H / (3 * mu)) - (1 - th), 0.0)
        dev = half * d - d[:, :3].sum(1, keepdims=True) / 3 * one
        ds = (kappa * d[:, :3].sum(1, keepdims=True) * one + 2 * mu * th[:, None] * dev
              - 2 * mu * (thb * np.einsum("ei,ei->e", nrm, d))[:, None] * nrm)
        sig = st - 2 * mu * dg[:, None] * nrm
        fe = fe + np.einsum("eij,ei,e->ej", B, sig, det)
        ke = ke + np.einsum("eij,ei,e->ej", B, ds, det)
    r = -_to_equations(fe, cells, p.sys.idn, p.sys.neq)
    return dict(rnorm=float(np.linalg.norm(r)), r=r,
                kdu=_to_equations(ke, cells, p.sys.idn, p.sys.neq))


def exact(case, seed):
    path = case["path"]
    if path == "batch":
        if sum(_system_work(*part)[0] for part in _batch_parts(case)) > EXACT_NEQ:
            return None
        state = prepare(case, seed)
        return [_solve_plain(s.ia, s.ja, *s.values(), s.b) for s in state["systems"]]
    if path in ("solve", "solv") and _system_work(case["element"], case["n"])[0] > EXACT_NEQ:
        return None
    state = prepare(case, seed)
    if path == "assemble":
        return _exact_assemble(state)
    if path == "j2":
        return _exact_j2(state)
    s = state["system"]
    ad, al = s.values()
    if path == "product":
        return _symmetric(s.ia, s.ja, ad, al) @ state["x"]
    x = _solve_plain(s.ia, s.ja, ad, al, s.b)
    return dict(m=1.0 / ad, x=x) if path == "solv" else x
