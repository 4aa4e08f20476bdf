"""PCG held on the chip (one cooperative kernel) against the launch-per-phase
iteration on the same context: the same method with sums in another order, so
both meet the same stopping rule and agree as two FP64 solutions of it do.

Tile counts around 256, 512 and 1,024 (one, two or four tiles per workgroup and
the largest system held), tiles of at most 512 and of up to 1,024 blocks, one
tile alone, both dof counts, both node orders, FP64 and the FP32 operator with
FP64 and FP32 sums, Jacobi and node blocks.  Both solves stop at ||r||_M <
1e-11 ||b||_M; x differs by at most the condition number of the scaled system
(below 1e4 here) times 2e-11, so 1e-6 would hold; 1e-8 is the library's bar.
Iteration counts: two orders of FP64 sums move CG's count by a step or two, the
mixed method's by its replacements."""
import threading

import numpy as np
import pytest

from elastic_amd import mesh as M

pytestmark = pytest.mark.gpu

FP64, MIXED, DIAG, BLOCKS = 64, 32, 2, 6


def _system(kind, n, opts):
    from elastic_amd.system import System

    m = {"hex8": lambda: M.hex8_cube(n, jitter=0.15, seed=n + 1),
         "tet4": lambda: M.tet4_cube(n, jitter=0.2, seed=n + 1),
         "quad4": lambda: M.quad4_square(n), "tria3": lambda: M.tria3_square(n)}[kind]()
    s = System(m)
    for k, v in opts.items():
        s.ctx.set_option(k, v)
    return s


# (element, size, options, tiles per workgroup expected: 0 = not held)
CASES = [
    ("hex8", 1, {}, 1), ("hex8", 2, {}, 1), ("quad4", 1, {}, 1), ("quad4", 9, {}, 1),
    ("tria3", 60, {}, 1),
    ("hex8", 7, {"tile_blocks": 32}, 1), ("hex8", 10, {"tile_blocks": 40}, 2),
    ("hex8", 12, {"tile_blocks": 40}, 4), ("hex8", 17, {"tile_blocks": 40}, 0),
    ("hex8", 9, {"tile_blocks": 64, "node_order": 1}, 1),
    ("quad4", 70, {"tile_blocks": 64}, 2), ("tria3", 110, {"tile_blocks": 64}, 4),
    ("hex8", 15, {"tile_blocks": 1024}, 1), ("hex8", 29, {}, 2), ("tet4", 14, {}, 1),
    ("hex8", 36, {}, 4),
]


@pytest.mark.parametrize("kind,n,opts,tpw", CASES)
def test_matches_the_launch_iteration(kind, n, opts, tpw):
    s = _system(kind, n, opts)
    tiles = s.ctx.layout_info()["ntiles"]
    assert s.ctx.get_option("resident") == (1 if tpw else 0)
    if tpw:
        assert (tpw == 1 or tiles > 128 * tpw) and tiles <= 256 * tpw, tiles
    runs = [(FP64, DIAG, 0), (MIXED, DIAG, 0)]
    if kind in ("hex8", "tet4"):
        runs += [(FP64, BLOCKS, 0), (MIXED, BLOCKS, 0), (MIXED, DIAG, 1), (MIXED, BLOCKS, 1)]
    for precision, precond, sums32 in runs:
        print("resident", kind, n, opts, tiles, precision, precond, sums32, flush=True)
        s.ctx.set_option("accum32", sums32)
        got = []
        for resident in (0, 1, 1):
            s.ctx.set_option("resident", resident)
            got.append(s.solve(precision=precision, precond=precond, tol=1e-11, maxit=20000))
        (x0, s0), (x1, s1), (x2, s2) = got
        assert np.array_equal(x1, x2) and s1["iters"] == s2["iters"]  # run to run
        assert np.linalg.norm(x1 - x0) <= 1e-8 * np.linalg.norm(x0)
        slack = 2 if precision == FP64 else max(6, s0["iters"] // 10)
        assert abs(s1["iters"] - s0["iters"]) <= slack, (s0["iters"], s1["iters"])
        assert s1["norm_m_r"] <= 1.1 * max(s0["norm_m_r"], s1["conv"])
    s.ctx.close()


def test_iteration_limit_and_zero_right_hand_side():
    s = _system("hex8", 8, {})
    for precision in (FP64, MIXED):
        s.ctx.set_option("resident", 0)
        x0, s0 = s.solve(precision=precision, tol=1e-11, maxit=7, allow_maxit=True)
        s.ctx.set_option("resident", 1)
        x1, s1 = s.solve(precision=precision, tol=1e-11, maxit=7, allow_maxit=True)
        assert s0["iters"] == s1["iters"] == 7 and s0["status"] == s1["status"] == 2
        assert np.linalg.norm(x1 - x0) <= 1e-9 * np.linalg.norm(x0)
        x, st = s.ctx.solve(np.zeros(s.neq), precision=precision)
        assert not x.any() and st["iters"] == 0
    s.ctx.close()


@pytest.mark.parametrize("precision", [FP64, MIXED])
def test_a_wait_that_runs_out_starts_over_with_launches(precision):
    """A limit of no looks makes workgroups give up at once; the solve must come
    out as if the resident kernel had never run."""
    s = _system("hex8", 12, {})
    s.ctx.set_option("resident", 0)
    x0, s0 = s.solve(precision=precision, tol=1e-10)
    s.ctx.set_option("resident", 1)
    s.ctx.set_option("resident_looks", 0)
    x1, s1 = s.solve(precision=precision, tol=1e-10)
    assert np.array_equal(x0, x1) and s0["iters"] == s1["iters"]
    s.ctx.close()


def test_threads_with_their_own_contexts():
    """Cooperative kernels of several contexts at once: each result is the one
    its context gives alone."""
    systems = [_system(k, n, {}) for k, n in (("hex8", 10), ("quad4", 60), ("hex8", 18))]
    alone = [s.solve(precision=FP64, tol=1e-11)[0] for s in systems]
    out = [[None] * 3 for _ in systems]

    def work(i):
        for r in range(3):
            out[i][r] = systems[i].solve(precision=FP64, tol=1e-11)[0]

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(systems))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for i, s in enumerate(systems):
        assert all(np.array_equal(x, alone[i]) for x in out[i])
        s.ctx.close()
