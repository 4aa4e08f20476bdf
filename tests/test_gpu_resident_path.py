"""Which path a solve took: "resident_tiles" is the number of tiles per workgroup
with which it iterated on the chip, 0 where it went by launches, so a plan that
returns nothing, a launch that is refused or a wait that runs out shows, though the
results do not tell.  Every combination below states what the rules (tiles, LDS,
node block, type of sums) give."""
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


# (element, size, options, tiles per workgroup)
@pytest.mark.parametrize("kind,n,opts,tpw", [
    ("hex8", 1, {}, 1), ("quad4", 1, {}, 1), ("quad4", 9, {}, 1), ("tria3", 60, {}, 1),
    ("hex8", 7, {"tile_blocks": 32}, 1), ("hex8", 10, {"tile_blocks": 40}, 2),
    ("hex8", 12, {"tile_blocks": 40}, 4), ("hex8", 17, {"tile_blocks": 40}, 0),
    ("hex8", 9, {"tile_blocks": 64, "node_order": 1}, 1),
    ("quad4", 70, {"tile_blocks": 64}, 2), ("tria3", 110, {"tile_blocks": 64}, 4),
    ("quad4", 20, {"tile_blocks": 1024}, 1),  # (at most 127 nodes, so 508 blocks, per tile)
    ("hex8", 15, {"tile_blocks": 1024}, 1), ("hex8", 29, {}, 2), ("tet4", 14, {}, 1),
    ("hex8", 36, {}, 4),
])
def test_pcg(kind, n, opts, tpw):
    s = _system(kind, n, opts)
    three = kind in ("hex8", "tet4")
    assert s.ctx.get_option("resident_tiles") == s.ctx.get_option("resident_lost") == 0
    for precision, precond, sums32 in [(FP64, DIAG, 0), (FP64, BLOCKS, 0), (MIXED, DIAG, 0),
                                       (MIXED, BLOCKS, 0), (MIXED, DIAG, 1), (MIXED, BLOCKS, 1)]:
        want = tpw if three or (precond == DIAG and not (precision == MIXED and sums32)) else 0
        s.ctx.set_option("accum32", sums32)
        for resident in (1, 0, 1):
            print("path", kind, n, opts, precision, precond, sums32, resident, flush=True)
            s.ctx.set_option("resident", resident)
            s.solve(precision=precision, precond=precond, tol=1e-8, maxit=20000)
            assert s.ctx.get_option("resident_tiles") == (want if resident else 0)
    assert s.ctx.get_option("resident_lost") == 0
    s.ctx.close()


# (element, size, options, BiCGSTAB, GMRES cycle, GMRES): tiles per workgroup
@pytest.mark.parametrize("kind,n,opts,bi,k,gm", [
    ("hex8", 1, {}, 1, 3, 1), ("hex8", 4, {}, 1, 1, 1), ("hex8", 11, {}, 1, 33, 1),
    ("hex8", 7, {"tile_blocks": 40}, 1, 50, 1), ("hex8", 10, {"tile_blocks": 40}, 2, 17, 2),
    ("hex8", 12, {"tile_blocks": 40}, 0, 16, 0),
    ("hex8", 9, {"tile_blocks": 64, "node_order": 1}, 1, 50, 1),
    ("hex8", 15, {"tile_blocks": 1024}, 1, 120, 0), ("quad4", 12, {}, 1, 31, 1),
    ("tria3", 30, {}, 1, 50, 1), ("hex8", 28, {}, 2, 257, 0),
])
def test_bicgstab_and_gmres(kind, n, opts, bi, k, gm):
    from elastic_amd.solver import BICGSTAB, GMRES

    s = _system(kind, n, opts)
    for precond in (DIAG, BLOCKS):
        on = precond == DIAG or kind == "hex8"
        for resident in (1, 0):
            print("path bicgstab gmres", kind, n, opts, precond, resident, flush=True)
            s.ctx.set_option("resident", resident)
            s.solve(solver=BICGSTAB, precond=precond, tol=1e-8, maxit=3, allow_maxit=True)
            assert s.ctx.get_option("resident_tiles") == (bi if on and resident else 0)
            s.solve(solver=BICGSTAB, precision=MIXED, precond=precond, maxit=3, allow_maxit=True)
            assert s.ctx.get_option("resident_tiles") == 0
            s.solve(solver=GMRES, precond=precond, tol=1e-30, maxit=1, ngram=k, allow_maxit=True)
            assert s.ctx.get_option("resident_tiles") == (gm if on and resident else 0)
    s.ctx.close()


def _batch(systems, precision):
    from elastic_amd.serving import Batch

    with Batch(0, max_slots=len(systems), iters_per_step=8) as b:
        for k, s in enumerate(systems):
            s.ctx.upload_rhs(s.b)
            assert b.submit(s.ctx, precision, 1e-9, 20000, k)
        done = 0
        for _ in range(20000):
            b.step()
            done += len(b.poll())
            if done == len(systems):
                break
    return [s.ctx.get_option("resident_tiles") for s in systems]


@pytest.mark.parametrize("kind,n,opts,precision,tiles", [
    ("quad4", 40, {}, FP64, 4), ("quad4", 33, {"batch_precond": 6}, FP64, 4),
    ("tria3", 25, {"accum32": 0}, MIXED, 4), ("quad4", 12, {"accum32": 1}, MIXED, 0),
    ("hex8", 9, {}, FP64, 4), ("hex8", 7, {"batch_precond": 6}, FP64, 4),
    ("hex8", 8, {"accum32": 0}, MIXED, 4), ("hex8", 8, {"accum32": 1}, MIXED, 4),
    ("hex8", 14, {"accum32": 1, "tile_blocks": 1024}, MIXED, 4),
    ("hex8", 9, {"accum32": 1, "batch_precond": 6}, MIXED, 0),
    ("hex8", 13, {"tile_blocks": 1024}, FP64, 0), ("hex8", 17, {"tile_blocks": 40}, FP64, 0),
])
def test_batch(kind, n, opts, precision, tiles):
    a, b = _system(kind, n, opts), _system(kind, n, dict(opts, resident=0))
    print("path batch", kind, n, opts, precision, flush=True)
    assert _batch([a, b], precision) == [tiles, 0]
    assert a.ctx.get_option("resident_lost") == 0
    a.ctx.close()
    b.ctx.close()


@pytest.mark.parametrize("solver", ["pcg", "mixed", "bicgstab", "gmres", "batch"])
def test_a_lost_solve_is_counted_and_not_repeated(solver):
    """with no look left for its peers' words a solve is launched on the chip, gives
    up and is counted; the next ones do not try again until the option is set, or a
    layout built"""
    from elastic_amd.solver import BICGSTAB, GMRES, PCG

    s = _system("hex8", 12, {})

    def solve():
        if solver == "batch":
            return _batch([s], FP64)[0]
        s.solve(solver={"bicgstab": BICGSTAB, "gmres": GMRES}.get(solver, PCG), tol=1e-8,
                precision=MIXED if solver == "mixed" else FP64)
        return s.ctx.get_option("resident_tiles")

    held = solve()
    assert held > 0
    looks = s.ctx.get_option("resident_looks")
    s.ctx.set_option("resident_looks", 0)
    for _ in range(2):
        assert solve() == 0
        assert s.ctx.get_option("resident_lost") == 1 and s.ctx.get_option("resident") == 0
    s.ctx.set_option("resident_looks", looks)
    assert solve() == 0
    s.ctx.set_option("resident", 1)
    assert solve() == held and s.ctx.get_option("resident_lost") == 1
    s.ctx.set_option("resident_looks", 0)
    assert solve() == 0 and s.ctx.get_option("resident_lost") == 2
    s.ctx.set_option("resident_looks", looks)
    s.ctx.set_structure(s.ia, s.ja)
    ad, al = _system("hex8", 12, {}).values()
    s.ctx.set_values(ad, al)
    assert solve() == held
    s.ctx.close()


def test_a_batch_that_lost_an_instance_takes_the_lists():
    """instances already on the chip stay there; later ones of the same batch go to
    the lists, a new batch takes the chip again"""
    from elastic_amd.serving import Batch

    lost, beside, later = (_system("hex8", n, {}) for n in (8, 9, 7))
    lost.ctx.set_option("resident_looks", 0)
    for s in (lost, beside, later):
        s.ctx.upload_rhs(s.b)
    with Batch(0, max_slots=3, iters_per_step=8) as b:
        assert b.submit(lost.ctx, FP64, 1e-9, 20000, 0) and b.submit(beside.ctx, FP64, 1e-9, 20000, 1)
        b.step()
        done = b.poll()
        assert b.submit(later.ctx, FP64, 1e-9, 20000, 2)
        while len(done) < 3:
            b.step()
            done += b.poll()
    tiles = [s.ctx.get_option("resident_tiles") for s in (lost, beside, later)]
    assert tiles == [0, 4, 0]
    assert [s.ctx.get_option("resident_lost") for s in (lost, beside, later)] == [1, 0, 0]
    assert _batch([later], FP64) == [4]
    for s in (lost, beside, later):
        s.ctx.close()
