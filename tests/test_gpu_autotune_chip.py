"""The autotuner times what a solve runs: where the chip holds a layout, the
iteration there.  A tuned system keeps its place on the chip and is no slower than
untuned (25% for the noise of short solves; the launches that a lost place would
cost take 2.5 times as long), and a batch's instances keep theirs."""
import pytest

from elastic_amd import mesh as M
from elastic_amd.solver import FP64, MIXED

pytestmark = pytest.mark.gpu


def _system(kind, n, opts=()):
    from elastic_amd.system import System

    s = System({"hex8": lambda: M.hex8_cube(n, jitter=0.15, seed=n), "quad4": lambda: M.quad4_square(n),
                "tria3": lambda: M.tria3_square(n)}[kind]())
    for k, v in dict(opts).items():
        s.ctx.set_option(k, v)
    s.ctx.upload_rhs(s.b)
    return s


def _iteration(s, precision):
    t = []
    for _ in range(6):
        st = s.ctx.solve_resident(precision=precision, tol=1e-9, maxit=300, allow_maxit=True)
        t.append(st["t_device_ms"] / st["iters"])
    return min(t), s.ctx.get_option("resident_tiles")


@pytest.mark.parametrize("kind,n,precision", [
    ("hex8", 29, FP64), ("hex8", 24, MIXED), ("hex8", 20, FP64), ("hex8", 38, MIXED),
    ("quad4", 160, FP64), ("quad4", 256, FP64), ("quad4", 300, MIXED), ("tria3", 256, FP64),
])
def test_a_tuned_system_keeps_the_chip(kind, n, precision):
    s = _system(kind, n)
    before, held = _iteration(s, precision)
    batch = s.ctx.get_option("resident_batch")
    assert held > 0
    print("autotune", kind, n, precision, flush=True)
    best, ms = s.ctx.autotune(precision=precision, reps=16)
    after, tiles = _iteration(s, precision)
    assert tiles > 0 and s.ctx.get_option("resident") == 1
    bit = 2 if precision == MIXED else 1
    assert s.ctx.get_option("resident_batch") & bit >= batch & bit
    assert after <= 1.25 * before and ms > 0
    s.ctx.close()


@pytest.mark.parametrize("opts,batch", [({}, 3), ({"tile_blocks": 1024}, 0), ({"accum32": 1}, 3),
                                        ({"accum32": 1, "batch_precond": 6}, 1),
                                        ({"accum32": 1, "tile_blocks": 1024}, 2), ({"resident": 0}, 0)])
def test_whether_a_batch_holds_it(opts, batch):
    s = _system("hex8", 14, opts)
    assert s.ctx.get_option("resident_batch") == batch
    s.ctx.close()


def test_off_the_chip_the_products_decide():
    s = _system("hex8", 12, {"resident": 0})
    best, ms = s.ctx.autotune(precision=FP64, reps=16)
    assert best in (256, 512, 768, 1024) and 0 < ms < 1 and s.ctx.get_option("resident") == 0
    assert _iteration(s, FP64)[1] == 0
    s.ctx.close()


def test_a_class_keeps_its_larger_requests_on_the_chip():
    """the tile size tuned on one request is not given to another that it would take
    off the chip (29^3 has 1,272 tiles of 256 blocks; 12^3 fits in any)"""
    from elastic_amd.serving import Server

    srv = Server(max_slots=2, mode="sequential", precision=FP64, autotune=True)
    for n, tile in ((29, 1024), (12, 256)):
        s = _system("hex8", n)
        srv.tuned[(3, FP64, int(s.ctx.neq).bit_length())] = (256, 256)
        srv._tune(s.ctx, FP64)
        assert s.ctx.get_option("tile_blocks") == tile and s.ctx.get_option("lanes64") == 256
        assert _iteration(s, FP64)[1] > 0
        s.ctx.close()
