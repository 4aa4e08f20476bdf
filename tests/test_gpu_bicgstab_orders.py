"""x of BiCGSTAB held on the chip and by launches differ in their last bits (sums
in another order), and are the same bits where both go by launches."""
import numpy as np
import pytest

from elastic_amd import mesh as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,opts,held", [
    (4, {}, True), (11, {}, True), (9, {"tile_blocks": 64, "node_order": 1}, True),
    (12, {"tile_blocks": 40}, False), (15, {"tile_blocks": 1024}, True), (28, {}, True),
])
def test_bits_differ_where_the_order_does(n, opts, held):
    from elastic_amd.solver import BICGSTAB
    from elastic_amd.system import System

    s = System(M.hex8_cube(n, jitter=0.15, seed=n + 1))
    for k, v in opts.items():
        s.ctx.set_option(k, v)
    x = []
    for resident in (0, 1):
        print("bicgstab orders", n, opts, resident, flush=True)
        s.ctx.set_option("resident", resident)
        x.append(s.solve(solver=BICGSTAB, tol=1e-11, maxit=20000)[0])
    assert np.array_equal(x[0], x[1]) is not held
    s.ctx.close()
