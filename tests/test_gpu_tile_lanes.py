"""Lanes per tile of the launched products until they are set: 512 for the tiles of
more than 512 blocks of 3-dof systems of less than 32,768 nodes, else 256.  The
product with either agrees with the oracle's, and so do solves by launches: FP64
sums of up to 81 products per row in another order, 1e-13 relative; FP32 values
round to 6e-8 each, 1e-6."""
import numpy as np
import pytest

from elastic_amd import mesh as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,opts,lanes", [
    (27, {}, 256), (28, {}, 512), (31, {}, 512), (32, {}, 256), (14, {"tile_blocks": 1024}, 512),
    (14, {"tile_blocks": 512}, 256), (14, {"tile_blocks": 1024, "lanes64": 256, "lanes32": 256}, 256),
])
def test_default_lanes(n, opts, lanes):
    from elastic_amd.solver import FP64, MIXED
    from elastic_amd.system import System
    from oracle import binding as O

    s = System(M.hex8_cube(n, jitter=0.15, seed=n))
    for k, v in opts.items():
        s.ctx.set_option(k, v)
    assert s.ctx.get_option("lanes64") == s.ctx.get_option("lanes32") == lanes
    ad, al = s.values()
    v = np.random.default_rng(n).standard_normal(s.neq)
    y = O.matvec(s.ia, s.ja, ad, al, v)
    print("lanes", n, opts, flush=True)
    assert np.linalg.norm(s.ctx.spmv(v, FP64) - y) <= 1e-13 * np.linalg.norm(y)
    assert np.linalg.norm(s.ctx.spmv(v, MIXED) - y) <= 1e-6 * np.linalg.norm(y)
    s.ctx.close()
