"""elastic_spmv_csrc_noalloc counts and places the entries of three consecutive
rows together: patterns whose rows match in threes (nodes of three dofs, from
row 0 or shifted by one or two), in twos, and not at all, with row counts of
every remainder.  Bit for bit the oracle's matvec_csrcsym1 (Matvec.f:528-621)."""
import numpy as np
import pytest

from oracle import binding as O
from tests.test_gpu_noalloc_lists import _pattern
from tests.test_zz_no_alloc import _product

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dofs,shift", [(3, 0), (3, 1), (3, 2), (2, 0), (2, 1), (1, 0)])
@pytest.mark.parametrize("n", [3, 4, 95, 96, 97, 400])
def test_rows_that_match_and_rows_that_do_not(dofs, shift, n):
    from elastic_amd import _lib

    print("noalloc triples", dofs, shift, n, flush=True)
    rng = np.random.default_rng(10 * n + dofs)
    node = (np.arange(n) + shift) // dofs
    pairs = rng.random((node[-1] + 1, node[-1] + 1)) < 0.1
    i, j = np.indices((n, n))
    ia, ja = _pattern(n, (j < i) & (pairs[node[:, None], node] | (node[:, None] == node)))
    ad, al, x = rng.standard_normal(n), rng.standard_normal(len(ja)), rng.standard_normal(n)
    y = _product(_lib.lib(), ia, ja, ad, al, x)
    assert np.array_equal(y, O.matvec(ia, ja, ad, al, x))
