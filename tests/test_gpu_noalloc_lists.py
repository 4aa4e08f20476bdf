"""elastic_spmv_csrc_noalloc on patterns whose rows and transposed lists reach
the limits of its register path (lists of 64 entries, 128 products per row) and
pass them, and on row counts around a wavefront's eight rows: every result
equals the oracle's matvec_csrcsym1 (Matvec.f:528-621) bit for bit."""
import numpy as np
import pytest

from oracle import binding as O
from tests.test_zz_no_alloc import _product

pytestmark = pytest.mark.gpu


def _pattern(n, lower):
    """CSRC pattern from a lower-triangle boolean matrix."""
    ia = np.ones(n + 1, np.int32)
    ia[1:] += np.cumsum(lower.sum(1)).astype(np.int32)
    return ia, (np.nonzero(lower)[1] + 1).astype(np.int32)


def _lower(kind, n):
    i, j = np.indices((n, n))
    band = {"band": n // 3, "dense": n}.get(kind, 0)
    m = (j < i) & (i - j <= band)
    if kind == "arrow":  # the first column and the last row are full
        m |= (j < i) & ((j == 0) | (i == n - 1))
    if kind == "diag":
        m[:] = False
    return m


@pytest.mark.parametrize("kind,n", [("diag", 1), ("dense", 2), ("dense", 9), ("dense", 65),
                                    ("dense", 66), ("dense", 200), ("arrow", 65), ("arrow", 66),
                                    ("arrow", 1000), ("band", 193), ("band", 195), ("band", 400)])
def test_lists_of_every_length(kind, n):
    from elastic_amd import _lib

    print("noalloc lists", kind, n, flush=True)
    rng = np.random.default_rng(n)
    ia, ja = _pattern(n, _lower(kind, n))
    ad, al, x = rng.standard_normal(n), rng.standard_normal(len(ja)), rng.standard_normal(n)
    y = _product(_lib.lib(), ia, ja, ad, al, x)
    assert np.array_equal(y, O.matvec(ia, ja, ad, al, x))
