"""Admission counts the words that a solve on the chip exchanges: on every system
that is held, footprint_bytes covers the layout's own number of them beside what it
counted before (CSRC, planes, words, partials, vectors)."""
import types

import pytest

from elastic_amd import mesh as M

# element nodes, dofs, (nodes, equations, external partials of the default layout)
SYSTEMS = [
    (4, 2, 4225, 8320, 2734), (4, 2, 66049, 131584, 66510), (3, 2, 66049, 131584, 61246),
    (8, 3, 1331, 3630, 2316), (8, 3, 9261, 26460, 22780), (8, 3, 21952, 63504, 63467),
    (8, 3, 32768, 95232, 72345), (8, 3, 68921, 201720, 80966),
]


def _words(neq, ndf, partials):
    return 8 * (16640 + 3 * neq + 2 * ndf * partials)


def _others(nen, ndf, nnode):
    neq = nnode * ndf
    nad = int(neq * ({3: 3.5, 4: 4.5, 8: 13.5}[nen] * ndf + 1))
    return 24 * nad + nad // 2 + 92 * neq + 64 * 1024 * 8


@pytest.mark.parametrize("nen,ndf,nnode,neq,partials", SYSTEMS)
def test_admission_covers_the_words(nen, ndf, nnode, neq, partials):
    from elastic_amd.serving import footprint_bytes

    fp = footprint_bytes(types.SimpleNamespace(nen=nen, ndf=ndf, nnode=nnode))
    extra = fp - _others(nen, ndf, nnode)
    assert _words(neq, ndf, partials) <= extra <= 2.5 * _words(neq, ndf, partials)


@pytest.mark.parametrize("nen,ndf,nnode", [(4, 2, 513 * 513), (8, 3, 61 ** 3)])
def test_systems_that_are_not_held_have_none(nen, ndf, nnode):
    from elastic_amd.serving import footprint_bytes

    assert footprint_bytes(types.SimpleNamespace(nen=nen, ndf=ndf, nnode=nnode)) == \
        _others(nen, ndf, nnode)


@pytest.mark.gpu
@pytest.mark.parametrize("k", [0, 2, 3, 5, 6])
def test_partials_are_those_of_the_layout(k):
    from elastic_amd.system import System

    nen, ndf, nnode, neq, partials = SYSTEMS[k]
    n = int(round(nnode ** (1.0 / ndf))) - 1
    s = System(M.hex8_cube(n) if nen == 8 else M.quad4_square(n) if nen == 4 else M.tria3_square(n))
    assert s.neq == neq and s.ctx.layout_info()["ext_partials"] == partials
    assert s.ctx.get_option("resident") == 1
    s.ctx.close()
