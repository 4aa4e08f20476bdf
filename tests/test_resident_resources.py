"""Scratch of the kernels of solves on the chip, from the gfx950 assembly that hipcc
writes for them with the build's flags: none but for the five named here, whose
1,024 lanes leave 128 registers each.  A spill in an iteration costs a round trip to
the caches, and no parity test would notice."""
import re

import pytest

from tests.test_kernel_resources import _kernel_resources

# bytes per lane, by the kernel's template arguments
SCRATCH = {
    "pcg_resident.hip": {"k_pcg_residentIddddLi3ELi4ELi4E": 88, "k_pcg_residentIfffdLi3ELi4ELi4E": 12},
    "bicgstab_resident.hip": {},
    "gmres_resident.hip": {},
    "batch.hip": {"k_bt_residentIdddLi3ELi2E": 44, "k_bt_residentIfddLi3ELi2E": 12,
                  "k_bt_residentIfffLi3ELi4E": 28},
}
KERNELS = {"pcg_resident.hip": 30, "bicgstab_resident.hip": 6, "gmres_resident.hip": 6, "batch.hip": 6}


@pytest.mark.parametrize("source", sorted(SCRATCH))
def test_scratch_is_what_is_stated(source, tmp_path):
    found = {k: v for k, v in _kernel_resources(source, tmp_path).items()
             if re.search(r"k_(pcg|bicgstab|gmres|bt)_residentI", k)}
    assert len(found) == KERNELS[source]
    for name, v in found.items():
        limit = [n for k, n in SCRATCH[source].items() if k in name]
        assert v["ScratchSize"] <= (limit[0] if limit else 0), (name, v)
