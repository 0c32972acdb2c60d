"""Scratch, registers and LDS of the tile kernels that split the inner dimension over a workgroup's waves, read from
the gfx950 code objects of this build: every instance (tile shape, layout, single, grouped, split over
workgroups, batched) runs without scratch, at two workgroups per CU or more."""
import os
import re

import pytest

import test_kernel_resources as metadata
from test_kernel_resources import _kernels, _workgroups_per_cu

BUILD = os.path.dirname(metadata.OBJ)
LAYOUTS = 4  # k-contiguous or row-contiguous A and B

pytestmark = [metadata.pytestmark,
              pytest.mark.skipif(not os.path.exists(os.path.join(BUILD, "tmm_ksplit_d.o")), reason="not built")]


# element type -> tile shapes, split shapes, batched instances per layout
@pytest.mark.parametrize("name,shapes,splits,batched", [("d", 12, 4, 1), ("s", 12, 4, 0), ("z", 7, 3, 0), ("c", 11, 3, 0)])
def test_ksplit_kernels_fit_without_scratch(monkeypatch, tmp_path, name, shapes, splits, batched):
    monkeypatch.setattr(metadata, "OBJ", os.path.join(BUILD, f"tmm_ksplit_{name}.o"))
    ks = {n: k for n, k in _kernels(tmp_path).items() if re.search(r"\dgemm_ks_(group_|split_|batched_)?kernelI", n)}
    assert len(ks) == LAYOUTS * (shapes + 1 + splits + batched), sorted(ks)
    spilled = {n: k["private_segment_fixed_size"] for n, k in ks.items() if k["private_segment_fixed_size"]}
    assert not spilled, spilled
    for n, k in ks.items():
        assert k["max_flat_workgroup_size"] == 256, n
        assert _workgroups_per_cu(k) >= 2, (n, k)
