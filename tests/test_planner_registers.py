"""The one-launch dispatch's kernels leave room for two workgroups of 1024 threads on a CU: 8 waves on a SIMD of
512 vector and 800 scalar registers, which are given out in eights and sixteens, 16 scalar ones of each wave for
the trap handler.  That leaves a wave 64 and 80."""

import re

from moonep_amd import build


def test_two_workgroups_to_a_cu(tmp_path):
    path = str(tmp_path / "planner.s")
    build.gemm_assembly(path, source="planner.hip")
    with open(path) as f:
        text = f.read()
    found = 0
    for block in re.split(r"^  - ", text[text.rfind("amdhsa.kernels:"):], flags=re.M)[1:]:
        name = re.search(r"^\s+\.name:\s+(\S+CopyArgs\S+)$", block, re.M)
        if not name:
            continue
        found += 1
        used = {key: int(re.search(rf"^\s+\.{key}:\s+(\d+)$", block, re.M).group(1))
                for key in ("vgpr_count", "sgpr_count", "vgpr_spill_count", "private_segment_fixed_size")}
        assert used["vgpr_count"] <= 64 and used["sgpr_count"] <= 80, (name.group(1), used)
        assert used["vgpr_spill_count"] == used["private_segment_fixed_size"] == 0, (name.group(1), used)
    assert found >= 8
