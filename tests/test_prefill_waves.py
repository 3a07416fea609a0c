"""What the prefill attention holds in registers leaves as many workgroups on a CU as its LDS has room for, or as many as it had."""
import os
import re
import shutil
import subprocess

import pytest

from return_amd.kernels import build

pytestmark = pytest.mark.skipif(not (shutil.which("hipcc") or os.path.exists("/opt/rocm/bin/hipcc")), reason="no hipcc")


def _workgroups(part, tmp_path):
    """(head size / 16, groups of rows a wave, groups of waves, extras) -> workgroups that a CU has room for, by LDS and by registers."""
    out = str(tmp_path / "kernel.s")
    subprocess.run([build._hipcc(), *build.FLAGS, f"-DPRE_PART={part}", "--cuda-device-only", "-S",
                    os.path.join(build.CSRC, "attention_prefill.hip"), "-o", out], check=True, stdout=subprocess.PIPE, stderr=subprocess.STDOUT)
    with open(out) as f:
        found = re.findall(r"\.amdhsa_kernel \S*ILi(\d+)ELi(\d+)ELi(\d+)ELi(\d+)E\S*(.*?)\.end_amdhsa_kernel", f.read(), re.S)
    rooms = {}
    for *form, text in found:
        size = {k: int(re.search(rf"\.amdhsa_{k} (\d+)", text).group(1))
                for k in ("next_free_vgpr", "group_segment_fixed_size", "private_segment_fixed_size")}
        assert size["private_segment_fixed_size"] == 0, form
        form = tuple(map(int, form))
        waves = min(8, 512 // (-(-size["next_free_vgpr"] // 8) * 8))              # of a SIMD; a group of four waves has one on each
        rooms[form] = min(163840 // size["group_segment_fixed_size"], waves // form[2])
    return rooms


@pytest.mark.parametrize("part,want", [(0, {(2, 2, 2, 0): 2, (2, 2, 2, 1): 2, (4, 2, 1, 0): 3, (4, 2, 2, 0): 1}),
                                       (1, {(8, 1, 2, 0): 1, (8, 2, 1, 0): 2, (8, 2, 2, 0): 1}),
                                       (2, {(9, 1, 1, 1): 4, (9, 1, 1, 2): 4, (10, 1, 1, 0): 3, (11, 1, 1, 0): 3, (11, 1, 1, 1): 3, (11, 1, 1, 2): 3,
                                            (12, 1, 1, 0): 3, (12, 1, 1, 1): 3, (12, 1, 1, 2): 3}),
                                       (3, {(13, 1, 1, 0): 2, (14, 1, 1, 0): 2, (16, 1, 1, 0): 2, (16, 1, 1, 2): 2})])
def test_workgroups_on_a_cu(part, want, tmp_path):
    rooms = _workgroups(part, tmp_path)
    assert {form: rooms[form] for form in want} == want
