"""Where the compiler places register spills in the kernels' listings (host only).

Kernels that need more registers than a wavefront has keep values in accumulation
registers or scratch memory.  At the join of a divergent branch the exec mask is
restored by an s_or_b64; a spill written in the join's block ahead of it is
written for the lanes of one side only, and the other lanes later read an older
value.  The compiler (ROCm 7.2) has placed spills so in two kernels: a loop
counter (the loop never ended) and a factor of a pair formula.  Both were written
as selects instead; no kernel of either B-spline order may have such a spill.
"""
import os
import re
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mpidopenmmplugin_amd", "csrc")
SPILL = re.compile(r"\s+(v_accvgpr_write|v_accvgpr_read|v_accvgpr_mov|scratch_store|scratch_load)")
VECTOR = re.compile(r"\s+(v_(?!accvgpr|writelane|readlane)|ds_|global_)")


def misplaced(lines):
    """(function, line) of the blocks whose exec restore comes after a spill and nothing else on the vector side."""
    found, function, in_block, spills = [], None, False, False
    for number, line in enumerate(lines, 1):
        name = re.match(r"(_Z\w+):", line)
        if name:
            function = name.group(1)
        if name or re.match(r"; %bb", line):
            in_block = spills = False
        elif re.match(r"\.LBB\w+:", line):
            in_block, spills = True, False
        elif in_block:
            if re.search(r"s_or_b64 exec, exec", line):
                if spills:
                    found.append((function, number))
                in_block = False
            elif "exec" in line or VECTOR.match(line):
                in_block = False
            elif SPILL.match(line):
                spills = True
    return found


def test_check_finds_a_misplaced_spill():
    block = ["_Z1kv:", ".LBB0_2:", "\tv_accvgpr_write_b32 a5, v153", "\ts_or_b64 exec, exec, s[2:3]"]
    assert misplaced(block) == [("_Z1kv", 4)]
    assert misplaced(block[:2] + block[:1:-1]) == []


def test_no_spill_ahead_of_an_exec_restore(tmp_path):
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    if not shutil.which(hipcc):
        pytest.skip("no hipcc")
    subprocess.run(["make", "-C", CSRC, "-j8", "listings", f"LISTDIR={tmp_path}"], check=True, capture_output=True,
                   timeout=600)
    listings = sorted(tmp_path.glob("*.s"))
    assert len(listings) == 12
    for path in listings:
        lines = path.read_text().splitlines()
        assert sum("s_endpgm" in line for line in lines) > 0, path.name
        assert misplaced(lines) == [], path.name
