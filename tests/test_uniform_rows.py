"""Rows are reached through buffer resources made from their addresses.  Where the compiler cannot tell that an address is the
same for the whole wave it puts a loop around every such access that tries the lanes' resources one after the other: right, and
several times the instructions.  Looked for in the assembly of the kernels as they are built."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "tilexr_amd", "csrc")


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="no compiler")
@pytest.mark.parametrize("source", ["ep_exchange.hip", "ep_small.hip", "moonep_stage.hip", "ep_reduce_small.hip"])
def test_no_access_looks_for_its_row_lane_by_lane(source, tmp_path):
    out = tmp_path / "kernels.s"
    subprocess.run(["hipcc", "-std=c++17", "-O3", "--offload-arch=gfx950", "-ffp-contract=off", "-fno-gpu-flush-denormals-to-zero",
                    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-I", os.path.join(ROOT, "include"), "-I", CSRC,
                    "--cuda-device-only", "-S", os.path.join(CSRC, source), "-o", str(out)], check=True, capture_output=True)
    lines = [line.split(";")[0].strip() for line in out.read_text().splitlines()]
    lines = [line for line in lines if re.match(r"[a-z]", line)]
    accesses = [i for i, line in enumerate(lines) if re.match(r"buffer_(load|store)", line)]
    assert accesses
    # the loop reads the first lane's resource, compares it with every lane's and runs the access for those that match
    looped = [lines[i] for i in accesses if sum("v_cmp_eq_u64" in line for line in lines[i - 6:i]) >= 2]
    assert looped == []
