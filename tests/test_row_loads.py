"""A reduce asks for the rows of several slots before it waits for the first of them.  Looked for in the assembly of the kernels
that are launched without flags: no row load stands behind a wait for all loads before it."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "tilexr_amd", "csrc")


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="no compiler")
@pytest.mark.parametrize("source", ["ep_reduce_vec_bf16.hip", "ep_reduce_vec_fp16.hip"])
def test_row_loads_do_not_wait_for_one_another(source, tmp_path):
    out = tmp_path / "kernels.s"
    subprocess.run(["hipcc", "-std=c++17", "-O3", "--offload-arch=gfx950", "-ffp-contract=off", "-fno-gpu-flush-denormals-to-zero",
                    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-I", os.path.join(ROOT, "include"), "-I", CSRC,
                    "--cuda-device-only", "-S", os.path.join(CSRC, source), "-o", str(out)], check=True, capture_output=True)
    kernels = re.findall(r"^(_ZN\S*ep_reduce_vec\S*):\s*; @(.*?)^\s*s_endpgm", out.read_text(), re.S | re.M)
    assert len(kernels) > 10
    for name, body in kernels:
        code = [line.split(";")[0].strip() for line in body.splitlines()]
        code = [line for line in code if re.match(r"[a-z]", line)]
        rows = [i for i, line in enumerate(code) if re.match(r"(global|buffer)_load_dwordx4 .* nt\b", line)]
        assert rows, name
        assert [code[i] for i in rows if any("vmcnt(0)" in line for line in code[max(0, i - 3):i])] == [], name
