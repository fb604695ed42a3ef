"""The copying workgroups of the plan-driven scatters reach tables and rows through global addresses, and the per-route one for
several ranks has its route word and the rank's receive tensor from the scalar unit, ahead of the row.  Looked for in the assembly:
an access whose address space was lost is a flat one, and an address that lanes load is a trip of its own behind the row's."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "tilexr_amd", "csrc")


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="no compiler")
def test_copies_use_global_and_scalar_addresses(tmp_path):
    out = tmp_path / "kernels.s"
    subprocess.run(["hipcc", "-std=c++17", "-O3", "--offload-arch=gfx950", "-ffp-contract=off", "-fno-gpu-flush-denormals-to-zero",
                    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-I", os.path.join(ROOT, "include"), "-I", CSRC,
                    "--cuda-device-only", "-S", os.path.join(CSRC, "moonep_stage.hip"), "-o", str(out)], check=True, capture_output=True)
    kernels = re.findall(r"^(_ZN\S*moon_scatter_(?:token_)?kernelILb\S*):\s*; @(.*?)^\s*s_endpgm", out.read_text(), re.S | re.M)
    scalar = [name for name, _ in kernels if re.search(r"moon_scatter_kernelILb[01]ELb1E", name)]
    assert len(scalar) == 2 and len(kernels) > 10
    for name, body in kernels:
        code = [line.split(";")[0].strip() for line in body.splitlines()]
        code = [line for line in code if re.match(r"[a-z]", line)]
        assert [line for line in code if line.startswith("flat_")] == [], name
        if name in scalar:
            # the copy is the kernel's last part: its row loads are the last two
            rows = [i for i, line in enumerate(code) if line.startswith("global_load_dwordx4")][-2:]
            stores = [i for i, line in enumerate(code) if re.match(r"global_store_dwordx4 .* nt\b", line)][-2:]
            assert rows[1] < stores[0], name
            copy = code[rows[0] - 12:stores[1]]
            assert [line for line in copy if re.match(r"(global|buffer)_load_(dword|ubyte|dwordx2)\b", line)] == [], name
            assert any(line.startswith("s_load_dword ") for line in copy), name
