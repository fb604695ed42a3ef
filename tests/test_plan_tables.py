"""Tables of the plan-driven stages for calls of several sizes through one world: tests/cxx/plan_tables_check.cpp compiles
the library's own host side against launches that only note where the tables are."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("ranks", [1, 3, 16])
def test_tagged_words_lie_apart_from_others_at_every_size(tmp_path, ranks):
    exe = str(tmp_path / "plan_tables_check")
    csrc = os.path.join(ROOT, "tilexr_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(ROOT, "include"), "-I", csrc,
                    "-I", os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "include"),
                    os.path.join(csrc, "moonep_api.cpp"), os.path.join(ROOT, "tests", "cxx", "plan_tables_check.cpp"),
                    "-o", exe], check=True)
    run = subprocess.run([exe, str(ranks)], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0, run.stdout
