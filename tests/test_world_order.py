"""What the calls of a logical world are ordered behind, for every rank that calls last: tests/cxx/world_order_check.cpp
compiles the library's own orchestration against a model of streams and events."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("world_order") / "world_order_check")
    csrc = os.path.join(ROOT, "tilexr_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(ROOT, "include"), "-I", csrc,
                    "-I", os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "include"),
                    os.path.join(csrc, "multi_rank.cpp"), os.path.join(ROOT, "tests", "cxx", "world_order_check.cpp"),
                    "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("half", ["dispatch", "combine"])
@pytest.mark.parametrize("scenario", ["late-work", "next-exchange", "per-thread-streams", "failed-launch"])
def test_order_of_a_worlds_calls(check, scenario, half):
    run = subprocess.run([check, scenario, half], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0, run.stdout


def test_tables_of_differently_sized_combines(check):
    """Tags are told from stale words by their epoch: what is no tag may not lie where another size's tags do."""
    run = subprocess.run([check, "shapes"], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0, run.stdout
