"""Launches of the plan-driven Dispatch by the sizes of a call: tests/cxx/plan_launches_check.cpp runs the library's own host side
against a runtime that only notes them."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "tilexr_amd", "csrc")
pytestmark = pytest.mark.skipif(shutil.which("hipcc") is None, reason="no compiler")


@pytest.fixture(scope="module")
def launches(tmp_path_factory):
    tmp = tmp_path_factory.mktemp("plan_launches")
    include = ["-I", os.path.join(ROOT, "include"), "-I", CSRC, "-I", os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "include")]
    subprocess.run(["hipcc", "-std=c++17", "-O1", "--offload-arch=gfx950", "--cuda-host-only", "-fPIC", *include, "-c",
                    os.path.join(CSRC, "moonep_stage.hip"), "-o", str(tmp / "stage.o")], check=True, capture_output=True)
    # (the kernels' code object is the one symbol that is left out)
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", *include,
                    os.path.join(ROOT, "tests", "cxx", "plan_launches_check.cpp"), str(tmp / "stage.o"),
                    "-Wl,--unresolved-symbols=ignore-all", "-o", str(tmp / "check")], check=True)

    def run(ranks, tokens, k, h, rows, fresh):
        out = subprocess.run([str(tmp / "check"), *(str(int(v)) for v in (ranks, tokens, k, h, rows, fresh))], check=True,
                             capture_output=True, text=True, timeout=60).stdout
        return [(name, int(x), int(y), int(lds)) for name, x, y, lds in (line.split() for line in out.splitlines())]

    return run


@pytest.mark.parametrize("fresh", [True, False])
@pytest.mark.parametrize("ranks,tokens,k,h,rows", [
    (2, 512, 8, 2048, 512 * 8 + 1), (4, 509, 8, 2048, 4200), (3, 100, 3, 1000, 321), (2, 2048, 8, 7168, 2048 * 8 + 70), (16, 9, 1, 64, 65)])
def test_every_rank_copies_on_the_xcds_of_its_tokens(launches, ranks, tokens, k, h, rows, fresh):
    """Workgroup b runs on XCD b % 8 counting through all ranks' shares of a launch: a share is a multiple of eight."""
    (name, x, y, _), = [launch for launch in launches(ranks, tokens, k, h, rows, fresh) if "moon_scatter" in launch[0]]
    assert "generic" not in name and y == ranks and x % 8 == 0


@pytest.mark.parametrize("tokens,k,rows", [(32, 8, 256), (32, 8, 2048), (32, 8, 2049), (4096, 8, 32768), (4096, 8, 40000)])
def test_a_workgroup_looks_after_as_many_rows_as_it_has_threads(launches, tokens, k, rows):
    """The workgroups that look for rows nobody copies to: beside capped copies each is a trip to memory of few at a time."""
    (_, x, _, _), = [launch for launch in launches(1, tokens, k, 1000, rows, False) if "moon_scatter" in launch[0]]
    assert x == (tokens + 31) // 32 * 8 + (rows + 2047) // 2048 * 8


@pytest.mark.parametrize("tokens,rows,fresh,lds", [
    (16384, 131072, True, 56 * 1024), (16385, 131080, True, 0), (16385, 131080, False, 56 * 1024), (60000, 480000, True, 0)])
def test_two_to_a_compute_unit_only_while_they_hold_the_plan(launches, tokens, rows, fresh, lds):
    """Rows that end within a line: the plan's workgroups, one per 256 rows, are ahead of the copies and under their cap."""
    (_, _, _, got), = [launch for launch in launches(1, tokens, 8, 1000, rows, fresh) if "moon_scatter" in launch[0]]
    assert got == lds


@pytest.mark.parametrize("rows,h,fused", [
    (64, 8, True), (524288, 64, True), (524289, 1024, True), (1048576, 504, True), (1048577, 504, False), (1048577, 512, True),
    (2097152, 1024, True), (2097153, 1024, False)])
@pytest.mark.parametrize("ranks", [1, 4])
def test_plans_that_the_scatter_launch_builds(launches, ranks, rows, h, fused):
    """Two launches where the scatter builds a fresh plan, launches of the plan and of the rest behind the copies where not."""
    names = [name for name, *_ in launches(ranks, rows // 8, 8, h, rows, True)]
    assert sum("moon_scatter" in name for name in names) == 1
    if fused:
        assert len(names) == 2 and "moon_records" in names[0] and "moon_scatter" in names[1]
    else:
        assert "moon_dedup_groups" in names[-2] and "moon_finish" in names[-1]
