"""Edges of the library's host planning (tests/host/plan_edges.cpp, compiled
with the host compiler), a section per test."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

pytestmark = pytest.mark.skipif(shutil.which("g++") is None or not os.path.isdir("/opt/rocm/include/hip"),
                                reason="needs g++ and the HIP headers")


@pytest.fixture(scope="module")
def section(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("edges") / "plan_edges")
    cmd = ["g++", "-std=c++17", "-O1", "-Wall", "-Wno-unused-function", "-D__HIP_PLATFORM_AMD__", "-I",
           os.path.join(ROOT, "radis_amd", "csrc"), "-I", os.path.join(ROOT, "include"), "-I", "/opt/rocm/include",
           os.path.join(ROOT, "tests", "host", "plan_edges.cpp"), "-o", exe, "-lpthread"]
    p = subprocess.run(cmd, capture_output=True, text=True, timeout=300)
    assert p.returncode == 0, p.stderr[-3000:]

    def run(name):
        p = subprocess.run([exe, name], capture_output=True, text=True, timeout=300)
        print(p.stdout)
        assert p.returncode == 0, (p.returncode, p.stderr[-3000:], p.stdout)

    return run


def test_tile_too_wide_for_two_rows_is_refused(section):
    section("wide_tile")


def test_admission_bytes(section):
    section("bytes")


def test_partial_spectra_in_y(section):
    section("shares_in_y")


def test_scratch_array_holds_every_split(section):
    section("scratch")


def test_axis_groups_from_the_launch(section):
    section("axis_groups")


def test_half_length_by_its_cost(section):
    section("half_cost")


def test_shares_beside_image_items(section):
    section("image_room")


def test_planning_a_lone_request_allocates_nothing(section):
    section("no_allocation")
