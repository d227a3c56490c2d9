"""The engine's host side without a GPU: a program of its C-ABI calls linked
with stand-ins of the HIP runtime functions (tests/cpp/fake_hip.cpp), which
record launches and allocations and can refuse them."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIBDIR = os.path.join(ROOT, "icempm_multi_amd")
CHECKS = ["empty_scene", "huge_tile_table", "no_memory_for_tiles", "fill_alignment", "coherent_staging",
          "two_devices", "no_pinned_memory", "indenter_workgroups", "census_by_points"]


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("engine_host") / "engine_host_test")
    src = [os.path.join(ROOT, "tests", "cpp", f) for f in ("engine_host_test.cpp", "fake_hip.cpp")]
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-rdynamic",
                    *src, "-o", exe, "-L", LIBDIR, "-licempm", "-Wl,-rpath," + LIBDIR, "-lpthread"], check=True)
    return exe


def test_all_checks_are_listed(program):
    out = subprocess.run([program], capture_output=True, text=True, check=True).stdout
    assert out.split() == CHECKS


@pytest.mark.parametrize("check", CHECKS)
def test_engine_host(program, check):
    r = subprocess.run([program, check], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-2000:]
