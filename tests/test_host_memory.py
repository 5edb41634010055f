"""Host-side memory handling on a stub HIP runtime (tests/csrc/hip_stub.hpp), which makes
allocations fail where a scenario asks for it, checks the bytes behind every block and holds
every launch's dynamic LDS against the limit set for its kernel."""
import os
import subprocess

import pytest

from bipp_amd import build

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def compile_host(exe, source):
    """A harness as host code only (no GPU code, no HIP runtime)."""
    try:
        hipcc = build.hipcc()
    except RuntimeError:
        pytest.skip("hipcc not available")
    subprocess.run([hipcc, "-x", "hip", "-std=c++17", "--cuda-host-only", "--offload-arch=gfx950",
                    "-no-hip-rt", "-O1", "-g", "-Wno-unused-value",
                    "-I" + os.path.join(ROOT, "include"),
                    "-I" + os.path.join(ROOT, "bipp_amd", "csrc"),
                    os.path.join(ROOT, "tests", "csrc", source), "-o", exe, "-pthread",
                    "-Wl,--unresolved-symbols=ignore-all"], check=True, capture_output=True)
    return exe


@pytest.fixture(scope="module")
def harness(tmp_path_factory):
    return compile_host(str(tmp_path_factory.mktemp("mem") / "memory_harness"),
                        "memory_harness.cpp")


@pytest.mark.parametrize("scenario", ["staging_growth_fails", "pool_gives_way",
                                      "failed_flush_waits"])
def test_memory(harness, scenario):
    r = subprocess.run([harness, scenario], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, f"exit {r.returncode}: {r.stderr[-2000:]}"


@pytest.fixture(scope="module")
def launch_harness(tmp_path_factory):
    return compile_host(str(tmp_path_factory.mktemp("launch") / "launch_harness"),
                        "launch_harness.cpp")


@pytest.mark.parametrize("scenario", ["limits", "limit_fails_once"])
def test_launch_limits(launch_harness, scenario):
    r = subprocess.run([launch_harness, scenario], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, f"exit {r.returncode}: {r.stdout}{r.stderr[-2000:]}"
