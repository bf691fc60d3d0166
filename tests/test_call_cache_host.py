"""The operators' kept scratch blocks, on the CPU: nscale_amd/csrc/call_cache.cpp built with the host compiler
against a stand-in for the HIP runtime (tests/call_cache_host.cpp)."""
import os
import shutil
import subprocess

import pytest

from tests._lib import ROOT


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if shutil.which("g++") is None or not os.path.isdir("/opt/rocm/include"):
        pytest.skip("host compiler or ROCm headers absent")
    exe = tmp_path_factory.mktemp("call_cache") / "host"
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I", os.path.join(ROOT, "include"), "-I", os.path.join(ROOT, "nscale_amd", "csrc"), "-o", str(exe),
                    os.path.join(ROOT, "tests", "call_cache_host.cpp"), os.path.join(ROOT, "nscale_amd", "csrc", "call_cache.cpp"),
                    "-lpthread"], check=True)
    return str(exe)


def _run(program, what):
    r = subprocess.run([program, what], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr


def test_a_capture_on_another_stream_goes_on(program):
    _run(program, "capture")


def test_a_failing_allocation_finds_the_unused_blocks(program):
    _run(program, "pressure")


def test_blocks_of_quiet_streams_go_back(program):
    _run(program, "age")
