"""The scratch cache (csrc/nebo_scratch.hip) over a host model of the HIP calls it
makes (tests/scratch_host.cpp): limits, eviction, memory that runs out, other threads'
captures.  The bits of calls that share blocks: test_gpu_scratch.py."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SOURCE = os.path.join(HERE, "..", "spatialops-threadfix_amd", "csrc", "nebo_scratch.hip")
CHECKS = ["other_threads_capture", "slots_are_reused", "failed_upload", "kept_within_the_limit", "lent_together",
          "little_memory_left", "blocks_between_streams", "memory_runs_out", "program_memory_runs_out",
          "captured_stream"]

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not installed")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("scratch") / "scratch_host")
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-x", "c++",
                    SOURCE, os.path.join(HERE, "scratch_host.cpp"), "-o", exe, "-lpthread"], check=True)
    return exe


@pytest.mark.parametrize("check", CHECKS)
def test_scratch(program, check):
    r = subprocess.run([program, check], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr
