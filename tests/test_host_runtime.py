"""What the host enqueues, followed without a GPU: tests/host/host_runtime.cpp
stands in for the HIP runtime under the built library, and checks each launch
against the clocks, memory, streams and devices it is made for."""
import os
import subprocess

import pytest

from acoustics_amd import capi

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SCENARIOS = [
    "batch_capture",   # a batch's blocks on a captured stream
    "failed_load",     # a snapshot that is not there
    "server_check",    # a request given up before its first row, on a finiteness check
    "cut_chunk",       # a time chunk stopped early
    "no_memory_for_lists",   # no device memory while scenes are listed anew
    "no_pinned_memory",      # nor pinned memory for listener rows
    "other_device",          # reads while another device is selected
    "captured_neighbour",    # blocks of two handles, one stream under capture
    "side_by_side",          # blocks of several handles
    "short_blocks",          # blocks of a few steps
    "tries_again",           # a handle that gave a block up
    "device_bytes",          # what fdtd_get_info says of it
]


@pytest.fixture(scope="session")
def host_runtime(tmp_path_factory):
    capi.load_library()
    exe = str(tmp_path_factory.mktemp("host") / "host_runtime")
    lib = os.path.join(ROOT, "acoustics_amd", "lib")
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I" + os.path.join(ROOT, "include"),
                    "-rdynamic", "-o", exe, os.path.join(ROOT, "tests", "host", "host_runtime.cpp"), "-L" + lib,
                    "-lfdtd_acoustics", "-Wl,-rpath," + lib], check=True)
    return exe


@pytest.mark.parametrize("name", SCENARIOS)
def test_host_path(host_runtime, name):
    r = subprocess.run([host_runtime, name], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
