"""Host transfers without a GPU: the library's host_copy linked with a stand-in
for the HIP runtime calls it makes (tests/host_copy_harness.cpp)."""
import os
import subprocess

import pytest

from conftest import PKG, ROOT

ROCM = "/opt/rocm/include"


@pytest.fixture(scope="module")
def harness(tmp_path_factory):
    if not os.path.exists(os.path.join(ROCM, "hip", "hip_runtime.h")):
        pytest.skip("no HIP headers")
    exe = tmp_path_factory.mktemp("host_copy") / "harness"
    csrc = os.path.join(PKG, "csrc")
    # only host_copy and what it calls runs: the rest of mpcf_capi.cpp stays unresolved
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-w", "-pthread", "-I", ROCM, "-I", csrc,
                    "-I", os.path.join(ROOT, "include"), os.path.join(ROOT, "tests", "host_copy_harness.cpp"),
                    os.path.join(csrc, "mpcf_capi.cpp"), "-o", str(exe), "-static",
                    "-Wl,--unresolved-symbols=ignore-all", "-Wl,--wrap=pthread_create"], check=True, timeout=120)
    return str(exe)


def run(harness, *mode):
    r = subprocess.run([harness, *mode], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr


def test_a_busy_stream_does_not_hold_up_another(harness):
    run(harness, "busy")


def test_streams_of_two_devices(harness):
    run(harness, "devices")


def test_sizes(harness):
    run(harness, "sizes")


def test_one_array_of_a_few_mb(harness):
    run(harness, "single")


def test_no_pinned_memory_left(harness):
    run(harness, "refused")


@pytest.mark.parametrize("threads", ["0", "2"])
def test_no_threads_left(harness, threads):
    """a host that gives no or only some of the copy threads"""
    run(harness, "threads", threads)
