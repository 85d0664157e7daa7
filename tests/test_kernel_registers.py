"""Two waves of a FAST build's single-case z sweep fit a SIMD: at most 256 vector
registers and no scratch memory, in the kernels as compiled for gfx950 (no GPU
involved).  One register more and every z sweep runs one wave per SIMD."""
import os
import re
import subprocess

import pytest

from conftest import PKG

HIPCC = "/opt/rocm/bin/hipcc"


BUILDS = {"fast": [], "p64": ["-DMPCF_P64=1"], "epair": ["-DMPCF_P64=1", "-DMPCF_EPAIR=1"]}


@pytest.fixture(scope="module")
def listings(tmp_path_factory):
    if not os.path.exists(HIPCC):
        pytest.skip("no hipcc")
    import build
    d = tmp_path_factory.mktemp("kernels")
    jobs = {k: subprocess.Popen([HIPCC, *build.common_flags(), "-ffp-contract=on", "-DMPCF_FAST=1", *f, "--cuda-device-only",
                                 "-S", os.path.join(PKG, "csrc", "mpcf_kernels.hip"), "-o", str(d / k)])
            for k, f in BUILDS.items()}
    assert all(j.wait(timeout=300) == 0 for j in jobs.values())
    return {k: (d / k).read_text() for k in BUILDS}


@pytest.mark.parametrize("build_name", list(BUILDS))
def test_two_waves_of_the_z_sweep_fit_a_simd(listings, build_name):
    seen = 0
    for name, body in re.findall(r"\.amdhsa_kernel (\S+)(.*?)\.end_amdhsa_kernel", listings[build_name], flags=re.S):
        # k_sweep_yz<2, MODE_*>, and the batched sweep (no batch holds E as a pair)
        if "k_sweep_yzILi2" in name or ("kb_sweep_z" in name and build_name != "epair"):
            seen += 1
            assert int(re.search(r"next_free_vgpr (\d+)", body).group(1)) <= 256, name
            assert int(re.search(r"private_segment_fixed_size (\d+)", body).group(1)) == 0, name
    assert seen >= 3
