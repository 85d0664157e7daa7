"""The edge primitives that a wave of the bit-exact and binary64 x+y sweeps passes
between its lanes through LDS, in the kernels as the source states them (device
code before any optimization, no GPU involved).  Four lanes write the four
positions of one row and primitive: each store has to touch its own scalar only,
where a store into a vector's element would read and write the whole vector, and
the writes have to be ordered by fences against the reads before and after."""
import os
import re
import subprocess

import pytest

from conftest import PKG

HIPCC = "/opt/rocm/bin/hipcc"


@pytest.mark.parametrize("defines", [["-DMPCF_FAST=0"], ["-DMPCF_FAST=0", "-DMPCF_F64=1"]])
def test_lanes_write_scalars_between_fences(tmp_path, defines):
    if not os.path.exists(HIPCC):
        pytest.skip("no hipcc")
    import build
    out = tmp_path / "raw.ll"
    subprocess.run([HIPCC, *build.common_flags(), "-ffp-contract=off", *defines, "--cuda-device-only", "-S", "-emit-llvm",
                    "-Xclang", "-disable-llvm-passes", os.path.join(PKG, "csrc", "mpcf_kernels.hip"), "-o", str(out)],
                   check=True, capture_output=True, timeout=120)
    text = out.read_text()
    arrays = re.findall(r"^@(\w*sweep_xy_body\w*sh_halo) = .*? addrspace\(3\) global (.*?) undef", text, flags=re.M)
    assert arrays
    for name, kind in arrays:
        assert "<" not in kind, (name, kind)              # scalars, no vectors
    # the functions that fill them (the ones that read load a vector): fences on either side of the stores
    fills = 0
    for body in re.findall(r"^define .*?^}", text, flags=re.M | re.S):
        if "sh_halo to ptr" not in body or "load <4 x" in body:
            continue
        first = body.index("sh_halo to ptr")
        last = max(m.start() for m in re.finditer(r"store (?:float|double) ", body))
        fences = [m.start() for m in re.finditer(r"call void @\w*wave_sync", body)]
        assert first < last and fences and fences[0] < first and fences[-1] > last
        fills += 1
    assert fills == len(arrays)
    sync = re.search(r"^define [^\n]*wave_sync.*?^}", text, flags=re.M | re.S).group(0)
    assert 'fence syncscope("wavefront") release' in sync and 'fence syncscope("wavefront") acquire' in sync
    assert sync.index("release") < sync.index("wave.barrier") < sync.index("acquire")
