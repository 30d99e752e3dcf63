"""The blocks of several instructions in qiw_dpp.h: no instruction may write a register that a
later one of the block reads as a factor.  Compiled for gfx950 where accumulators and factors hold
the same values, and read from the compiler's assembly."""
import os
import re
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
HIPCC = "/opt/rocm/bin/hipcc"


def test_factors_outlive_the_block(tmp_path):
    if shutil.which(HIPCC) is None:
        pytest.skip("hipcc not available")
    out = str(tmp_path / "dpp.txt")
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "--offload-device-only", "-S", "-w",
                    "-I", os.path.join(HERE, "..", "qinchworm.jl_amd", "csrc"), os.path.join(HERE, "native", "dpp_block.hip"),
                    "-o", out], check=True)
    blocks = re.findall(r"ASMSTART(.*?)ASMEND", open(out).read(), re.S)
    sizes = []
    for block in blocks:
        ops = [re.findall(r"v\[\d+:\d+\]", line)[:3] for line in block.splitlines() if "v_fmac_f64_dpp" in line]
        sizes.append(len(ops))
        for i, (written, _, _) in enumerate(ops):
            for _, a, y in ops[i + 1:]:
                assert written not in (a, y), block
    assert sorted(sizes) == [1, 1, 2, 2, 4, 4]
