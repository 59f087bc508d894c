"""Registers of kernels whose speed hangs on the waves a SIMD holds, as the compiler reports them (no GPU)."""
import os
import re
import subprocess

import pytest

from loken_amd import build


@pytest.mark.skipif(not os.path.exists(build.HIPCC), reason="needs hipcc")
def test_q4_k_down_and_fold_holds_two_waves_a_simd(tmp_path):
    # Two workgroups of four waves a CU is what the launch's count of passes assumes. One wave a SIMD (more than 256
    # registers) cost rows of four super-blocks 9 to 14 % of the launch; a spill costs scratch traffic instead.
    run = subprocess.run([build.HIPCC, *build.FLAGS, "-S", "--offload-device-only", "-Rpass-analysis=kernel-resource-usage",
                          "-o", str(tmp_path / "fold.s"), str(build.CSRC / "moe_down_fold.hip")], capture_output=True, text=True)
    assert run.returncode == 0, run.stderr[-2000:]
    kernels = {}
    for part in re.split(r"Function Name: ", run.stderr)[1:]:
        name = part.split()[0]
        kernels[name] = (int(re.search(r"Occupancy \[waves/SIMD\]: (\d+)", part)[1]), int(re.search(r"VGPRs Spill: (\d+)", part)[1]))
    q4_k = {n: v for n, v in kernels.items() if "moe_down_fold_kernel" in n and "LaneQ4KILb0E" in n}
    assert len(q4_k) == 6   # rows of two, three and four super-blocks, up to four and up to eight pairs a token
    assert all(waves >= 2 for waves, _ in q4_k.values()), q4_k
    assert all(spill == 0 for _, spill in kernels.values()), kernels
