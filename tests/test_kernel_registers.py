"""Kernels whose early loads live in registers: none is spilled, and as many
blocks fit a CU as did when they were read late.  By the compiler's own report."""

import os
import re
import subprocess

import pytest

from csrc.build import CSRC, FLAGS


@pytest.fixture(scope="module")
def kernels():
    p = subprocess.run(
        ["hipcc", *FLAGS, "--offload-device-only", "-S", "-o", os.devnull,
         "-Rpass-analysis=kernel-resource-usage",
         os.path.join(CSRC, "gqa_attn.hip")], capture_output=True, text=True)
    assert p.returncode == 0, p.stderr[-2000:]
    out = {}
    for line in p.stderr.splitlines():
        name = re.search(r"Function Name: (\S+)", line)
        if name:
            now = out[name.group(1)] = {}
        for key in ("VGPRs Spill", "Occupancy [waves/SIMD]"):
            n = re.search(re.escape(key) + r": (\d+)", line)
            if n:
                now[key.split()[0]] = int(n.group(1))
    return out


# waves a SIMD of keys and values of each padded size (a block has one on each)
@pytest.mark.parametrize("kind,DP,VP,waves", [
    ("f", 64, 64, 3), ("f", 64, 128, 2), ("f", 128, 64, 2), ("f", 128, 128, 1),
    ("f", 256, 256, 1), ("t", 64, 64, 4), ("t", 64, 128, 2), ("t", 128, 64, 3),
    ("t", 128, 128, 2), ("t", 256, 256, 1)])
def test_new_tokens_attention(kernels, kind, DP, VP, waves):
    k = [v for n, v in kernels.items()
         if f"k_gqa_tokenI{kind}Li{DP}ELi{VP}E" in n]
    assert len(k) == 1
    assert k[0]["VGPRs"] == 0 and k[0]["Occupancy"] >= waves
