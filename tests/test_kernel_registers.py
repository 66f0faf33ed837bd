"""Kernels whose speed hangs on their values staying in registers, and on how many of their workgroups share a CU: no scratch memory,
and no more registers than that number leaves.  Host only (the device code is compiled, not run)."""
import os
import re
import subprocess

import pytest

from terapipe_amd import build


@pytest.mark.parametrize("source,kernels", [
    # up to 16 rows two workgroups of eight waves share a CU; tiles of 8 weight rows have one to themselves
    ("gemm_skinny.hip", [(r"gemm_skinny_kernelI\w+?Li1ELi[124]ELb0E", 12, 128), (r"gemm_skinny_kernel", 22, 256)]),
    # two of four waves, three at head dimension 64; one of eight
    ("attention_long.hip", [(r"attn_dq_long_kernel", 16, 256), (r"attn_dq_long_kernelI\w+?Li64E", 4, 168), (r"attn_dq_pairs_kernel", 8, 256)])],
    ids=["few rows", "dq"])
def test_registers(source, kernels, tmp_path):
    try:
        hipcc = build.hipcc_path()
    except RuntimeError:
        pytest.skip("no hipcc")
    out = subprocess.run([hipcc] + build.HIPCC_FLAGS + ["-Rpass-analysis=kernel-resource-usage", "--cuda-device-only", "-c",
                          os.path.join(build.CSRC, source), "-o", str(tmp_path / "out.o")], capture_output=True, text=True, check=True).stderr
    found = re.findall(r"Function Name: (\S+).*?VGPRs: (\d+).*?ScratchSize \[bytes/lane\]: (\d+)", out, re.S)
    for kernel, count, registers in kernels:
        named = {name: (int(used), int(scratch)) for name, used, scratch in found if re.search(kernel, name)}
        assert len(named) == count and all(used <= registers and not scratch for used, scratch in named.values()), named
