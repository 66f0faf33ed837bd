"""What the compiler makes of kernels whose speed hangs on their values staying in registers: no scratch memory.  Host only (the
device code is compiled, not run)."""
import os
import re
import subprocess

import pytest

from terapipe_amd import build


@pytest.mark.parametrize("source,kernel", [("layernorm.hip", r"ln_fwd_kernel|ln_bwd_rows_kernel")], ids=["layernorm"])
def test_no_scratch_memory(source, kernel, tmp_path):
    try:
        hipcc = build.hipcc_path()
    except RuntimeError:
        pytest.skip("no hipcc")
    out = subprocess.run([hipcc] + build.HIPCC_FLAGS + ["-Rpass-analysis=kernel-resource-usage", "--cuda-device-only", "-c",
                          os.path.join(build.CSRC, source), "-o", str(tmp_path / "out.o")], capture_output=True, text=True, check=True).stderr
    found = re.findall(r"Function Name: (\S+).*?ScratchSize \[bytes/lane\]: (\d+)", out, re.S)
    named = {name: int(size) for name, size in found if re.search(kernel, name)}
    assert len(named) >= 6 and not any(named.values()), named
