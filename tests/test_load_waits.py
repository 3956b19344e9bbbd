"""Loads written in inline assembly whose results nobody reads any more: the compiler takes their registers as free while
they are still on their way, so nothing may be put there before the wait that ends a kernel's main loop.  Looked up in the
device assembly of the kernels that have such loads."""
import os
import re
import subprocess

import pytest

from minit_amd import build

WRITES = re.compile(r"v_(?!mfma)")   # accumulators are no targets of loads


@pytest.mark.parametrize("source,kernel,count", [("gptq_gemm_tall.hip", "gptq_gemm_tall_kernel", 8),
                                                 ("gptq_gemm_wide.hip", "gptq_gemm_wide_kernel", 2)])
def test_nothing_is_put_into_registers_of_loads_in_flight(tmp_path, source, kernel, count):
    out = tmp_path / "device.s"
    subprocess.run([build.find_hipcc(), *build.HIPCC_FLAGS, "--cuda-device-only", "-S", os.path.join(build.CSRC, source),
                    "-o", str(out)], check=True, capture_output=True, timeout=300)
    lines = out.read_text().split("\n")
    found, name = {}, None
    for i, line in enumerate(lines):
        if line.startswith("_Z") and ":" in line:
            name = line.split(":")[0]
        if "s_waitcnt vmcnt(0)" in line and "#ASMSTART" in lines[i - 1]:
            # back to the end of the last round: a branch, its target or the barrier
            between, j = [], i - 2
            while not lines[j].startswith(".LBB") and "s_cbranch" not in lines[j] and "s_barrier" not in lines[j]:
                if WRITES.match(lines[j].strip()):
                    between.append(lines[j].strip())
                j -= 1
            found[name] = between   # the last such wait of a kernel is the one behind its main loop
    kernels = {n: b for n, b in found.items() if kernel in n}
    assert len(kernels) == count
    assert not any(kernels.values()), kernels
