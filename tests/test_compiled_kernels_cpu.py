"""What has to hold of the machine code of the kernels, looked up in the library as it is built: waits that keep LDS reads and writes of
different wavefronts apart, which no result shows to be missing as long as the loads behind them are slow."""

import os
import re
import subprocess

import pytest

from paged_attention_engine_amd.kernels import build

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


def functions_of(folder, name):
    """{symbol: instructions} of the library's device functions whose symbol holds `name`."""
    lib = os.path.join(folder, "lib.so")
    os.symlink(build.ensure_built(), lib)
    subprocess.run([OBJDUMP, "--offloading", lib], check=True, capture_output=True, cwd=folder)
    out = {}
    for part in sorted(os.listdir(folder)):
        if not part.endswith(build.ARCH):
            continue
        symbols = subprocess.run([OBJDUMP, "-t", part], check=True, capture_output=True, text=True, cwd=folder).stdout
        if name not in symbols:
            continue
        text = subprocess.run([OBJDUMP, "-d", part], check=True, capture_output=True, text=True, cwd=folder).stdout
        for head, body in re.findall(r"^[0-9a-f]+ <([^>]+)>:\n(.*?)(?=^[0-9a-f]+ <|\Z)", text, re.M | re.S):
            if name in head:
                out[head] = [line.split("//")[0].strip() for line in body.splitlines() if line.strip()]
    return out


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no disassembler")
def test_no_barrier_of_the_large_tiles_is_passed_with_a_read_of_what_is_written_next(tmp_path):
    """The halves of a workgroup's wavefronts lie one barrier apart, and a half of the stage's rows is written again while
    the later ones' next products wait for what they read.  At a barrier a wavefront may have asked LDS for the eight operands that it read last,
    and for nothing older: LDS answers in order, so counting is enough."""
    kernels = functions_of(tmp_path, "wide_large_kernel")
    assert len(kernels) >= 15  # five kinds of result by three ways to cut what is left over
    for name, code in kernels.items():
        asked, most = 0, 0
        for line in code:
            if line.startswith("ds_read"):
                asked += 1
            elif line.startswith("s_waitcnt"):
                wait = re.search(r"lgkmcnt\((\d+)\)", line)
                asked = min(asked, int(wait.group(1))) if wait else asked
            elif line == "s_barrier":
                most = max(most, asked)
        assert most == 8, (name, most)
