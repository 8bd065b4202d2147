"""CPU tests of the loads from global memory straight into LDS: a scalar write of M0 needs one wait state before the load
that takes its LDS address from it, and the compiler does not look into assembly strings."""
import glob
import os
import re
import shutil
import subprocess

import pytest

from conftest import PKG

CSRC = os.path.join(PKG, "csrc")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

USES = r"""
#include "abq_lds_dma.h"
using namespace abq;
extern "C" __global__ void uses(const char *base, const uint32_t *off, unsigned at, unsigned *out)
{
    extern __shared__ unsigned smem[];
    const uint32_t o = off[threadIdx.x];
    lds_dma16(base + o, at);
    lds_dma16(base, o, at + 1024);
    lds_dma4(base, o, at + 2048);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    out[threadIdx.x] = smem[threadIdx.x];
}
"""


def instructions(asm):
    """mnemonic and operands of each instruction, comments, labels and directives left out"""
    for line in asm.splitlines():
        line = re.split(r";|//", line)[0].strip()
        if line and not line.startswith(".") and not line.endswith(":"):
            yield line


def loads_without_wait_state(code):
    """LDS loads whose M0 was written by the instruction in front of them"""
    code = list(code)
    return [i for i, c in enumerate(code) if i and re.match(r"(global|buffer|scratch)_load_lds", c) and re.match(r"s_\w+ m0\b", code[i - 1])]


def test_the_scan_itself():
    bad = ["s_mov_b32 m0, s0", "global_load_lds_dword v0, s[2:3]"]
    assert loads_without_wait_state(bad) == [1] and not loads_without_wait_state([bad[0], "s_nop 0", bad[1]])


def test_no_source_writes_m0_right_before_a_load_into_lds():
    seen = 0
    for path in sorted(glob.glob(os.path.join(CSRC, "*.h")) + glob.glob(os.path.join(CSRC, "*.hip"))):
        for string in re.findall(r'asm volatile\(((?:\s*"(?:[^"\\]|\\.)*")+)', open(path).read()):
            code = [s for s in re.split(r"\\n|\\t|;", re.sub(r'"\s*"', "", string).strip().strip('"')) if s.strip()]
            seen += any("m0" in c for c in code)
            assert not loads_without_wait_state(code), (os.path.basename(path), string)
    assert seen == 3  # the helpers of abq_lds_dma.h, and nothing beside them


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs hipcc")
def test_compiled_loads_into_lds_keep_the_wait_state(tmp_path):
    src, out = tmp_path / "uses.hip", tmp_path / "uses.s"
    src.write_text(USES)
    subprocess.check_call([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-I" + CSRC, "--offload-device-only", "-S", str(src), "-o", str(out)])
    code = list(instructions(out.read_text()))
    assert sum("load_lds" in c for c in code) == 3
    assert not loads_without_wait_state(code), code
