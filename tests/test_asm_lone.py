"""The blocks of one channel per lane, as the assembler gets them (see test_asm_blocks)."""
import os
import re
import shutil
import subprocess

import pytest

from tests.test_asm_blocks import CSRC, _needs_wait

PROBE = """
#include "%s"
using namespace adkv;
__global__ void keys(Lone *s, const uint2 *e, uint32_t *x) { lone_eight(s[threadIdx.x], e + 4 * threadIdx.x, x + 4 * threadIdx.x); }
__global__ void columns(Lone *s, const uint2 *e, uint32_t *x) { lone_eight<true>(s[threadIdx.x], e + 4 * threadIdx.x, x + 4 * threadIdx.x); }
__global__ void values(Lone *s, const uint2 *e, const uint4 *w, float *acc) {
    lone_eight_weighted(s[threadIdx.x], e + 4 * threadIdx.x, w[threadIdx.x], acc[threadIdx.x]);
}
"""


def test_results_are_waited_for(tmp_path):
    if shutil.which("hipcc") is None:
        pytest.skip("no hipcc")
    (tmp_path / "probe.hip").write_text(PROBE % os.path.join(CSRC, "adkv_device.h"))
    subprocess.run(["hipcc", "-O3", "--offload-arch=gfx950", "-std=c++17", "-ffp-contract=off", "-Xclang", "-target-feature",
                    "-Xclang", "-packed-fp32-ops", "--cuda-device-only", "-S", "-o", str(tmp_path / "probe.s"), str(tmp_path / "probe.hip")],
                   check=True, capture_output=True)
    found = re.findall(r"#ASMSTART\n(.*?)\n\s*;;?#ASMEND", (tmp_path / "probe.s").read_text(), re.S)
    found = [[l.strip() for l in b.strip().split("\n")] for b in found]
    found = [b for b in found if len(b) > 8]
    assert len(found) == 3
    assert [b[-1] for b in found].count("s_nop 1") == 1        # ahead of a matrix instruction
    for b in found:
        assert sum(i.startswith("v_pk_") for i in b) == 24
        for a, nxt in zip(b, b[1:]):
            reg = _needs_wait(a)
            assert reg is None or not re.search(rf"\b{reg}\b", nxt.split(None, 1)[1]), (a, nxt)
        assert _needs_wait(b[-1]) is None
