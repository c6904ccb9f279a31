"""The 64-token block of the encoder, as the assembler gets it: results that need a wait (see test_asm_blocks),
and rows that are read only after the wait for them."""
import os
import re
import shutil
import subprocess

import pytest

from tests.test_asm_blocks import CSRC, _needs_wait

PROBE = """
#include "%s"
using namespace adkv;
template <int BITS, bool BF16> __global__ void run(Chan1Neg *c, uint32_t *p, float *f) {
    Chan1Neg ch = c[threadIdx.x];
    uint32_t w[32 / (32 / BITS) * 2];
    float nan = 0;
    enc_run64<BITS, BF16>(ch, p[0], p[1], p[2], p[3], f[0], f[1], f[2 + threadIdx.x], w, nan);
    c[threadIdx.x] = ch;
    for (int k = 0; k < 2 * BITS; k++) p[64 * k + threadIdx.x] = w[k];
    f[100 + threadIdx.x] = nan;
}
template __global__ void run<2, false>(Chan1Neg *, uint32_t *, float *);
template __global__ void run<2, true>(Chan1Neg *, uint32_t *, float *);
template __global__ void run<4, false>(Chan1Neg *, uint32_t *, float *);
template __global__ void run<4, true>(Chan1Neg *, uint32_t *, float *);
"""


@pytest.fixture(scope="module")
def blocks(tmp_path_factory):
    if shutil.which("hipcc") is None:
        pytest.skip("no hipcc")
    d = tmp_path_factory.mktemp("asm")
    (d / "probe.hip").write_text(PROBE % os.path.join(CSRC, "adkv_device.h"))
    subprocess.run(["hipcc", "-O3", "--offload-arch=gfx950", "-std=c++17", "-ffp-contract=off", "-Xclang", "-target-feature",
                    "-Xclang", "-packed-fp32-ops", "--cuda-device-only", "-S", "-o", str(d / "probe.s"), str(d / "probe.hip")],
                   check=True, capture_output=True)
    found = re.findall(r"#ASMSTART\n(.*?)\n\s*;;?#ASMEND", (d / "probe.s").read_text(), re.S)
    found = [[l.strip() for l in b.strip().split("\n") if l.strip()] for b in found]
    found = [b for b in found if len(b) > 500]
    assert len(found) == 4
    return found


def test_results_and_rows_are_waited_for(blocks):
    for b in blocks:
        assert sum("v_alignbit" in i for i in b) == 64 and sum("ds_read_b64_tr_b16" in i for i in b) == 16
        for a, nxt in zip(b, b[1:]):
            reg = _needs_wait(a)
            if a.startswith(("v_pk_", "v_cvt_pk_")):
                reg = re.split(r"[ ,]+", a)[1]
            assert reg is None or not re.search(rf"\b{reg}\b", nxt.split(None, 1)[1]), (a, nxt)
        assert _needs_wait(b[-1]) is None
        pending = set()
        for i in b:
            regs = {int(r) for r in re.findall(r"\bv(\d+)\b", i)} | {
                r for lo, hi in re.findall(r"v\[(\d+):(\d+)\]", i) for r in range(int(lo), int(hi) + 1)}
            if i.startswith("ds_read"):
                dst = re.search(r"v\[(\d+):(\d+)\]", i)
                pending |= set(range(int(dst[1]), int(dst[2]) + 1))
            elif i.startswith("s_waitcnt"):
                assert "lgkmcnt(0)" in i
                pending = set()
            else:
                assert not regs & pending, (i, pending)
        assert not pending
