"""The hand-laid instruction blocks of adkv_device.h, as the assembler gets them: the hardware does not
wait by itself where the result of a transcendental, packed or half-register instruction is read by the
very next instruction, the compiler does not look inside a block, and a block does not know what comes
after it."""
import os
import re
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "adkv_amd", "csrc")

PROBE = """
#include "%s"
using namespace adkv;
template <int BITS> __global__ void enc(Chan1 *c, const uint16_t *x, uint32_t *p, float *f) {
    uint16_t y[8];
    for (int i = 0; i < 8; i++) y[i] = x[i * 64 + threadIdx.x];
    Chan1 ch = c[threadIdx.x];
    uint32_t w = 0;
    float nan = 0;
    enc_eight_tokens<BITS>(ch, y, p[0], p[1], p[2], f[0], f[1 + threadIdx.x], w, nan);
    c[threadIdx.x] = ch;
    p[3 + threadIdx.x] = w;
    f[100 + threadIdx.x] = nan;
}
template __global__ void enc<2>(Chan1 *, const uint16_t *, uint32_t *, float *);
template __global__ void enc<4>(Chan1 *, const uint16_t *, uint32_t *, float *);
__global__ void rep(Pair *p, const uint2 *e, uint32_t *x) { replay_eight(p[threadIdx.x], e + 8 * threadIdx.x, x + 8 * threadIdx.x); }
__global__ void repw(Pair *p, const uint2 *e, const uint4 *w, float *acc) {
    replay_eight_weighted(p[threadIdx.x], e + 8 * threadIdx.x, w[threadIdx.x], acc + 2 * threadIdx.x);
}
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
    text = (d / "probe.s").read_text()
    found = [[l.strip() for l in b.strip().split("\n")] for b in re.findall(r"#ASMSTART\n(.*?)\n\s*;;?#ASMEND", text, re.S)]
    found = [b for b in found if len(b) > 8]
    assert len(found) == 4   # two widths of the encoder, two replays
    return found


def _needs_wait(ins):
    """The register an instruction writes whose reader must not come next, or None."""
    op, *args = re.split(r"[ ,]+", ins)
    packed, half = op.startswith("v_pk_"), op in ("v_fma_f16",) or "dst_sel:WORD" in ins
    return args[0] if packed or half or op.startswith(("v_rcp", "v_exp", "v_log", "v_rsq", "v_sqrt", "v_sin", "v_cos")) else None


def test_no_result_is_read_too_early(blocks):
    for b in blocks:
        for a, nxt in zip(b, b[1:]):
            reg = _needs_wait(a)
            assert reg is None or not re.search(rf"\b{reg}\b", nxt.split(None, 1)[1]), (a, nxt)


def test_no_result_is_left_to_what_follows(blocks):
    for b in blocks:
        assert _needs_wait(b[-1]) is None, b[-1]
