"""The fp32 recurrence of launches whose workgroups are all resident: rows go to the chain and its results come
back four tokens of a channel at a time.  Ends of quads, groups and chunks, ragged channels, and channels whose
scale could become a NaN before it is clamped; bit-identical to the oracle."""
import math

import numpy as np
import pytest
import torch

from adkv_amd.train import quant_f32
from tests.test_gpu_fp32_large import NAMES, _same

pytestmark = pytest.mark.gpu


def _run(gpu, oracle, B, T, C, dtype, extra, odd, limits=(math.exp(-4.0), math.exp(4.0))):
    g = torch.Generator().manual_seed(T + C)
    p = dict(zp=0.3 * torch.randn(C, generator=g), sc=0.5 + torch.rand(C, generator=g),
             alpha=0.9 + 0.099 * torch.rand(C, generator=g), beta=0.05 * torch.rand(C, generator=g), tgt=torch.full((C,), 3.5))
    x = (torch.randn(B, T, C, generator=g) * 2.0).to(dtype)
    if odd:
        inf, nan = float("inf"), float("nan")
        # products that overflow, alone and against a zero or an opposite infinity; state and inputs that are not numbers
        for i, (k, v) in enumerate([("beta", 3e38), ("beta", inf), ("beta", nan), ("tgt", inf), ("tgt", nan), ("sc", nan),
                                    ("sc", 1e30), ("sc", inf), ("sc", -0.25), ("sc", 1e-12), ("alpha", inf), ("zp", nan),
                                    ("beta", 1e17), ("tgt", -3e38), ("beta", 0.0)]):
            p[k][(7 * i + 1) % C] = v
        p["beta"][5], p["tgt"][5], p["sc"][5] = 3e38, 2.0, 1e3
        x[0, T // 2, C - 1], x[0, T - 1, 0], x[0, 0, 9] = nan, inf, -inf
    want = oracle.quant_f32(x.float().numpy(), *[p[k].numpy() for k in NAMES], sc_min=limits[0], sc_max=limits[1], want_seq=True)
    d = {k: v.to(gpu) for k, v in p.items()}
    state = [torch.empty(B, C, device=gpu) for _ in range(2)]
    xhat, codes, zs, ss = quant_f32(x.to(gpu), d["alpha"], d["beta"], d["tgt"], -8, 7, *limits, zp_state=state[0],
                                    sc_state=state[1], zp_init=d["zp"], sc_init=d["sc"], want_codes="codes" in extra,
                                    output_states="states" in extra)
    torch.cuda.synchronize()
    assert _same(xhat, torch.from_numpy(want["xhat"]).to(dtype).float().numpy())
    assert _same(state[0], want["zp"]) and _same(state[1], want["sc"])
    if "codes" in extra:
        assert np.array_equal(codes.cpu().numpy(), want["codes"])
    if "states" in extra:
        assert _same(zs, want["zp_seq"]) and _same(ss, want["sc_seq"])


@pytest.mark.parametrize("T", (2, 3, 4, 5, 7, 8, 9, 12, 31, 32, 33, 38, 64, 71, 130))
@pytest.mark.parametrize("extra,C,dtype", [("", 64, torch.float32), ("codes", 100, torch.bfloat16), ("states", 130, torch.float16),
                                           ("codes states", 63, torch.float32)])
def test_ends(gpu, oracle, T, extra, C, dtype):
    _run(gpu, oracle, 2, T, C, dtype, extra, False)


@pytest.mark.parametrize("T", (2, 9, 33, 70))
@pytest.mark.parametrize("B", (1, 700))                      # 700: a lane per channel straight from memory
@pytest.mark.parametrize("limits", [(math.exp(-4.0), math.exp(4.0)), (0.0, 1e30), (-1e35, 8.0)])
def test_scales_that_could_overflow(gpu, oracle, T, B, limits):
    _run(gpu, oracle, B, T, 128, torch.float32, "states", True, limits)
