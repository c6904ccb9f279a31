"""The fp32 recurrence in launches with more workgroups than are resident at once (1024, 512 with codes or
states, 256 with both, on 256 CUs), which take a lane per channel straight from memory in groups of 8 tokens:
bit-identical to the oracle like the others."""
import math

import numpy as np
import pytest
import torch

from adkv_amd.train import quant_f32
from adkv_amd.train.train_model import quant_f32_pair

pytestmark = pytest.mark.gpu

NAMES = ("zp", "sc", "alpha", "beta", "tgt")
C = 1000   # 16 blocks of 64 channels, the last one ragged


def _params(seed, bits=4):
    g = torch.Generator().manual_seed(seed)
    return dict(zp=0.3 * torch.randn(C, generator=g), sc=0.5 + torch.rand(C, generator=g),
                alpha=0.9 + 0.099 * torch.rand(C, generator=g), beta=0.05 * torch.rand(C, generator=g),
                tgt=torch.full((C,), (2 ** (bits - 1) - 1) / 2.0))


def _stream(B, T, p, seed):
    """Ordinary rows with what makes a group be repeated: ties of the first token and their neighbours,
    and non-finite inputs in the first, a middle and the last group."""
    x = torch.randn(B, T, C, generator=torch.Generator().manual_seed(seed)) * 2.0
    tie = p["zp"] + (torch.arange(C) % 16 - 7.5) * p["sc"]
    x[0, 0] = tie
    x[1, 0] = torch.nextafter(tie, torch.full_like(tie, 1e9))
    for i, t in enumerate((1, T // 2, T - 1)):
        x[2 + i, t, 3 + i] = (float("nan"), float("inf"), -1.0e30)[i]
        x[B - 1 - i, t, C - 1 - i] = (float("inf"), float("nan"), 3.0e38)[i]
    return x


def _same(got, want):
    g, w = got.detach().float().cpu().numpy(), np.asarray(want, dtype=np.float32)
    both_nan = np.isnan(g) & np.isnan(w)
    return np.array_equal(np.where(both_nan, 0, g.view(np.int32)), np.where(both_nan, 0, w.view(np.int32)))


@pytest.mark.parametrize("T", (2, 7, 8, 9, 16, 17, 24, 33, 64))
@pytest.mark.parametrize("extra,B", [("", 65), ("codes", 33), ("states", 33), ("codes states", 17)])
def test_one_tensor(gpu, oracle, extra, B, T):
    p = _params(T)
    x = _stream(B, T, p, T)
    want = oracle.quant_f32(x.numpy(), *[p[k].numpy() for k in NAMES], want_seq=True)
    state = [torch.empty(B, C, device=gpu) for _ in range(2)]
    d = {k: v.to(gpu) for k, v in p.items()}
    xhat, codes, zs, ss = quant_f32(x.to(gpu), d["alpha"], d["beta"], d["tgt"], -8, 7, math.exp(-4.0), math.exp(4.0),
                                    zp_state=state[0], sc_state=state[1], zp_init=d["zp"], sc_init=d["sc"],
                                    want_codes="codes" in extra, output_states="states" in extra)
    torch.cuda.synchronize()
    assert _same(xhat, want["xhat"]) and _same(state[0], want["zp"]) and _same(state[1], want["sc"])
    assert np.isnan(want["zp"]).any()
    if "codes" in extra:
        assert np.array_equal(codes.cpu().numpy(), want["codes"])
    if "states" in extra:
        assert _same(zs, want["zp_seq"]) and _same(ss, want["sc_seq"])


@pytest.mark.parametrize("dtype", (torch.float32, torch.float16, torch.bfloat16))
@pytest.mark.parametrize("T", (3, 16, 41))
@pytest.mark.parametrize("in_place", (True, False))
def test_pair(gpu, oracle, dtype, T, in_place):
    """K and V in one launch, in place on a strided view or from rows of another pitch; a scale under its
    floor to start from."""
    B = 33
    tensors, wants = [], []
    for i in range(2):
        p = _params(40 + i)
        p["sc"][::5] = -0.25
        x = _stream(B, T, p, T + i).to(dtype)
        wants.append(oracle.quant_f32(x.float().numpy(), *[p[k].numpy() for k in NAMES]))
        src = torch.zeros(B, T + 5, C + 3, dtype=dtype, device=gpu)[:, :T, :C]
        src.copy_(x)
        dst = src if in_place else torch.zeros(B, T + 3, C, dtype=dtype, device=gpu)[:, :T]
        tensors.append((src, dst, {k: v.to(gpu) for k, v in p.items()}, [torch.empty(B, C, device=gpu) for _ in range(2)]))
    quant_f32_pair([t[0] for t in tensors], [(t[2]["alpha"], t[2]["beta"], t[2]["tgt"]) for t in tensors], -8, 7,
                   math.exp(-4.0), math.exp(4.0), states=[t[3] for t in tensors], out=[t[1] for t in tensors],
                   init=[(t[2]["zp"], t[2]["sc"]) for t in tensors])
    torch.cuda.synchronize()
    for (_, dst, _, (zp, sc)), want in zip(tensors, wants):
        assert _same(dst, torch.from_numpy(want["xhat"]).to(dtype).float())
        assert torch.count_nonzero(dst._base[:, T:]) == 0 and torch.count_nonzero(dst._base[:, :, C:]) == 0
        assert _same(zp, want["zp"]) and _same(sc, want["sc"])


def test_scale_floor_inside_the_limits(gpu, oracle):
    """sc_min below 1e-8: the scale that divides and the scale that is kept are two numbers."""
    B, T = 65, 40
    p = _params(9)
    p["sc"][::3] = 0.0
    p["beta"][::7] = 0.0
    x = torch.randn(B, T, C, generator=torch.Generator().manual_seed(1)) * 2.0
    want = oracle.quant_f32(x.numpy(), *[p[k].numpy() for k in NAMES], sc_min=0.0, sc_max=8.0)
    d = {k: v.to(gpu) for k, v in p.items()}
    zp, sc = torch.empty(B, C, device=gpu), torch.empty(B, C, device=gpu)
    xhat, _, _, _ = quant_f32(x.to(gpu), d["alpha"], d["beta"], d["tgt"], -8, 7, 0.0, 8.0, zp_state=zp, sc_state=sc,
                              zp_init=d["zp"], sc_init=d["sc"])
    torch.cuda.synchronize()
    assert _same(xhat, want["xhat"]) and _same(zp, want["zp"]) and _same(sc, want["sc"])
