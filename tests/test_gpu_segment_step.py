"""adkv_decode_step in two launches (every segment through keys, softmax and values, then the segments put
together) against the three calls that it stands for and against 64 bits: every shape of its kernel, ragged and
one-token last segments, masks that leave a segment or a row nothing, non-finite logits."""
import math

import numpy as np
import pytest
import torch

from adkv_amd import _lib, synth
from adkv_amd.kernel import gemv

pytestmark = pytest.mark.gpu
SMIN, SMAX = math.exp(-4.0), math.exp(4.0)


def _case(gpu, B, Hq, H, D, T, bits=4, S=256, dtype=torch.float16, mask=None, scaling=None, q_scale=1.0, more=None):
    g = torch.Generator(device=gpu).manual_seed(T + Hq)
    kp, vp = ([t.to(gpu) for t in synth.make_params(H, D, bits=bits, seed=i).astuple()] for i in (3, 4))
    tps = 32 // bits
    k = synth.make_k(B, H, T + 1, D, seed=1, dtype=torch.float16, device=gpu)
    v = synth.make_v(B, H, T + 1, D, seed=2, dtype=torch.float16, device=gpu)
    q = (q_scale * torch.randn(B, Hq, 1, D, generator=g, device=gpu)).to(dtype)
    kn, vn = k[:, :, T:].to(dtype).contiguous(), v[:, :, T:].to(dtype).contiguous()
    caches = [synth.alloc_cache(B, H, T + tps, D, gpu, bits=bits) for _ in range(2)]
    cks = [torch.zeros(B, H, (T + tps) // S + 1, D, 2, dtype=torch.float16, device=gpu) if S else None for _ in range(2)]
    states = [torch.zeros(B, H, D, 2, dtype=torch.float16, device=gpu) for _ in range(2)]
    if T:
        gemv.append_kv_pair(*caches, k[:, :, :T], v[:, :, :T], kp, vp, 0, *states, k_ckpt=cks[0], v_ckpt=cks[1],
                            ckpt_interval=S, bits=bits)
    c2, ck2 = [c.clone() for c in caches], [c.clone() if S else None for c in cks]
    scaling = D ** -0.5 if scaling is None else scaling
    assert _lib.lib().adkv_decode_step_launches(B, Hq, H, T, D, bits, cks[0].shape[2] if S else 0, S, mask is not None) == 2
    out, w = gemv.decode_step(q, *caches, kn, vn, kp, vp, T, scaling, mask, k_ckpt=cks[0], v_ckpt=cks[1], ckpt_interval=S, bits=bits)
    logits = gemv.forward_qk(q.half(), c2[0], kn.half(), *kp, T, SMIN, SMAX, ckpt=ck2[0], ckpt_interval=S, bits=bits)
    w_want = gemv.softmax_scale_mask(logits, scaling, mask)
    o_want = gemv.forward_ov(w_want, c2[1], vn.half(), *vp, SMIN, SMAX, ckpt=ck2[1], ckpt_interval=S, bits=bits)
    torch.cuda.synchronize()
    for a, b in zip(caches, c2):
        assert torch.equal(a, b)
    for a, b in zip(cks, ck2):
        assert not S or torch.equal(a.view(torch.int16), b.view(torch.int16))
    if more is not None:
        more.update(q=q.half(), caches=caches, params=(kp, vp))
    return out.float(), w.float(), o_want.float(), w_want.float()


def _replayed(oracle, cache, params, bits, n, heads):
    """float64 [len(heads), n, D]: the oracle's values of `n` tokens of these (sequence, head)s."""
    np16 = lambda t: t.detach().cpu().contiguous().view(torch.int16).numpy().view(np.float16)
    with oracle.code_bits(bits):
        return torch.stack([torch.from_numpy(oracle.replay_f16(
            cache[b:b + 1, h:h + 1].cpu().numpy(), *[np16(p[h:h + 1]) for p in params], n)[0][0, 0]).double() for b, h in heads])


def _compare(out, w, o_want, w_want, bf16=False):
    # a logit (|l| < 64) may round the other way, 2^-5 x 128^-1/2 = 2.8e-3 of a weight; the weight itself to 2^-11 each time
    assert torch.all((w - w_want).abs() <= 4e-3 * w_want + 6e-8)
    # rows sum to one: an output moves by at most that share of the largest value (|v| < 8), and its own rounding
    tol = 4e-3 * 0.5 + (2.0 ** -8) * o_want.abs() * bf16 + 2.0 ** -10 * o_want.abs()
    assert torch.all((out - o_want).abs() <= tol), (out - o_want).abs().max()


@pytest.mark.parametrize("B,Hq,H,D,T,bits,S", [
    (1, 8, 2, 128, 0, 4, 0), (1, 8, 2, 128, 0, 4, 256), (2, 8, 2, 128, 7, 4, 256), (1, 8, 1, 128, 257, 4, 256),
    (2, 4, 2, 128, 512, 4, 256), (3, 4, 2, 128, 1025, 2, 256), (1, 8, 1, 128, 263, 4, 0), (1, 8, 1, 128, 255, 2, 0),
    (1, 4, 1, 128, 519, 4, 0), (2, 8, 1, 128, 2063, 2, 256), (5, 2, 2, 128, 700, 2, 512), (1, 3, 3, 128, 4096, 4, 256),
    (3, 32, 32, 128, 3333, 4, 256), (13, 32, 32, 128, 1999, 4, 256), (11, 32, 8, 128, 9000, 4, 256), (8, 32, 8, 128, 16001, 4, 256),
    (70, 32, 32, 128, 641, 4, 256), (33, 31, 31, 128, 1281, 4, 256),                                # four channels per lane
    (1, 2, 2, 256, 300, 4, 256), (3, 8, 8, 256, 8190, 4, 256), (16, 16, 16, 256, 3584, 4, 256),
    (1, 1, 1, 512, 519, 4, 0), (2, 3, 3, 512, 770, 4, 256), (9, 8, 8, 512, 1790, 4, 256),
])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_against_the_three_calls(gpu, oracle, B, Hq, H, D, T, bits, S, dtype):
    more = {}
    out, w, o_want, w_want = _case(gpu, B, Hq, H, D, T, bits, S, dtype, more=more)
    _compare(out, w, o_want, w_want, bf16=dtype == torch.bfloat16)
    # The outputs are sums over the returned weights, up to roundings that know nothing of each other: of the weights
    # there and here (2^-12 of each at most, or 2^-25 below 2^-14: a variance of a third of the square) and of
    # the output.  Seven deviations of the sum; a token left out is tens of them.
    heads = sorted({(0, 0), (B - 1, H - 1)})
    v = _replayed(oracle, more["caches"][1], more["params"][1], bits, T + 1, heads)
    rows = lambda t: torch.stack([t[b, h * (Hq // H):(h + 1) * (Hq // H)] for b, h in heads]).double().cpu()
    w, out = rows(w), rows(out)
    sigma = torch.sqrt(2 / 3 * (torch.clamp(w * 2.0 ** -11, min=2.0 ** -25) ** 2) @ v ** 2)
    tol = 7 * sigma + (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11) * (w @ v).abs() + 2.0 ** -25
    err = (out - w @ v).abs()
    assert torch.all(err <= tol), (err / tol).max()


@pytest.mark.parametrize("B,Hq,H,D,T,bits", [(24, 16, 2, 128, 700, 4), (24, 8, 2, 128, 2063, 2), (12, 8, 8, 256, 1290, 4),
                                             (13, 32, 32, 128, 1100, 4)])
@pytest.mark.parametrize("q_scale", [0.3, 1.0])
def test_error_against_64_bits(gpu, oracle, B, Hq, H, D, T, bits, q_scale):
    """Outputs are no further from softmax and sum in 64 bits over the cache's values than those of the three
    calls: both round a logit and a weight to fp16, by independent amounts; 5 % covers the chance in 10^5 outputs."""
    more = {}
    out, _, o_want, _ = _case(gpu, B, Hq, H, D, T, bits, q_scale=q_scale, more=more)
    heads = [(b, h) for b in range(B) for h in range(0, H, max(1, H // 4))]
    k, v = (_replayed(oracle, c, p, bits, T + 1, heads) for c, p in zip(more["caches"], more["params"]))
    rows = lambda t: torch.stack([t[b, h * (Hq // H):(h + 1) * (Hq // H)] for b, h in heads]).double().cpu()
    want = torch.softmax(rows(more["q"][:, :, 0]) @ k.transpose(1, 2).contiguous() * D ** -0.5, -1) @ v
    rms = [float(((rows(o) - want) ** 2).mean().sqrt()) for o in (out, o_want)]
    print(f"rms error {rms[0]:.3e}, of the three calls {rms[1]:.3e}, of a value of {float((want ** 2).mean().sqrt()):.3e}")
    assert rms[0] <= 1.05 * rms[1]


@pytest.mark.parametrize("low", [torch.finfo(torch.float32).min, torch.finfo(torch.bfloat16).min, -math.inf])
@pytest.mark.parametrize("B,Hq,H,D,T", [(3, 8, 2, 128, 1000), (2, 8, 8, 256, 777), (33, 32, 32, 128, 1025)])
def test_masked_segments_and_rows(gpu, B, Hq, H, D, T, low):
    mask = torch.zeros(B, 1, 1, T + 1, device=gpu)
    mask[0, ..., :300] = low                 # a whole segment and a part of the next
    mask[1, ..., 5::3] = low
    if B > 2:
        mask[2] = low                        # a whole row: uniform weights, or NaN for -inf
    r = _case(gpu, B, Hq, H, D, T, mask=mask)
    if B > 2 and low == -math.inf:
        for t in r:
            assert torch.all(torch.isnan(t[2]))
        r = [torch.cat([t[:2], t[3:]]) for t in r]
    for t in r:
        assert torch.all(torch.isfinite(t))
    _compare(*r)


def test_infinite_logits_and_zero_scaling(gpu):
    out, w, o_want, w_want = _case(gpu, 2, 8, 2, 128, 600, q_scale=3e4)      # logits overflow fp16
    assert torch.equal(torch.isnan(w), torch.isnan(w_want)) and torch.equal(torch.isnan(out), torch.isnan(o_want))
    assert torch.any(torch.isnan(w))
    _compare(*_case(gpu, 2, 8, 2, 128, 600, scaling=0.0))
    _compare(*_case(gpu, 2, 8, 8, 256, 600, scaling=-0.05))
