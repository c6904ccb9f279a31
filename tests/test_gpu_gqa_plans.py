"""Launches of four channels per lane whose segments are nearly equal, or more groups of uneven ones than the even plan has: against
the same calls without checkpoints, one segment.  The last shape is a shared-table launch, the others are matrix-core ones."""
import ctypes
import math

import pytest
import torch

from adkv_amd import _lib, synth
from adkv_amd.kernel import gemv

SMIN, SMAX = math.exp(-4.0), math.exp(4.0)
# sequences, query heads, KV heads, tokens, interval, bits -> segments, balanced
SHAPES = [((17, 32, 8, 3899, 64, 4), 60, True), ((17, 16, 8, 3904, 64, 2), 60, True), ((17, 8, 8, 3841, 64, 2), 60, True),
          ((34, 32, 8, 961, 16, 4), 28, False), ((128, 8, 2, 1257, 16, 4), 32, False), ((69, 8, 2, 2912, 16, 4), 56, False),
          ((10, 32, 32, 1257, 16, 4), 25, True)]


def _bounds(B, Hq, H, T, S, bits):
    b = (ctypes.c_int * 600)()
    n = _lib.lib().adkv_decode_segments(B, Hq, H, T, 128, bits, T // S + 1, S, b, 600, None)
    return list(b[:n + 1])


@pytest.mark.parametrize("sizes,n,balanced", SHAPES)
def test_plans(sizes, n, balanced):
    """Without a GPU (256 CUs)."""
    T, S = sizes[3], sizes[4]
    b = _bounds(*sizes)
    assert len(b) == n + 1 and b[0] == 0 and b[-1] == T and not any(x % S for x in b[:-1])
    lens = [(y - x + S - 1) // S for x, y in zip(b, b[1:])]
    assert sum(lens) == (T + S - 1) // S and min(lens) >= 1
    assert (max(lens) - min(lens) <= 1) == balanced
    if not balanced:                                       # shares of the wave slots, the oldest slot's last in its group
        assert n % 4 == 0 and all(lens[i] <= lens[i + 3] for i in range(0, n, 4))


@pytest.mark.gpu
@pytest.mark.parametrize("sizes,n,balanced", SHAPES)
def test_against_one_segment(gpu, sizes, n, balanced):
    B, Hq, H, T, S, bits = sizes
    D, tps = 128, 32 // bits
    kp, vp = ([t.to(gpu) for t in synth.make_params(H, D, bits=bits, seed=i).astuple()] for i in (3, 4))
    k, v = (f(B, H, T + 1, D, seed=i, dtype=torch.float16, device=gpu) for i, f in enumerate((synth.make_k, synth.make_v)))
    g = torch.Generator(device=gpu).manual_seed(5)
    q = torch.randn(B, Hq, 1, D, generator=g, device=gpu).half()
    caches = [synth.alloc_cache(B, H, T + tps, D, gpu, bits=bits) for _ in "kv"]
    cks = [torch.zeros(B, H, (T + tps) // S + 1, D, 2, dtype=torch.float16, device=gpu) for _ in "kv"]
    states = [torch.zeros(B, H, D, 2, dtype=torch.float16, device=gpu) for _ in "kv"]
    gemv.append_kv_pair(*caches, k[:, :, :T], v[:, :, :T], kp, vp, 0, *states, k_ckpt=cks[0], v_ckpt=cks[1], ckpt_interval=S, bits=bits)
    kn, vn = k[:, :, T:].contiguous(), v[:, :, T:].contiguous()
    c1 = [c.clone() for c in caches]
    logits = gemv.forward_qk(q, caches[0], kn, *kp, T, SMIN, SMAX, ckpt=cks[0], ckpt_interval=S, bits=bits)
    want = gemv.forward_qk(q, c1[0], kn, *kp, T, SMIN, SMAX, bits=bits)
    # two sums of the same 128 products in fp32, a rounding to fp16 each
    assert torch.all((logits.float() - want.float()).abs() <= 2.0 ** -10 * want.float().abs() + 2.0 ** -9)
    w = gemv.softmax_scale_mask(want, D ** -0.5)
    out = gemv.forward_ov(w, caches[1], vn, *vp, SMIN, SMAX, ckpt=cks[1], ckpt_interval=S, bits=bits)
    o_want = gemv.forward_ov(w, c1[1], vn, *vp, SMIN, SMAX, bits=bits)
    # sums of the same products in fp32 in another order (|v| < 16, weights that sum to one), a rounding to fp16 each
    assert torch.all((out.float() - o_want.float()).abs() <= 2.0 ** -10 * o_want.float().abs() + 2.0 ** -17)
    for a, b in zip(caches, c1):
        assert torch.equal(a, b)
