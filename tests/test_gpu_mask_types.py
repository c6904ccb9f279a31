"""Masks of fp16 and bfloat16 are widened as they are read: every launch that a step can take gives the bits that
the same mask in fp32 gives, rows of odd lengths included."""
import pytest
import torch

from adkv_amd import _lib, synth
from adkv_amd.kernel import gemv

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mask_dtype", (torch.float16, torch.bfloat16, torch.float64))
@pytest.mark.parametrize("per_head", (False, True))
@pytest.mark.parametrize("launches,B,Hq,H,T,S", [
    (1, 2, 3, 3, 0, 0), (1, 2, 3, 3, 6, 256), (1, 2, 3, 3, 530, 256), (1, 3, 4, 4, 777, 256),
    (2, 2, 8, 2, 300, 256), (2, 2, 8, 1, 1201, 256), (2, 3, 4, 4, 1777, 256),
    (3, 2, 2, 2, 530, 64), (3, 3, 32, 32, 1030, 64),                 # a wave per row
    (3, 1, 3, 3, 4096, 64), (3, 2, 2, 2, 9001, 0),                   # a workgroup per row
    (3, 1, 2, 2, 30001, 0), (3, 1, 2, 2, 61003, 64)])                # rows in chunks
def test_same_bits_as_fp32(gpu, mask_dtype, per_head, launches, B, Hq, H, T, S):
    D, n = 128, T + 1
    g = torch.Generator().manual_seed(T)
    kp, vp = ([t.to(gpu) for t in synth.make_params(H, D, seed=i).astuple()] for i in (3, 4))
    k = synth.make_k(B, H, n, D, seed=1, dtype=torch.float16, device=gpu)
    v = synth.make_v(B, H, n, D, seed=2, dtype=torch.float16, device=gpu)
    q = torch.randn(B, Hq, 1, D, generator=g).half().to(gpu)
    caches = [synth.alloc_cache(B, H, T + 8, D, gpu) for _ in range(2)]
    cks = [torch.zeros(B, H, (T + 8) // S + 1, D, 2, dtype=torch.float16, device=gpu) if S else None for _ in range(2)]
    states = [torch.zeros(B, H, D, 2, dtype=torch.float16, device=gpu) for _ in range(2)]
    if T:
        gemv.append_kv_pair(*caches, k[:, :, :T], v[:, :, :T], kp, vp, 0, *states, k_ckpt=cks[0], v_ckpt=cks[1], ckpt_interval=S)
    mask = torch.randn(B, Hq if per_head else 1, 1, n, generator=g)
    mask[0, :, :, : n // 3] = torch.finfo(torch.float16).min
    mask[-1, :, :, n - 1 - n // 5:n - 1] = -float("inf")
    mask = mask.to(mask_dtype).to(gpu)
    assert _lib.lib().adkv_decode_step_launches(B, Hq, H, T, D, 4, cks[0].shape[2] if S else 0, S, 1) == launches
    got = []
    for m in (mask, mask.float()):
        c = [t.clone() for t in caches]
        got.append(gemv.decode_step(q, *c, k[:, :, T:].contiguous(), v[:, :, T:].contiguous(), kp, vp, T, D ** -0.5, m,
                                    k_ckpt=cks[0], v_ckpt=cks[1], ckpt_interval=S))
    torch.cuda.synchronize()
    for a, b in zip(*got):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))
        assert torch.isfinite(a).all()
