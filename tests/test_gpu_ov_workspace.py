"""forward_ov of launches whose best number of segments is not that of the equal ones: with a workspace for either number, and
refused with less than the equal ones take, also where it runs fewer."""
import math

import pytest
import torch

from adkv_amd import _lib, synth
from adkv_amd.kernel import gemv

pytestmark = pytest.mark.gpu
E_WORKSPACE, E_ALIGN = -7, -5
# sequences, query heads, KV heads, tokens, interval, bits -> equal segments, those of the full workspace's plan
SHAPES = [((17, 32, 8, 3899, 64, 4), 61, 60), ((17, 16, 8, 3904, 64, 2), 61, 60), ((34, 32, 8, 961, 16, 4), 61, 28),
          ((128, 8, 2, 1257, 16, 4), 27, 32), ((69, 8, 2, 2912, 16, 4), 46, 56), ((10, 32, 32, 1257, 16, 4), 20, 25),
          ((20, 40, 40, 829, 16, 4), 18, 10)]


@pytest.mark.parametrize("sizes,equal,best", SHAPES)
def test_workspaces_between_the_two_plans(gpu, sizes, equal, best):
    (B, Hq, H, T, S, bits), D = sizes, 128
    L, tps, unit = _lib.lib(), 32 // bits, B * Hq * D * 4
    full = L.adkv_forward_ov_gqa_workspace_bytes(B, Hq, H, T, D, T // S + 1, S)
    assert full >= max(equal, best) * unit
    vp = [t.to(gpu) for t in synth.make_params(H, D, bits=bits, seed=4).astuple()]
    v = synth.make_v(B, H, T + 1, D, seed=1, dtype=torch.float16, device=gpu)
    caches = [synth.alloc_cache(B, H, T + tps, D, gpu, bits=bits) for _ in "kv"]
    cks = [torch.zeros(B, H, T // S + 1, D, 2, dtype=torch.float16, device=gpu) for _ in "kv"]
    states = [torch.zeros(B, H, D, 2, dtype=torch.float16, device=gpu) for _ in "kv"]
    gemv.append_kv_pair(*caches, v[:, :, :T], v[:, :, :T], vp, vp, 0, *states, k_ckpt=cks[0], v_ckpt=cks[1], ckpt_interval=S, bits=bits)
    vn, cache, ck = v[:, :, T].contiguous(), caches[1], cks[1]
    g = torch.Generator(device=gpu).manual_seed(5)
    w = torch.softmax(torch.randn(B, Hq, T + 1, generator=g, device=gpu), -1).half()

    def call(nbytes, ckpt=ck, at=0):
        out = torch.zeros(B, Hq, D, dtype=torch.float16, device=gpu)
        ws = torch.full((full + 4096 + at,), 0x5A, dtype=torch.uint8, device=gpu)[at:]
        rc = L.adkv_forward_ov_gqa(w.data_ptr(), cache.data_ptr(), vn.data_ptr(), out.data_ptr(), *[t.data_ptr() for t in vp], B, Hq, H, T, D,
                                   cache.shape[2], bits, 0, None, ckpt.data_ptr() if ckpt is not None else None, ck.shape[2], S, ws.data_ptr(),
                                   nbytes, _lib.current_stream_ptr(gpu))
        assert rc or torch.all(ws[nbytes:] == 0x5A)                          # nothing behind what it was given
        return rc, out.float()

    rc, want = call(0, ckpt=None)                                          # one segment
    assert rc == 0
    codes = cache.clone()
    for nbytes in (equal * unit, best * unit, full):
        rc, out = call(nbytes)
        if nbytes < equal * unit:
            assert rc == E_WORKSPACE and not torch.any(out)
            continue
        assert rc == 0 and torch.equal(cache, codes)
        # sums of the same products in fp32 in another order (|v| < 16, weights that sum to one), a rounding to fp16 each
        assert torch.all((out - want).abs() <= 2.0 ** -10 * want.abs() + 2.0 ** -17)
    assert call(equal * unit - 1)[0] == E_WORKSPACE and call(0)[0] == E_WORKSPACE
    assert call(full, at=8)[0] == E_ALIGN
