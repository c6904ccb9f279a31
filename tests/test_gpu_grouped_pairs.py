"""Grouped queries and 2-bit codes with two channels per lane (a KV head per wave), and where the launch
goes over to four: every shape of workgroup, the context ending inside and at the end of a segment."""
import numpy as np
import pytest
import torch

from adkv_amd import _lib, synth
from adkv_amd.kernel import gemv
from test_gpu_parity import SMAX, SMIN, _inputs, _np16, _ulp16

pytestmark = pytest.mark.gpu

B, H, D = 4, 4, 128


# 16 equal (sequence, KV head) pairs, a checkpoint every 8 or 16 tokens: 16 waves of two channels per segment
@pytest.mark.parametrize("bits,G,T,pair", [
    (4, 4, 81, True), (4, 8, 161, True), (2, 4, 527, True), (2, 8, 337, True),   # at most 8 waves per CU: four-wave workgroups
    (4, 2, 1160, True), (2, 1, 2559, True),                                      # 12-wave workgroups
    (4, 4, 2047, True), (4, 8, 1601, True), (2, 2, 4096, True),                  # 16-wave workgroups
    (4, 4, 2049, False), (2, 2, 4097, False),                                    # one segment more than fits two waves per SIMD
])
def test_two_channels_per_lane(gpu, oracle, bits, G, T, pair):
    S = 32 // bits
    name = _lib.lib().adkv_decode_kernel_name(B, H * G, H, T, D, bits, T // S + 1, S)
    assert (b"two channels" in name) == pair, name
    x, p = _inputs(1, 1, T + 1, D, seed=T % 5, bits=bits)
    pn = [_np16(t) for t in p.astuple()]
    g = torch.Generator().manual_seed(T)
    q = torch.randn(1, G, 1, D, generator=g).half()
    attn = torch.softmax(2.0 * torch.randn(1, G, T + 1, generator=g), dim=-1).half()
    with oracle.code_bits(bits):
        cache = oracle.alloc_cache(1, 1, T + S, D)
        oracle.encode_kv_f16(cache, _np16(x)[:, :, :T], *pn)
        lw, ow = np.zeros((G, T + 1)), np.zeros((G, D))
        for j in range(G):
            want = cache.copy()
            lw[j] = oracle.forward_qk_f16(_np16(q)[:, j:j + 1], want, _np16(x)[:, :, T:], *pn, T)[0][0, 0]
            ow[j] = oracle.forward_ov_f16(_np16(attn)[:, j:j + 1], cache.copy(), _np16(x)[:, :, T:], *pn)[0][0, 0]
    every = lambda t, n=H: t.to(gpu).expand(B, n, *t.shape[2:]).contiguous()      # of every (sequence, head) pair
    par = [t.to(gpu).expand(H, D).contiguous() for t in p.astuple()]
    kc, vc = (synth.alloc_cache(B, H, T + S, D, gpu, bits=bits) for _ in range(2))
    kck, vck = (torch.zeros(B, H, T // S + 1, D, 2, dtype=torch.float16, device=gpu) for _ in range(2))
    st = [torch.zeros(B, H, D, 2, dtype=torch.float16, device=gpu) for _ in range(2)]
    rows, xn = every(x[:, :, :T]), every(x[:, :, T:])
    gemv.append_kv_pair(kc, vc, rows, rows, par, par, 0, *st, k_ckpt=kck, v_ckpt=vck, ckpt_interval=S, bits=bits)
    logits = gemv.forward_qk(q.to(gpu).repeat(B, H, 1, 1), kc, xn, *par, T, SMIN, SMAX, ckpt=kck, ckpt_interval=S, bits=bits)
    out = gemv.forward_ov(attn.to(gpu).repeat(B, H, 1), vc, xn, *par, SMIN, SMAX, ckpt=vck, ckpt_interval=S, bits=bits)
    torch.cuda.synchronize()
    for c in (kc, vc):
        assert torch.equal(c.cpu(), torch.from_numpy(want).expand(B, H, *want.shape[2:]))
    assert torch.equal(kck.view(torch.int16), vck.view(torch.int16))
    lg, og = logits.view(B * H, G, T + 1).cpu(), out.view(B * H, G, D).cpu()
    assert torch.equal(lg, lg[:1].expand_as(lg)) and torch.equal(og, og[:1].expand_as(og))
    lg, og = _np16(lg[0]).astype(np.float64), _np16(og[0]).astype(np.float64)
    assert np.all(np.abs(lg - lw) <= _ulp16(lw) + 1e-3)
    assert np.all(np.abs(og - ow) <= _ulp16(ow) + 1e-3)


@pytest.mark.parametrize("bits", [4, 2])
@pytest.mark.parametrize("G", [2, 4, 8])
@pytest.mark.parametrize("segments", [127, 128, 129, 192, 193])          # two and three waves per SIMD, and either side
def test_values_from_rows_of_any_alignment(gpu, bits, G, segments):
    """Two or four channels per lane, which the rows' alignment decides as well: the same sums, bit for bit."""
    S = 32 // bits
    T = S * segments - 3
    x, p = _inputs(B, H, T + 1, D, seed=segments, bits=bits)
    p = [t.to(gpu) for t in p.astuple()]
    cache = synth.alloc_cache(B, H, T + S, D, gpu, bits=bits)
    ckpt = torch.zeros(B, H, T // S + 1, D, 2, dtype=torch.float16, device=gpu)
    state = torch.zeros(B, H, D, 2, dtype=torch.float16, device=gpu)
    gemv.append_kv(cache, x[:, :, :T].contiguous().to(gpu), *p, 0, state, ckpt=ckpt, ckpt_interval=S, bits=bits)
    rows = torch.rand(B, H * G, (T + 8) // 8 * 8, generator=torch.Generator().manual_seed(G)).half().to(gpu)[:, :, :T + 1]
    got = [gemv.forward_ov(w, cache.clone(), x[:, :, T:].contiguous().to(gpu), *p, SMIN, SMAX, ckpt=ckpt.clone(), ckpt_interval=S, bits=bits)
           for w in (rows, rows.contiguous())]
    assert torch.equal(*got) and torch.all(torch.isfinite(got[0]))
