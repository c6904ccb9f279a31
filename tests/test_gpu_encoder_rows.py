"""Rows that reach the encoder through the LDS (one channel per lane, whole runs of 64 tokens, 16-byte aligned
rows), where the runs, the pieces and the alignment end.  Codes, states and checkpoints are those of the
oracle bit for bit."""
import numpy as np
import pytest
import torch

from adkv_amd import synth
from adkv_amd.kernel import gemv
from tests.test_encoder_forms import _np16, _same16

pytestmark = pytest.mark.gpu

D = 128


@pytest.mark.parametrize("bits", (4, 2))
@pytest.mark.parametrize("dtype", (torch.float16, torch.bfloat16))
@pytest.mark.parametrize("cuts,S,pad,bad", [
    ((0, 63), 0, 0, ()), ((0, 64), 64, 0, ()), ((0, 65), 0, 64, ()), ((0, 127), 64, 8, ()), ((0, 128), 128, 0, (127,)),
    ((0, 129, 200), 64, 0, ()),             # resumed inside a word, checkpoints between runs that do not start at one
    ((0, 128, 321), 64, 24, (191, 192)),    # resumed at a run, a run that fails at its last and first token
    ((0, 200), 48, 0, ()),                  # checkpoints inside runs
    ((0, 200), 64, 4, ()), ((0, 200), 64, 1, (64,)),   # rows 8 and 2 bytes off: not through the LDS
    ((0, 120), 0, 0, (70,)), ((0, 190), 64, 0, (150, 188)), ((0, 66, 250), 64, 8, ()),   # words behind the last run, and a NaN there
    ((0, 7, 64, 576), 256, 16, (575,))])
def test_runs_through_the_lds(gpu, oracle, bits, dtype, cuts, S, pad, bad):
    B, H, T = 2, 3, cuts[-1]
    params, rows, want = [], [], []
    for i in range(2):
        ps = [t.clone() for t in synth.make_params(H, D, bits=bits, seed=7 + i).astuple()]
        x = (2.0 * torch.randn(B, T, H * D + pad, generator=torch.Generator().manual_seed(T + i))).to(dtype)
        x[..., H * D:] = float("nan")                                # never read
        for t in bad:
            x[1, t, 17 + 64 * i] = float("inf")
        xh = x[..., :H * D].view(B, T, H, D).transpose(1, 2)
        rows.append(x.to(gpu)[..., :H * D].view(B, T, H, D).transpose(1, 2))
        params.append([t.to(gpu) for t in ps])
        pn, xn = [_np16(t) for t in ps], _np16(xh.to(torch.float16))
        with oracle.code_bits(bits):
            c = oracle.alloc_cache(B, H, T + 16, D)
            st = oracle.encode_kv_f16(c, xn, *pn)
            cks = []
            for j in range(T // S if S else 0):
                part = oracle.alloc_cache(B, H, (j + 1) * S, D)
                cks.append(oracle.encode_kv_f16(part, xn[:, :, :(j + 1) * S], *pn))
        want.append((c, st, cks))
    caches = [synth.alloc_cache(B, H, T + 16, D, gpu, bits=bits) for _ in range(2)]
    states = [torch.zeros(B, H, D, 2, dtype=torch.float16, device=gpu) for _ in range(2)]
    cks = [torch.zeros(B, H, T // S + 1, D, 2, dtype=torch.float16, device=gpu) if S else None for _ in range(2)]
    for a, b in zip(cuts, cuts[1:]):
        gemv.append_kv_pair(*caches, *(r[:, :, a:b] for r in rows), *params, a, *states, k_ckpt=cks[0], v_ckpt=cks[1],
                            ckpt_interval=S, bits=bits)
    torch.cuda.synchronize()
    for c, s, k, (wc, ws, wk) in zip(caches, states, cks, want):
        assert np.array_equal(c.cpu().numpy(), wc) and _same16(_np16(s), ws)
        for j, w in enumerate(wk):
            assert _same16(_np16(k[:, :, j]), w), j


@pytest.mark.parametrize("bits", (4, 2))
@pytest.mark.parametrize("B,T,S", [(17, 384, 64), (24, 449, 0), (21, 400, 48), (25, 385, 64), (17, 383, 64)])
def test_two_rounds_of_one_channel_per_lane(gpu, bits, B, T, S):
    """32 heads: 17 to 24 sequences are more than two and at most three waves per SIMD.  Sequences 0 and B - 1 are
    what they are alone, where their few channels take one channel per lane with a wave to a SIMD."""
    H = 32
    params = [[t.to(gpu) for t in synth.make_params(H, D, bits=bits, seed=7 + i).astuple()] for i in range(2)]
    rows = [torch.randn(B, T, H * D, generator=torch.Generator().manual_seed(i)).to(torch.bfloat16) for i in range(2)]
    rows[1][B - 1, T - 2, 77] = float("nan")
    rows = [r.to(gpu).view(B, T, H, D).transpose(1, 2) for r in rows]

    def run(rs):
        n = rs[0].shape[0]
        caches = [synth.alloc_cache(n, H, T + 16, D, gpu, bits=bits) for _ in range(2)]
        states = [torch.zeros(n, H, D, 2, dtype=torch.float16, device=gpu) for _ in range(2)]
        cks = [torch.zeros(n, H, T // S + 1, D, 2, dtype=torch.float16, device=gpu) if S else None for _ in range(2)]
        gemv.append_kv_pair(*caches, *rs, *params, 0, *states, k_ckpt=cks[0], v_ckpt=cks[1], ckpt_interval=S, bits=bits)
        return caches, states, cks

    got, torch_nan = run(rows), lambda t: torch.nan_to_num(t.float(), nan=123.0)
    for b in (0, B - 1):
        want = run([r[b:b + 1] for r in rows])
        for g, w in zip(got[0], want[0]):
            assert torch.equal(g[b:b + 1], w)
        for g, w in [*zip(got[1], want[1]), *(zip(got[2], want[2]) if S else ())]:
            assert torch.equal(torch_nan(g[b:b + 1]), torch_nan(w))
