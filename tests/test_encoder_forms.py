"""Both forms of the encoder (a lane with one channel, and with two where a launch has more than 64 channels
per SIMD) on inputs that leave their main loop: quotients that are not numbers, and rounding ties."""
import time

import numpy as np
import pytest
import torch

from adkv_amd import synth
from adkv_amd.kernel import gemv

pytestmark = pytest.mark.gpu

D = 128
FORMS = {"one_channel": (1, 3), "two_channels": (17, 32)}   # batch, heads: 384 and 69 632 channels


def _np16(t):
    return t.detach().cpu().contiguous().view(torch.int16).numpy().view(np.float16)


def _same16(a, b):
    """Equal bits, any NaN equal to any other."""
    a, b = (x.view(np.uint16) for x in (a, b))
    nan = lambda x: (x & 0x7FFF) > 0x7C00
    return np.array_equal(np.where(nan(a), 0x7E00, a), np.where(nan(b), 0x7E00, b))


def _check(gpu, oracle, form, bits, x, params, S, cuts=()):
    """Codes, carried state and checkpoints of a stream appended in the pieces of ``cuts`` against the oracle."""
    B, H, T, _ = x.shape
    pn, pg = [_np16(t) for t in params], [t.to(gpu) for t in params]
    xn, xg = _np16(x), x.to(gpu)
    cache = synth.alloc_cache(B, H, T + 16, D, gpu, bits=bits)
    state = torch.zeros(B, H, D, 2, dtype=torch.float16, device=gpu)
    ck = torch.zeros(B, H, T // S + 1, D, 2, dtype=torch.float16, device=gpu) if S else None
    edges = [0, *cuts, T]
    for a, b in zip(edges, edges[1:]):
        gemv.append_kv(cache, xg[:, :, a:b].contiguous(), *pg, a, state, ckpt=ck, ckpt_interval=S, bits=bits)
    torch.cuda.synchronize()
    with oracle.code_bits(bits):
        want = oracle.alloc_cache(B, H, T + 16, D)
        st = oracle.encode_kv_f16(want, xn, *pn)
        assert np.array_equal(cache.cpu().numpy(), want)
        assert _same16(_np16(state), st)
        n = T // S if S else 0
        for j in sorted({0, n // 2, n - 1}) if n else ():
            c = oracle.alloc_cache(B, H, (j + 1) * S, D)
            sj = oracle.encode_kv_f16(c, xn[:, :, :(j + 1) * S], *pn)
            assert _same16(_np16(ck[:, :, j]), sj), j


@pytest.mark.parametrize("form,bits,T,S,cuts", [
    ("one_channel", 4, 8, 0, ()), ("one_channel", 4, 64, 64, ()), ("one_channel", 4, 71, 64, ()), ("one_channel", 4, 200, 8, ()),
    ("one_channel", 4, 2500, 64, (5, 150)), ("one_channel", 2, 32, 0, ()), ("one_channel", 2, 100, 16, ()),
    ("one_channel", 2, 2500, 64, (33,)), ("two_channels", 4, 32, 0, ()), ("two_channels", 4, 71, 8, ()),
    ("two_channels", 4, 133, 64, (5,)), ("two_channels", 2, 32, 16, ()), ("two_channels", 2, 133, 64, (33,))])
def test_quotients_that_are_not_numbers(gpu, oracle, form, bits, T, S, cuts):
    """Channels whose every quotient is a NaN (a scale of zero, a state that became infinite), single
    non-finite inputs at the first and last token of a run and of the stream, and stretches of them: the run
    is done again, more of it when the next one fails as well, and the fast form taken up again behind."""
    B, H = FORMS[form]
    g = torch.Generator().manual_seed(T + bits)
    params = [t.clone() for t in synth.make_params(H, D, bits=bits, seed=2).astuple()]
    params[1][0, 5] = 0.0                                            # zero scale: stays zero
    params[4][H - 1, 70], params[3][H - 1, 70] = -60.0, 2.0           # the scale runs away to infinity
    x = (2.0 * torch.randn(B, H, T, D, generator=g)).half()
    bad = [float("inf"), float("nan"), -float("inf")]
    for i, t in enumerate((0, 7, 8, 31, 32, 63, 64, 127, 128, T - 1)):
        if t < T:
            x[i % B, i % H, t, (11 * i) % D] = bad[i % 3]
    x[B - 1, 1, T // 4: 3 * T // 4, 100] = float("nan")               # a stretch, then numbers again
    _check(gpu, oracle, form, bits, x, params, S, cuts)


@pytest.mark.parametrize("bits", (4, 2))
def test_rows_that_a_buffer_descriptor_cannot_span(gpu, oracle, bits):
    """Rows 8 MiB apart: the stream is taken in pieces of 128 tokens, and a run that meets a NaN is done
    again inside its piece."""
    T, pitch = 300, 1 << 22
    params = [t.clone() for t in synth.make_params(1, D, bits=bits, seed=2).astuple()]
    params[1][0, 5] = 0.0
    x = torch.randn(1, 1, T, D, generator=torch.Generator().manual_seed(0)).half()
    x[0, 0, 130, 9] = float("nan")
    big = torch.empty(T, pitch, dtype=torch.float16, device=gpu)
    big[:, :D] = x[0, 0].to(gpu)
    rows = big.as_strided((1, 1, T, D), (T * pitch, T * pitch, pitch, 1))
    pg = tuple(t.to(gpu) for t in params)
    caches = [synth.alloc_cache(1, 1, T + 16, D, gpu, bits=bits) for _ in range(2)]
    states = [torch.zeros(1, 1, D, 2, dtype=torch.float16, device=gpu) for _ in range(2)]
    gemv.append_kv_pair(*caches, rows, rows, pg, pg, 0, *states, bits=bits)
    torch.cuda.synchronize()
    with oracle.code_bits(bits):
        want = oracle.alloc_cache(1, 1, T + 16, D)
        st = oracle.encode_kv_f16(want, _np16(x), *[_np16(t) for t in params])
    for c, s in zip(caches, states):
        assert np.array_equal(c.cpu().numpy(), want) and _same16(_np16(s), st)


@pytest.mark.parametrize("bits", (4, 2))
@pytest.mark.parametrize("mib", (10, 11, 12, 13))
def test_checkpoints_of_pieces_that_start_inside_a_run(gpu, oracle, bits, mib):
    """Rows 10 to 13 MiB apart: a piece of 2-bit codes is 96, 80 or 64 tokens, and checkpoints every 64 lie inside
    the runs that such a piece counts from its own start."""
    T, S, pitch = 300, 64, mib << 19
    params = synth.make_params(1, D, bits=bits, seed=2).astuple()
    x = torch.randn(1, 1, T, D, generator=torch.Generator().manual_seed(mib)).half()
    big = torch.empty(T, pitch, dtype=torch.float16, device=gpu)
    big[:, :D] = x[0, 0].to(gpu)
    rows = big.as_strided((1, 1, T, D), (T * pitch, T * pitch, pitch, 1))
    pg = tuple(t.to(gpu) for t in params)
    caches = [synth.alloc_cache(1, 1, T + 16, D, gpu, bits=bits) for _ in range(2)]
    states = [torch.zeros(1, 1, D, 2, dtype=torch.float16, device=gpu) for _ in range(2)]
    cks = [torch.zeros(1, 1, T // S + 1, D, 2, dtype=torch.float16, device=gpu) for _ in range(2)]
    gemv.append_kv_pair(*caches, rows, rows, pg, pg, 0, *states, k_ckpt=cks[0], v_ckpt=cks[1], ckpt_interval=S, bits=bits)
    torch.cuda.synchronize()
    pn, xn = [_np16(t) for t in params], _np16(x)
    with oracle.code_bits(bits):
        want = oracle.alloc_cache(1, 1, T + 16, D)
        st = oracle.encode_kv_f16(want, xn, *pn)
        at = [oracle.encode_kv_f16(oracle.alloc_cache(1, 1, (j + 1) * S, D), xn[:, :, :(j + 1) * S], *pn) for j in range(T // S)]
    for c, s, k in zip(caches, states, cks):
        assert np.array_equal(c.cpu().numpy(), want) and _same16(_np16(s), st)
        for j, a in enumerate(at):
            assert _same16(_np16(k[:, :, j]), a), j
        assert not torch.any(k[:, :, T // S:])


@pytest.mark.parametrize("form,T", [("one_channel", 8192), ("two_channels", 2048)])
def test_one_bad_channel_does_not_stall_the_launch(gpu, form, T):
    """A channel with a zero scale sends its wave through the plain division for the whole stream, and the
    launch waits for that wave: some 2.4 times as long as without it (83 ns per token against 34, one channel per
    lane).  When every token waits for a load of its own it is 3.8 times."""
    B, H = FORMS[form]
    params = [t.to(gpu) for t in synth.make_params(H, D, seed=2).astuple()]
    x = synth.make_k(B, H, T, D, dtype=torch.float16, device=gpu)
    cache = synth.alloc_cache(B, H, T, D, gpu)
    state = torch.zeros(B, H, D, 2, dtype=torch.float16, device=gpu)

    def best():
        times = []
        for _ in range(5):
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            gemv.append_kv(cache, x, *params, 0, state)
            torch.cuda.synchronize()
            times.append(time.perf_counter() - t0)
        return min(times[1:])

    clean = best()
    params[1][0, 5] = 0.0
    bad = best()
    print(f"{form}: {clean * 1e6:.0f} us, with a bad channel {bad * 1e6:.0f} us")
    assert bad < 3 * clean


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("bits", (4, 2))
def test_rounding_ties(gpu, oracle, form, bits):
    """(x - zp) / sc = k + 1/2 exactly (ties go to even) and one fp16 step to either side, with scales that are
    powers of two and not, in whole runs and in the tokens behind them."""
    B, H = FORMS[form]
    T = 75
    g = torch.Generator().manual_seed(11 + bits)
    sc = torch.tensor([0.25, 0.5, 1.0, 2.0, 0.75, 1.5, 3.0, 0.3330078125])[torch.randint(0, 8, (H, D), generator=g)].half()
    k = torch.randint(-11, 11, (B, H, T, D), generator=g).float()
    x = ((k + 0.5) * sc.float()[None, :, None, :]).half()
    x = (x.view(torch.int16) + torch.randint(-1, 2, x.shape, generator=g).to(torch.int16)).view(torch.float16)
    zero = torch.zeros(H, D).half()
    _check(gpu, oracle, form, bits, x, [zero, sc, zero, zero, torch.full((H, D), 3.5 if bits == 4 else 0.5).half()], 0)


@pytest.mark.parametrize("form,H", [("one_channel", 3), ("two_channels", 32)])
@pytest.mark.parametrize("bits,cuts", [(4, (0, 75)), (4, (0, 37, 150)), (2, (0, 107)), (2, (0, 21, 150))])
def test_bfloat16_pair(gpu, oracle, form, H, bits, cuts):
    """K and V in one launch from bfloat16 projection outputs, in whole runs and resumed inside a word."""
    B, T = (1 if form == "one_channel" else 9), cuts[-1]          # 36 864 channels per tensor, 73 728 in the launch
    rows, params, want = [], [], []
    for i in range(2):
        ps = [t.clone() for t in synth.make_params(H, D, bits=bits, seed=4 + i).astuple()]
        ps[1][H - 1, 3] = 0.0
        x = (2.0 * torch.randn(B, T, H, D, generator=torch.Generator().manual_seed(i))).to(torch.bfloat16)
        x[0, T // 2, 0, 9] = float("nan")
        rows.append(x.to(gpu).transpose(1, 2))
        params.append(tuple(t.to(gpu) for t in ps))
        with oracle.code_bits(bits):
            c = oracle.alloc_cache(B, H, T + 16, D)
            st = oracle.encode_kv_f16(c, _np16(x.transpose(1, 2).to(torch.float16)), *[_np16(t) for t in ps])
        want.append((c, st))
    caches = [synth.alloc_cache(B, H, T + 16, D, gpu, bits=bits) for _ in range(2)]
    states = [torch.zeros(B, H, D, 2, dtype=torch.float16, device=gpu) for _ in range(2)]
    for a, b in zip(cuts, cuts[1:]):
        gemv.append_kv_pair(*caches, *(r[:, :, a:b] for r in rows), *params, a, *states, bits=bits)
    torch.cuda.synchronize()
    for c, s, (wc, ws) in zip(caches, states, want):
        assert np.array_equal(c.cpu().numpy(), wc) and _same16(_np16(s), ws)
