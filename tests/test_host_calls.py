"""The host calls (csrc/host_calls.cpp): what they take gives what the Python functions give, and what they do
not take goes to the Python functions."""
import types

import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from adkv_amd import _lib, synth
from adkv_amd.hf import cache as C
from adkv_amd.kernel import gemv
from adkv_amd.train.train_model import quant_f32

NOTHING = types.SimpleNamespace(**{n: (lambda *a: None) for n in ("rope_qk", "decode", "append", "quant_f32", "quant_f32_pair")})


class _Sub(torch.Tensor):
    pass


def test_other_arguments_are_left_to_python():
    h = _lib.host()
    x = torch.zeros(1, 1, 1, 128, dtype=torch.float16)
    assert h.rope_qk(x, x, x[0], x[0]) is None                                   # not on a device
    for args in ((), (x,), (1, 2, 3, 4), (x, x, None, None)):
        assert h.rope_qk(*args) is None
    for f, n in ((h.decode, 14), (h.append, 14), (h.quant_f32, 8), (h.quant_f32_pair, 11)):
        assert f() is None and f(*[None] * n) is None and f(*[x] * n) is None and f(*[1 << 70] * n) is None
    p = tuple(torch.zeros(128) for _ in range(5))
    assert h.quant_f32(torch.zeros(1, 2, 128), p, -8, 7, 0.1, 2.0, False, False) is None       # not on a device


def test_iterators_that_are_left_to_python_still_hold_their_tensors(monkeypatch):
    """CPU tensors are refused by the device check, which sees every tensor of the call."""
    from adkv_amd.train import train_model
    seen = []
    for m in (gemv, train_model):
        monkeypatch.setattr(m, "_need_device", lambda *t: (seen.append(len(t)), gemv._chk(False, "no device"))[0])
    p = synth.make_params(1, 128).astuple()
    k, caches = torch.zeros(1, 1, 8, 128).half(), [synth.alloc_cache(1, 1, 8, 128, "cpu") for _ in range(2)]
    with pytest.raises(RuntimeError, match="no device"):
        gemv.append_kv_pair(*caches, k, k, iter(p), iter(p), 0, *[torch.zeros(1, 1, 128, 2).half() for _ in range(2)])
    x, three, two = [torch.zeros(1, 8, 128)] * 2, [torch.ones(128)] * 3, [torch.zeros(1, 128)] * 2
    twice = lambda t: iter([iter(t), iter(t)])
    with pytest.raises(RuntimeError, match="no device"):
        train_model.quant_f32_pair(x, twice(three), -8, 7, 0.1, 2.0, states=twice(two), out=x, init=twice([t[0] for t in two]))
    assert seen == [16, 18]


class _Count(TorchDispatchMode):
    seen = 0

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        _Count.seen += 1
        return func(*args, **(kwargs or {}))


@pytest.mark.gpu
def test_watched_or_unusual_tensors_are_left_to_python(gpu):
    h = _lib.host()
    q = torch.randn(2, 4, 3, 128, device=gpu).half()
    cs = torch.randn(2, 3, 128, device=gpu).half()
    took = lambda *a: h.rope_qk(*a) is not None
    assert took(q, q, cs, cs)
    assert took(q.transpose(1, 2).contiguous().transpose(1, 2), q, cs, cs) and took(q, q, cs[:1], cs[:1])
    assert not took(q.as_subclass(_Sub), q, cs, cs) and not took(q, q.cpu(), cs, cs) and not took(q, q.bfloat16(), cs, cs)
    assert not took(torch.randn(2, 4, 3, 129, device=gpu).half()[..., :128], q, cs, cs)     # odd strides
    assert not took(q.float(), q.float(), cs.float(), cs.float()) and not took(q, q[:, :, :2], cs, cs)
    with _Count():
        assert not took(q, q, cs, cs)
        gemv.rope_qk(q, q, cs, cs)
    assert _Count.seen > 0                                                                     # the mode saw the Python function's work
    got = []
    torch.func.vmap(lambda a: (got.append(took(a, q, cs, cs)), a)[1])(q[None])
    assert got == [False]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D,Hq,H,bits,T,mask_dtype,mask_heads", [
    (128, 4, 4, 4, 300, None, 1), (128, 8, 2, 2, 700, torch.bfloat16, 1), (256, 2, 2, 4, 300, torch.float32, 2), (128, 4, 1, 4, 0, None, 1)])
def test_layer_calls_equal_the_python_functions(gpu, monkeypatch, dtype, D, Hq, H, bits, T, mask_dtype, mask_heads):
    B = 2
    params = [t.reshape(-1).to(gpu) for i in (1, 2) for t in synth.make_params(H, D, bits=bits, seed=i).astuple()]
    g = torch.Generator(device=gpu).manual_seed(T)
    heads = lambda n, t: torch.randn(B, t, n, D, generator=g, device=gpu).to(dtype).transpose(1, 2)
    k, v, cos, sin = heads(H, T), heads(H, T), *(torch.randn(B, 1, D, generator=g, device=gpu).to(dtype) for _ in range(2))
    new = [[heads(n, 1) for n in (Hq, H, H)] for _ in range(3)]
    masks = [None if mask_dtype is None else torch.randn(B, mask_heads, 1, T + i + 1, generator=g, device=gpu).to(mask_dtype) for i in range(3)]
    def run():
        layer, res = C.KVCacheLayer_ADKV(bits), []
        if T:
            layer.prefill(k, v, *params)
        for (q, kn, vn), m in zip(new, masks):
            q, kn = gemv.rope_qk(q, kn, cos, sin)
            out, w = layer.decode(q, kn, vn, *params, attention_mask=m, scaling=D ** -0.5)
            assert out.dtype == dtype and w.shape == (B, Hq, layer.get_seq_length())
            res += [q, kn, out, w.clone()]
        used = -(-layer.get_seq_length() // (32 // bits))
        return res + [t[:, :, :used] for t in (layer.key_states, layer.value_states)]
    run()                                                                          # the workspace is there from now on
    mine = run()
    monkeypatch.setattr(_lib, "host", lambda: NOTHING)
    for a, b in zip(mine, run()):
        assert a.dtype == b.dtype and torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("states", [False, True])
def test_fp32_quantiser_equals_the_python_function(gpu, monkeypatch, dtype, states):
    x = torch.randn(3, 77, 192, device=gpu).to(dtype)
    a, b, t, z, s = (torch.rand(192, device=gpu) * 0.1 + 0.05 for _ in range(5))
    f = lambda: quant_f32(x, a, b, t, -8, 7, 0.01, 50.0, zp_init=z, sc_init=s, output_states=states)
    mine = f()
    monkeypatch.setattr(_lib, "host", lambda: NOTHING)
    for p, q in zip(mine, f()):
        assert (p is None) == (q is None) and (p is None or torch.equal(p, q))


@pytest.mark.gpu
def test_fp32_calls_that_are_left_to_python(gpu):
    """quant_f32 with all of its arguments: taken as it should be, refused for one of them at a time."""
    h = _lib.host()
    x = torch.randn(2, 5, 128, device=gpu)
    p = tuple(torch.rand(128, device=gpu) * 0.1 + 0.05 for _ in range(5))
    took = lambda x=x, p=p, lower=-8, upper=7, lo=0.1, hi=2.0, states=False, free=False: (
        h.quant_f32(x, p, lower, upper, lo, hi, states, free) is not None)
    assert took() and took(states=True) and took(free=True) and took(x=x.half()) and took(x=x.bfloat16())
    assert not took(x=x.cpu()) and not took(x=x.double()) and not took(x=x[0]) and not took(x=x[:, ::2]) and not took(x=x[:0])
    assert not took(x=x.as_subclass(_Sub)) and not took(p=p[:4]) and not took(p=list(p)) and not took(p=(p[0].half(), *p[1:]))
    assert not took(p=(p[0][:64], *p[1:])) and not took(p=(p[0].cpu(), *p[1:])) and not took(lo=1) and not took(hi=None)
    assert not took(lower=1 << 70) and not took(upper=1 << 40) and not took(lower=-(1 << 40)) and not took(lower=0.5)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_evaluation_cache_equals_the_python_function(gpu, monkeypatch, dtype):
    from adkv_amd.hf import llama_adkv_eval as E
    x = [torch.randn(2, n, 256, device=gpu).to(dtype) for n in (77, 1, 30)]
    p = [torch.rand(256, device=gpu) * 0.1 + 0.05 for _ in range(10)]
    def run():
        layer = E.KVCacheLayer_ADKV()
        for t in x:
            keys, values = layer.update(t, -t, *p)
        return [t.clone() for t in (keys, values, layer.key_dc, layer.value_dc, layer.key_scale, layer.value_scale)]
    mine = run()
    monkeypatch.setattr(_lib, "host", lambda: NOTHING)
    for a, b in zip(mine, run()):
        assert torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("fresh", [True, 1, torch.ones(1, dtype=torch.bool)])
def test_any_truth_value_makes_a_cache_fresh(gpu, fresh):
    """Slots and checkpoints behind the prompt are zeroed, whatever says that the memory is uninitialised."""
    B, H, D, T, S = 1, 2, 128, 70, 64
    p = [t.to(gpu) for t in synth.make_params(H, D, seed=1).astuple()]
    x = torch.randn(B, H, T, D, device=gpu).half()
    junk = lambda *shape: torch.full(shape, 0x5A, dtype=torch.uint8, device=gpu)
    caches = [junk(B, H, 16, D // 4, 4, 4) for _ in range(2)]
    state, ckpt = ([junk(B, H, *n, D, 4).view(torch.float16) for _ in range(2)] for n in ((), (3,)))
    gemv.append_kv_pair(*caches, x, x, p, p, 0, *state, k_ckpt=ckpt[0], v_ckpt=ckpt[1], ckpt_interval=S, fresh=fresh)
    for c, k in zip(caches, ckpt):
        assert not torch.any(c[:, :, 9:]) and not torch.any(k[:, :, 1:].view(torch.int16)) and torch.any(k[:, :, 0] != 0)


@pytest.mark.gpu
def test_written_tensors_that_share_their_storage_lazily_become_their_own(gpu):
    from adkv_amd.train.train_model import quant_f32_pair
    B, T, C = 2, 9, 64
    x = [torch.randn(B, T, C, device=gpu) for _ in range(2)]
    p = [tuple(torch.rand(C, device=gpu) * 0.1 + 0.05 for _ in range(3)) for _ in range(2)]
    shared = [torch.ones(n, device=gpu).view(*s) for n, s in [(B * T * C, (B, T, C))] * 2 + [(B * C, (B, C))] * 4]
    mine = [torch._lazy_clone(t) for t in shared]
    plain = [t.clone() for t in shared]
    for out in (mine, plain):
        quant_f32_pair(x, p, -8, 7, 0.1, 2.0, states=[tuple(out[2:4]), tuple(out[4:])], out=out[:2])
    for t, a, b in zip(shared, mine, plain):
        assert torch.all(t == 1.0) and torch.equal(a, b)


@pytest.mark.gpu
def test_a_profiler_sees_the_tensors_that_a_call_makes(gpu):
    h = _lib.host()
    q, cs = torch.randn(2, 4, 3, 128, device=gpu).half(), torch.randn(2, 3, 128, device=gpu).half()
    x, p = torch.randn(1, 8, 128, device=gpu), tuple(torch.full((128,), 0.5, device=gpu) for _ in range(5))
    for call in (lambda: h.rope_qk(q, q, cs, cs), lambda: h.quant_f32(x, p, -8, 7, 0.1, 2.0, False, False)):
        want = call()
        assert want is not None
        with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as seen:
            got = call()
        assert [e.count for e in seen.key_averages() if e.key == "aten::empty"] == [2]
        for a, b in zip(want, got):
            assert not isinstance(a, torch.Tensor) or torch.equal(a, b)
