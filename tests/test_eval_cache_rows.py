"""Evaluation cache: rows that are more than their bytes are copied into the buffers by torch, so that
whatever rides on that copy (a tangent, a graph, a pending negation, a recording of it) is kept.

The quantiser is replaced by one that moves bytes between storages, as a kernel does, and leaves the
values as they are.
"""
import warnings

import pytest
import torch
from torch.autograd import forward_ad

from adkv_amd.hf import llama_adkv_eval as M

B, T, C = 2, 5, 64


@pytest.fixture(autouse=True)
def byte_copying_quantiser(monkeypatch):
    def raw(t):   # the memory of t, with nothing of what torch knows about it
        return torch.empty(0, dtype=t.dtype).set_(t.untyped_storage(), t.storage_offset(), t.shape, t.stride())

    def quant(x, params, *limits, states, out, init=None):
        with torch.no_grad():
            for src, dst in zip(x, out):
                if src.data_ptr() != dst.data_ptr():
                    raw(dst).numpy()[...] = raw(src).numpy()

    monkeypatch.setattr(M, "quant_f32_pair", quant)


def update(k, v, layer=None):
    layer = layer or M.KVCacheLayer_ADKV()
    return layer.update(k, v, *(torch.ones(C) for _ in range(10)))


def rows(seed, tokens=T):
    return torch.randn(B, tokens, C, generator=torch.Generator().manual_seed(seed))


@pytest.mark.parametrize("which", (0, 1))
def test_forward_mode_tangent(which):
    x, t = [rows(1), rows(2)], rows(3)
    with forward_ad.dual_level():
        y = list(x)
        y[which] = forward_ad.make_dual(x[which], t)
        out = update(*y)
        got = forward_ad.unpack_dual(out[which])
        assert got.tangent is not None and torch.equal(got.tangent, t)
        assert torch.equal(got.primal, x[which])
        assert forward_ad.unpack_dual(out[1 - which]).tangent is None


def test_lazily_negated_rows():
    k, v = rows(1), rows(2)
    keys, values = update(torch._neg_view(k), torch._neg_view(v))
    assert torch.equal(keys, -k) and torch.equal(values, -v)


def test_rows_after_rows_with_a_graph():
    """The buffer then belongs to a graph: a later write that the graph does not see is an error there."""
    k = rows(1).requires_grad_()
    layer = M.KVCacheLayer_ADKV()
    keys, _ = update(k, rows(2), layer)
    loss = (keys * keys).sum()
    update(rows(3, 1), rows(4, 1), layer)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        loss.backward()


def test_copy_is_recorded_by_a_trace():
    with warnings.catch_warnings():
        warnings.simplefilter("ignore", torch.jit.TracerWarning)
        traced = torch.jit.trace(lambda k, v: update(k, v), (rows(1), rows(2)), check_trace=False)
    keys, values = traced(rows(3), rows(4))
    assert torch.equal(keys, rows(3)) and torch.equal(values, rows(4))


def test_copy_is_recorded_by_a_dispatch_mode():
    from torch.utils._python_dispatch import TorchDispatchMode

    class Copies(TorchDispatchMode):
        n = 0

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.n += func is torch.ops.aten.copy_.default
            return func(*args, **(kwargs or {}))

    k, v = rows(1), rows(2)
    with Copies() as mode:
        update(k, v)
    assert mode.n >= 2


def test_transformed_rows_are_refused_as_by_a_copy():
    k, v = rows(1), rows(2)
    with pytest.raises(RuntimeError, match="inplace arithmetic"):
        torch.vmap(lambda k: update(k, v)[0])(torch.stack([k, v]))


def test_plain_rows_are_read_in_place():
    k, v = rows(1), rows(2)
    layer = M.KVCacheLayer_ADKV()
    layer._append_tokens = None   # the copying route is not taken
    keys, values = update(k, v, layer)
    assert torch.equal(keys, k) and torch.equal(values, v)
