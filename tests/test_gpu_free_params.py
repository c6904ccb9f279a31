"""The training forward constrains its parameters inside the launch: the bits of torch's sigmoid and exp, extreme
parameters included, and a model that constrains them in its own way keeps it."""
import pytest
import torch

from adkv_amd import _lib
from adkv_amd.train import ADKVTrainModel, quant_f32
from tests.test_host_calls import NOTHING


def _model(C, cls=ADKVTrainModel):
    m = cls(C)
    g = torch.Generator().manual_seed(C)
    with torch.no_grad():
        for p in (m.alpha, m.beta, m.init_log_sc, m.init_zp):
            p.copy_(torch.randn(C, generator=g))
        for p in (m.alpha, m.beta, m.init_log_sc):
            p[:10] = torch.tensor([0.0, -0.0, 90.0, -90.0, 104.0, -104.0, 1e-38, float("inf"), -float("inf"), float("nan")])
    return m.cuda()


def _want(m, x, states):
    return quant_f32(x, m.get_alpha(), m.get_beta(), m.target, m.lower_limit, m.upper_limit, m.sc_min, m.sc_max,
                     zp_init=m.init_zp, sc_init=m.get_sc(), output_states=states)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", (torch.float32, torch.bfloat16))
@pytest.mark.parametrize("B,T", [(1, 1), (2, 77), (600, 9)])          # 600: a lane per channel straight from memory
@pytest.mark.parametrize("in_python", (False, True))
def test_same_bits_as_torch(gpu, monkeypatch, dtype, B, T, in_python):
    m = _model(192)
    x = (2.0 * torch.randn(B, T, 192, generator=torch.Generator().manual_seed(T))).to(dtype).to(gpu)
    out, _, zs, ss = _want(m, x, True)
    if in_python:
        monkeypatch.setattr(_lib, "host", lambda: NOTHING)
    for got, want in zip(m(x, output_states=True), (out, zs, ss)):
        assert torch.equal(torch.nan_to_num(got.float(), nan=123.0), torch.nan_to_num(want.float(), nan=123.0))
    assert torch.equal(torch.nan_to_num(m(x).float()), torch.nan_to_num(out.float()))


@pytest.mark.gpu
def test_own_constraints_stay(gpu):
    class Own(ADKVTrainModel):
        def get_beta(self):
            return 0.01 * torch.sigmoid(self.beta)

    x = torch.randn(2, 40, 64, device=gpu)
    for m in (_model(64, Own), _model(64).half(), _model(64).double()):
        assert torch.equal(torch.nan_to_num(m(x)), torch.nan_to_num(_want(m, x, False)[0]))
    m = _model(64)
    m.get_alpha = lambda: torch.full((64,), 0.5, device=gpu)
    assert torch.equal(torch.nan_to_num(m(x)), torch.nan_to_num(_want(m, x, False)[0]))


@pytest.mark.parametrize("name", ("get_alpha", "get_beta", "get_sc"))
def test_constraints_set_on_the_class_stay(monkeypatch, name):
    """What the forward gives the quantiser, without a device."""
    from adkv_amd.train import train_model
    given = {}
    monkeypatch.setattr(train_model, "quant_f32", lambda x, *a, **kw: given.update(kw, a=a) or (x, None, None, None))
    m, x = ADKVTrainModel(64), torch.zeros(1, 2, 64)
    m(x)
    assert given["free_params"] and given["a"][0] is m.alpha and given["sc_init"] is m.init_log_sc
    own = torch.full((64,), 0.5)
    monkeypatch.setattr(ADKVTrainModel, name, lambda self: own)
    m(x)
    assert not given["free_params"]
    assert {"get_alpha": given["a"][0], "get_beta": given["a"][1], "get_sc": given["sc_init"]}[name] is own
