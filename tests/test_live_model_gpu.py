"""A predictor follows its model: whatever is exchanged between two calls, the next one computes what a predictor
made of the model as it then is computes."""

import copy
import math

import pytest
import torch
from torch import nn

pytestmark = pytest.mark.gpu


def _model(seed):
    from ar_nanotabpfn_amd.model import ARTabPFN

    torch.manual_seed(seed)
    m = ARTabPFN(d_model=128, n_heads=4, n_layers=2, d_ff=256, num_features=2, buffer_size=6, num_components=4)
    with torch.no_grad():
        m.head.std_bias.fill_(math.log(math.expm1(0.5)))
    return m.eval()


def _assign(m, other):
    m.load_state_dict({k: v.clone() for k, v in other.state_dict().items()}, assign=True)


def _assign_twice(m, other):  # (the memory of the first weights can come back as the last ones')
    _assign(m, copy.deepcopy(other))
    torch.cuda.synchronize()
    _assign(m, other)


def _one_weight(m, other):
    m.backbone.layers[1].ff[0].weight = nn.Parameter(other.backbone.layers[1].ff[0].weight.detach().clone())


def _data(m, other):
    for p, q in zip(m.parameters(), other.parameters()):
        p.data = q.detach().clone()


def _head(m, other):
    m.head.head = copy.deepcopy(other.head.head)


def _constants(m, other):
    m.backbone.layers[0].norm1.eps = m.backbone.layers[1].norm1.eps = 0.3
    m.backbone.norm.eps = 0.2
    m.head.std_min = 0.7


# float32 and K = 4: both layouts take the run in one launch; the recorded steps with whole_run_decode off
@pytest.mark.parametrize("whole_run", [True, False], ids=["run", "steps"])
@pytest.mark.parametrize("backend", ["triton_shared_context", "flex_attention"], ids=["shared", "own"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("change", [_assign, _assign_twice, _one_weight, _data, _head, _constants], ids=lambda f: f.__name__[1:])
def test_the_next_call_takes_the_new_model(device, backend, dtype, whole_run, change):
    from ar_nanotabpfn_amd.inference import ARTabPFNPredictor

    B, Nc, Nt = 6, 40, 5
    g = torch.Generator().manual_seed(4)
    xc, yc = torch.randn(1, Nc, 2, generator=g).expand(B, -1, -1).to(device, dtype), torch.randn(1, Nc, generator=g).expand(B, -1).to(device, dtype)
    xt, yt = torch.randn(B, Nt, 2, generator=g).to(device, dtype), torch.randn(B, Nt, generator=g).to(device, dtype)

    def results(predictor):
        for _ in range(2):  # (a first run of the recorded route draws variates while it records)
            torch.manual_seed(5)
            drawn = predictor.sample_sequence(xc, yc, xt)
        return [drawn, predictor.evaluate_joint_density(xc, yc, xt, yt)]

    def predictor_of(m):
        p = ARTabPFNPredictor.from_trained_model(m, backend=backend)
        p.whole_run_decode = whole_run
        return p

    model, other = _model(1).to(device, dtype), _model(2).to(device, dtype)
    predictor = predictor_of(model)
    before = results(predictor)
    change(model, other)
    predictor.ar_tokens = model.ar_tokens
    got = results(predictor)
    fresh = _model(3).to(device, dtype)
    fresh.load_state_dict(model.state_dict())
    for a, b in zip(fresh.modules(), model.modules()):
        for name in ("eps", "std_min"):
            if hasattr(b, name):
                setattr(a, name, getattr(b, name))
    want = results(predictor_of(fresh))
    for b, x, w in zip(before, got, want):
        assert torch.equal(x, w) and not torch.equal(x, b)
