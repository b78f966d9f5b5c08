"""A training step whose modules are not those the fused kernels stand for runs as modules: loss and gradients are
those of the module route, and what was put in place is run."""

import types

import pytest
import torch
from torch import nn

import ar_nanotabpfn_amd.model as model_mod
from ar_nanotabpfn_amd.attention import MultiheadAttention, create_dense_mask, create_row_mask

pytestmark = pytest.mark.gpu

D, H, B, NC, NB, NT = 128, 4, 3, 17, 4, 12


class _Adapter(nn.Module):
    """A projection with a trained correction, in the form adapter libraries give it."""

    def __init__(self, base):
        super().__init__()
        self.base, self.delta = base, nn.Linear(D, D, bias=False, device=base.weight.device)

    @property
    def weight(self):
        return self.base.weight

    @property
    def bias(self):
        return None

    def forward(self, x):
        return self.base(x) + self.delta(x)


class _Layer(model_mod.TwoStageTransformerLayer):
    def _forward_recording(self, x_row, mask_rows):
        out, kv = super()._forward_recording(x_row, mask_rows)
        return 0.5 * out, kv


class _Attention(MultiheadAttention):
    def forward(self, q, k, v, mask):
        out, kv = super().forward(q, k, v, mask)
        return 2 * out, kv


class _Embedder(model_mod.Embedder):
    def embed_context(self, x, y):
        return 2 * super().embed_context(x, y)


def _relu(m):
    m.backbone.layers[1].ff[1] = nn.ReLU()


def _tanh_gelu(m):
    m.backbone.layers[0].ff[1] = nn.GELU(approximate="tanh")


def _adapter(m):
    a = m.backbone.layers[0].attn_rows
    a.q_proj = _Adapter(a.q_proj)


def _layer_class(m):
    m.backbone.layers[1].__class__ = _Layer


def _attention_class(m):
    m.backbone.layers[1].attn_rows.__class__ = _Attention


def _bound_forward(m):
    ff = m.backbone.layers[0].ff
    ff.forward = types.MethodType(lambda self, x: 2 * nn.Sequential.forward(self, x), ff)


def _projection_bias(m):
    m.backbone.layers[0].attn_features.out_proj = nn.Linear(D, D).cuda()


def _plain_norm(m):
    m.backbone.norm = nn.LayerNorm(D, elementwise_affine=False).cuda()


def _norm_16_bit(m):
    m.backbone.norm.to(torch.bfloat16)


def _extra_module(m):
    m.backbone.layers[0].ff.append(nn.Tanh())


def _hook(m):
    m.calls = []
    m.backbone.layers[1].ff[0].register_forward_hook(lambda *a: m.calls.append(1))


def _backward_hook(m):
    m.calls = []
    m.backbone.layers[0].norm2.register_full_backward_hook(lambda *a: m.calls.append(1))


def _backbone_hook(m):
    m.calls = []
    m.backbone.register_forward_pre_hook(lambda *a: m.calls.append(1))


def _embedder_class(m):
    m.embedder.__class__ = _Embedder


def _embedder_hook(m):
    m.calls = []
    m.embedder.y_embed.register_forward_hook(lambda *a: m.calls.append(1))


BACKBONE = [_relu, _tanh_gelu, _adapter, _layer_class, _attention_class, _bound_forward, _projection_bias, _plain_norm, _norm_16_bit,
            _extra_module, _hook, _backward_hook, _backbone_hook]
EMBEDDER = [_embedder_class, _embedder_hook]


def _step(model, device):
    g = torch.Generator().manual_seed(2)
    mk = lambda *s: torch.randn(*s, generator=g).to(device)  # noqa: E731
    data, y = (mk(B, NC, 2), mk(B, NC), mk(B, NB, 2), mk(B, NB), mk(B, NT, 2)), mk(B, NT)
    model.zero_grad(set_to_none=True)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        loss = model(*data, create_dense_mask(1), create_row_mask(NC + NB + NT, NC, NB), y_target=y)
    loss.backward()
    return loss.item(), {n: p.grad.clone() for n, p in model.named_parameters()}


def _model(device):
    torch.manual_seed(1)
    return model_mod.ARTabPFN(d_model=D, n_heads=H, n_layers=2, d_ff=256, num_features=2, buffer_size=NB, num_components=5).to(device)


def _routes(monkeypatch):
    """Counts the calls of the two fused forms."""
    calls = {"layer_stack": 0, "embed_rows": 0}

    def counted(name, f):
        def call(*a):
            out = f(*a)
            calls[name] += out is not None
            return out
        return call

    for name in calls:
        monkeypatch.setattr(model_mod, name, counted(name, getattr(model_mod, name)))
    return calls


@pytest.mark.parametrize("change", BACKBONE + EMBEDDER, ids=lambda f: f.__name__[1:])
def test_other_modules_are_run(device, monkeypatch, change):
    model = _model(device)
    calls = _routes(monkeypatch)
    _step(model, device)
    assert calls == {"layer_stack": 1, "embed_rows": 1}
    torch.manual_seed(3)
    change(model)
    loss, grads = _step(model, device)
    assert calls["layer_stack" if change in BACKBONE else "embed_rows"] == 1
    if hasattr(model, "calls"):
        assert model.calls
    monkeypatch.setattr(model_mod, "layer_stack_supported", lambda *a: False)
    monkeypatch.setattr(model_mod, "embed_rows", lambda *a: None)
    ref_loss, ref = _step(model, device)
    assert abs(loss - ref_loss) <= 5e-3 * abs(ref_loss)
    assert grads.keys() == ref.keys()
    for n, r in ref.items():  # (the bound of the test that compares the two routes)
        assert float((grads[n] - r).norm()) <= 4e-2 * float(r.norm()) + 1e-6, n


def test_hooks_on_every_module_are_run(device, monkeypatch):
    model, seen = _model(device), set()
    calls = _routes(monkeypatch)
    hook = nn.modules.module.register_module_forward_hook(lambda m, a, out: seen.add(m))
    try:
        _step(model, device)
    finally:
        hook.remove()
    assert calls == {"layer_stack": 0, "embed_rows": 0} and set(model.backbone.layers[0].ff) <= seen
    _step(model, device)
    assert calls == {"layer_stack": 1, "embed_rows": 1}
