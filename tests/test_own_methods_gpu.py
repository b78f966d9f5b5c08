"""Methods, modules and hooks of a program's own are called, also where a call in one launch would pass them by: the
results are those of the step-by-step, layer-by-layer routes."""

import pytest
import torch
from torch import nn

from ar_nanotabpfn_amd.inference import ARTabPFNPredictor
from ar_nanotabpfn_amd.model import ARTabPFN, Embedder, MixtureGaussianHead, TwoStageTransformerLayer

pytestmark = pytest.mark.gpu


class _Head(MixtureGaussianHead):
    def sample(self, z, num_samples=1):
        return 0.25 * super().sample(z, num_samples)


class _Parameters(MixtureGaussianHead):
    def _parameterize(self, z):
        mean, *rest = super()._parameterize(z)
        return (mean + 1, *rest)


class _Embedder(Embedder):
    def embed_target(self, x):
        return super().embed_target(5 - x)


class _Layer(TwoStageTransformerLayer):
    def finish(self, x_row, attn_heads):
        return super().finish(x_row, 0.5 * attn_heads)

    def finish_then_pre(self, x_row, attn_heads, next_layer):
        return next_layer.pre_attention(self.finish(x_row, attn_heads))


class _Predictor(ARTabPFNPredictor):
    def transformer_decode(self, embedding, commit):
        return -super().transformer_decode(embedding, commit)


def _class(attribute, cls):
    def change(p):
        getattr(p, attribute).__class__ = cls
    change.__name__ = cls.__name__
    return change


def _layer_class(p):
    p.backbone.layers[1].__class__ = _Layer


def _predictor_class(p):
    p.__class__ = _Predictor


def _bound_sample(p):
    p.head.sample = lambda z, num_samples=1: torch.zeros(z.shape[0], z.shape[1], num_samples, 1, device=z.device, dtype=z.dtype)


def _head_hook(p):
    p.head.head[0].register_forward_hook(lambda m, args, out: 2 * out)


def _embedding_hook(p):
    p.embedder.x_embed.register_forward_pre_hook(lambda m, args: (5 - args[0],))


def _relu(p):
    p.head.head[1] = nn.ReLU()


def _tanh_gelu(p):
    p.head.head[1] = nn.Sequential(nn.GELU(approximate="tanh"), nn.Tanh())


CHANGES = [_class("head", _Head), _class("head", _Parameters), _class("embedder", _Embedder), _layer_class, _predictor_class,
           _bound_sample, _head_hook, _embedding_hook, _relu, _tanh_gelu]


@pytest.mark.parametrize("backend", ["triton_shared_context", "flex_attention"], ids=["shared", "own"])
@pytest.mark.parametrize("change", CHANGES, ids=lambda f: f.__name__)
def test_what_a_program_puts_in_place_is_called(device, backend, change):
    B, Nc, Nt = 5, 40, 2  # (two targets: fewer than a recorded step is made for)
    g = torch.Generator().manual_seed(4)
    xc, yc = (torch.randn(B, Nc, *d, generator=g)[:1].expand(B, *[-1] * (1 + len(d))).to(device) for d in ((2,), ()))
    xt, yt = (torch.randn(B, Nt, *d, generator=g).to(device) for d in ((2,), ()))

    def results(changed, one_launch):
        torch.manual_seed(1)
        model = ARTabPFN(d_model=128, n_heads=4, n_layers=2, d_ff=256, num_features=2, buffer_size=6, num_components=4)
        p = ARTabPFNPredictor.from_trained_model(model.eval().to(device), backend=backend)
        p.use_hip_graph = one_launch  # (off: every step launch by launch)
        if not one_launch:
            p._stack_pass = lambda *a: None
        if changed:
            # a call before the change, as a program that changes a model later makes it
            p.sample_sequence(xc, yc, xt)
            change(p)
        torch.manual_seed(5)
        return [p.sample_sequence(xc, yc, xt), p.evaluate_joint_density(xc, yc, xt, yt)]

    want, got, plain = results(True, False), results(True, True), results(False, True)
    for g_, w in zip(got, want):
        assert torch.allclose(g_, w, rtol=1e-3, atol=1e-3)
    assert any(float((w - q).abs().max()) > 0.05 for w, q in zip(want, plain))
