"""What prepared calls go by (``ar_nanotabpfn_amd.live``): every exchange of a parameter, a module or a constant is seen,
an unchanged model is not prepared again."""

import torch
from torch import nn

from ar_nanotabpfn_amd.live import ModelState, Sources
from ar_nanotabpfn_amd.model import ARTabPFN, MixtureGaussianHead


def _model():
    torch.manual_seed(0)
    return ARTabPFN(d_model=32, n_heads=2, n_layers=2, d_ff=64, num_features=2, buffer_size=4, num_components=3)


def _changes():
    def weight(m):
        m.backbone.layers[1].ff[0].weight = nn.Parameter(m.backbone.layers[1].ff[0].weight.detach().clone())

    def assign(m):
        m.load_state_dict({k: v.clone() for k, v in m.state_dict().items()}, assign=True)

    def head(m):
        m.head = MixtureGaussianHead(32, 64, num_components=3)

    def data(m):
        m.backbone.layers[0].norm1.bias.data = torch.ones(32)

    def in_place(m):
        with torch.no_grad():
            m.embedder.x_embed.weight.mul_(2)

    def layer(m):
        m.backbone.layers[0], m.backbone.layers[1] = m.backbone.layers[1], m.backbone.layers[0]

    def eps(m):
        m.backbone.layers[1].norm2.eps = 1e-3

    def std_min(m):
        m.head.std_min = 0.5

    def heads(m):
        m.backbone.layers[0].attn_rows.n_heads = 4

    def tokens(m):
        m.ar_tokens = nn.Parameter(torch.zeros(4, 32))

    def activation(m):
        m.head.head[1] = nn.ReLU()

    def no_bias(m):
        m.head.head[0].bias = None

    return [f for f in locals().values() if callable(f)]


def test_every_change_is_seen_and_nothing_else():
    for change in _changes():
        m, state = _model(), ModelState()
        look = lambda: state.look((m.backbone, m.embedder, m.head), m.ar_tokens)  # noqa: E731
        first = look()
        assert look() == first
        m.state_dict()
        assert look() == first
        change(m)
        second = look()
        assert second != first, change.__name__
        assert look() == second, change.__name__


def test_an_address_that_comes_back_is_not_the_same_tensor():
    # a parameter exchanged twice between two looks can get the memory of the first one, and starts at version 0
    # as the first did: its memory is held instead
    p = [nn.Parameter(torch.randn(1000))]
    sources, at = Sources(p), p[0].data_ptr()
    for _ in range(50):
        p[0] = nn.Parameter(torch.randn(1000))
        assert not sources.unchanged(p) and p[0].data_ptr() != at
    q = nn.Parameter(torch.randn(1000))
    sources, at = Sources([q]), q.data_ptr()
    for _ in range(50):
        q.data = torch.randn(1000)
        assert not sources.unchanged([q]) and q.data_ptr() != at
