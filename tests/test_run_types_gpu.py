"""A model or a cache that is not of the one type and size that the whole-run launch reads: what the step-by-step route
does with it, an error or values, happens with the launch switched on too."""

import pytest
import torch
from torch import nn

pytestmark = pytest.mark.gpu


def _head_32_bit(p):
    p.head.float()


def _head_16_bit(p):
    p.head.bfloat16()


def _tokens_64_bit(p):
    p.ar_tokens = nn.Parameter(p.ar_tokens.detach().double())


def _embedder_64_bit(p):
    p.embedder.double()



def _short_weight(p):
    ff = p.backbone.layers[1].ff
    ff[2].weight = nn.Parameter(ff[2].weight.detach()[:, :128].contiguous())


def _short_tokens(p):
    p.ar_tokens = nn.Parameter(p.ar_tokens.detach()[:1].contiguous())


CASES = [_head_32_bit, _head_16_bit, _tokens_64_bit, _embedder_64_bit, _short_weight, _short_tokens]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("change", CASES, ids=lambda f: f.__name__[1:])
def test_both_routes_do_the_same(device, change, dtype):
    from ar_nanotabpfn_amd.inference import ARTabPFNPredictor
    from ar_nanotabpfn_amd.model import ARTabPFN

    B, Nc, Nt = 4, 20, 3
    g = torch.Generator().manual_seed(4)
    xc, yc, xt = (torch.randn(*s, generator=g).to(device, dtype) for s in ((B, Nc, 2), (B, Nc), (B, Nt, 2)))

    def outcome(whole):
        torch.manual_seed(1)
        model = ARTabPFN(d_model=128, n_heads=4, n_layers=2, d_ff=256, num_features=2, buffer_size=6, num_components=4)
        p = ARTabPFNPredictor.from_trained_model(model.eval().to(device, dtype), backend="flex_attention")
        p.whole_run_decode = whole
        p.init_kv_cache(B, Nc + Nt, device, dtype)
        p.prefill_context(xc, yc)
        change(p)
        torch.manual_seed(5)
        try:
            return p.decode_targets(xt), None
        except (RuntimeError, ValueError) as err:
            return None, type(err)

    (got, error), (want, want_error) = outcome(True), outcome(False)
    assert error is want_error
    if want is not None:
        assert got.dtype == want.dtype and torch.allclose(got.float(), want.float(), rtol=3e-2, atol=3e-2)


def test_caches_of_several_sizes_are_left_to_the_other_route(device):
    from ar_nanotabpfn_amd.inference import ARTabPFNPredictor
    from ar_nanotabpfn_amd.model import ARTabPFN

    B, Nc, Nt = 4, 20, 3
    model = ARTabPFN(d_model=128, n_heads=4, n_layers=2, d_ff=256, num_features=2, buffer_size=6, num_components=4).eval().to(device)
    x = torch.randn(B, Nt, 2, device=device)
    for backend, name in (("flex_attention", "v_cache"), ("triton_shared_context", "k_buf_cache"), ("triton_shared_context", "v_ctx_cache")):
        p = ARTabPFNPredictor.from_trained_model(model, backend=backend)
        p.init_kv_cache(B, Nc + Nt, device, torch.float32)
        p.prefill_context(torch.randn(B, Nc, 2, device=device), torch.randn(B, Nc, device=device))
        layer = model.backbone.layers[1]
        kept = getattr(layer, name)
        setattr(layer, name, torch.cat([kept, kept], dim=-2))
        assert p._sample_whole_run(x) is None  # (nothing is launched)
        setattr(layer, name, kept)
        assert p._sample_whole_run(x) is not None
