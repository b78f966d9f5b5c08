"""The layer stack as one call against the layer-by-layer form: the same launches, the same bits."""

import pytest
import torch

from ar_nanotabpfn_amd.inference import ARTabPFNPredictor
from ar_nanotabpfn_amd.model import ARTabPFN

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("backend", ["shared_context", "per_dataset"])
# one row, odd counts around a 16-row tile, a prefill whose keys are sliced, three head sizes
@pytest.mark.parametrize("B,Nc,Nt,D,H", [(1, 1, 1, 128, 4), (3, 17, 5, 128, 2), (2, 333, 45, 256, 8), (1, 1100, 16, 512, 4)])
def test_one_call_equals_layer_by_layer(device, monkeypatch, dtype, backend, B, Nc, Nt, D, H):
    torch.manual_seed(Nc)
    model = ARTabPFN(d_model=D, n_heads=H, n_layers=3, d_ff=256, num_features=2).to(device, dtype).eval()
    g = torch.Generator().manual_seed(Nt)
    xc, xt = (torch.randn(B, n, 2, generator=g).to(device, dtype) for n in (Nc, Nt))
    yc, yt = (torch.randn(B, n, generator=g).to(device, dtype) for n in (Nc, Nt))
    names = ("k_ctx_cache", "v_ctx_cache") if backend == "shared_context" else ("k_cache", "v_cache")

    def run(one_call):
        p = ARTabPFNPredictor.from_trained_model(model, backend=backend)
        taken = []
        stack = p._stack_pass
        monkeypatch.setattr(p, "_stack_pass", lambda *a: taken.append(stack(*a) if one_call else None) or taken[-1])
        out = p.evaluate_joint_density(xc, yc, xt, yt)
        assert len(taken) == 2 and all((t is not None) == one_call for t in taken)
        again = p.evaluate_joint_density(xc, yc, xt, yt)
        assert torch.equal(out, again)
        return [out] + [getattr(layer, n).clone() for layer in model.backbone.layers for n in names]

    for a, b in zip(run(True), run(False)):
        assert torch.equal(a, b)
    # a weight written to in place is seen by the next call
    before = run(True)[0]
    with torch.no_grad():
        model.backbone.layers[1].ff[0].weight.mul_(1.5)
        model.backbone.layers[2].norm2.bias.add_(0.5)
    after = run(True)
    assert not torch.equal(after[0], before)
    for a, b in zip(after, run(False)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("backend", ["shared_context", "per_dataset"])
# one row, odd counts around the 16-row tile, more tiles than compute units
@pytest.mark.parametrize("B,Nc,Nt,D,H", [(1, 1, 1, 128, 4), (3, 17, 5, 256, 8), (2, 333, 45, 512, 16), (64, 129, 65, 128, 2),
                                         (41, 201, 103, 256, 4)])
def test_float32_layers(device, monkeypatch, backend, B, Nc, Nt, D, H):
    """The float32 layer kernels against the library's products around the same attention."""
    torch.manual_seed(Nc)
    model = ARTabPFN(d_model=D, n_heads=H, n_layers=3, d_ff=256, num_features=2).to(device).eval()
    g = torch.Generator().manual_seed(Nt)
    xc, xt = (torch.randn(B, n, 2, generator=g).to(device) for n in (Nc, Nt))
    yc, yt = (torch.randn(B, n, generator=g).to(device) for n in (Nc, Nt))
    names = ("k_ctx_cache", "v_ctx_cache") if backend == "shared_context" else ("k_cache", "v_cache")

    def run(one_call):
        p = ARTabPFNPredictor.from_trained_model(model, backend=backend)
        stack = p._stack_pass
        taken = []
        monkeypatch.setattr(p, "_stack_pass", lambda *a: taken.append(stack(*a) if one_call else None) or taken[-1])
        out = p.evaluate_joint_density(xc, yc, xt, yt)
        assert len(taken) == 2 and all((t is not None) == one_call for t in taken)
        return [out] + [getattr(layer, n).clone() for layer in model.backbone.layers for n in names]

    # Sums of up to 512 float32 products in another order: each rounds at 2^-24 of its terms; three layers of five
    # products and three norms, whose gain is of order one, stay under 1e-5 of the result's size.
    for a, b in zip(run(True), run(False)):
        assert ((a - b).double().norm() / b.double().norm().clamp(min=1e-30)).item() < 1e-5
        assert torch.isfinite(a).all()


@pytest.mark.parametrize("D", [256, 512])
@pytest.mark.parametrize("rows", [4096, 4097, 4128, 8193])
def test_layer_boundary_tiles(device, D, rows):
    """Rows on both sides of the line between 16- and 32-row tiles: the same rows, alone and in the middle of more."""
    from ar_nanotabpfn_amd.model import TwoStageTransformerLayer

    torch.manual_seed(rows)
    la, lb = (TwoStageTransformerLayer(D, D // 32, 256).to(device, torch.bfloat16) for _ in range(2))
    x = torch.randn(1, rows, D, device=device).bfloat16()
    attn = torch.randn(1, rows, D // 32, 32, device=device).bfloat16().transpose(1, 2)
    with torch.no_grad():
        many = la.finish_then_pre(x, attn, lb)
        some = la.finish_then_pre(x[:, -200:], attn[:, :, -200:], lb)
    y, y_some = many[0][:, -200:].float(), some[0].float()
    # another order of the float32 sums: now and then a bfloat16 rounding of an intermediate goes the other way (2^-8)
    assert ((y - y_some).norm() / y_some.norm()).item() < 2.0 ** -8
    for a, b in zip(many[1:], some[1:]):
        a, b = a[:, :, -200:].float(), b.float()
        assert ((a - b).norm() / b.norm()).item() < 2.0 ** -7
