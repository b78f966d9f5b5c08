"""Both ends of a prefill or a density as one launch each, against the modules in float64 and in the model's type."""

import copy
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

UNIT = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -24}  # the largest error of one rounding
DTYPES = pytest.mark.parametrize("dtype", list(UNIT), ids=["bf16", "f16", "f32"])


def _model(device, dtype, D, K, bs=7):
    from ar_nanotabpfn_amd.model import ARTabPFN

    torch.manual_seed(D + K)
    model = ARTabPFN(d_model=D, n_heads=D // 32, n_layers=1, d_ff=256, num_features=3, buffer_size=bs, num_components=K)
    with torch.no_grad():
        for p in (model.embedder.marker_embed.weight, model.ar_tokens, model.backbone.norm.weight, model.backbone.norm.bias):
            p.add_(0.3 * torch.randn_like(p))
    return model.to(device, dtype).eval()


def _rel(a, b):
    return float((a.double() - b).norm() / b.norm().clamp(min=1e-30))


@DTYPES
@pytest.mark.parametrize("D,B,N,C,layout", [(128, 1, 1, 1, "dense"), (256, 3, 33, 4, "expanded"), (512, 2, 9, 21, "slice"), (128, 5, 70, 2, "columns")])
@torch.no_grad()
def test_embedded_rows(device, dtype, D, B, N, C, layout):
    from ar_nanotabpfn_amd.glue import embed_context_rows

    model = _model(device, dtype, D, 3)
    g = torch.Generator().manual_seed(N)
    if layout == "expanded":
        x, y = (torch.randn(1, *s, generator=g).to(device, dtype).expand(B, *s) for s in ((N, C), (N,)))
    else:
        x, y = torch.randn(B, N + 5, C, generator=g).to(device, dtype), torch.randn(B, N + 5, generator=g).to(device, dtype)
        if layout == "columns":
            x = torch.randn(C, B, N + 5, generator=g).to(device, dtype).permute(1, 2, 0)
        x, y = (x[:, 3:N + 3], y[:, 3:N + 3]) if layout == "slice" else (x[:, :N].contiguous(), y[:, :N].contiguous()) if layout == "dense" else (x[:, :N], y[:, :N])
    e, wide = model.embedder, copy.deepcopy(model).double().embedder
    xd, yd, tokens = x.double(), y.double(), model.ar_tokens[torch.arange(N, device=device) % 7]
    for got, modules, want in (
            (embed_context_rows(e, x, y), e.embed_context(x, y), wide.embed_context(xd, yd)),
            (embed_context_rows(e, x, y.unsqueeze(-1), model.ar_tokens), torch.cat([e.embed_buffer(x, y) + tokens, e.embed_target(x)], dim=1),
             torch.cat([wide.embed_buffer(xd, yd) + tokens.double(), wide.embed_target(xd)], dim=1))):
        assert got.shape == want.shape and got.dtype == dtype and got.is_contiguous()
        # one rounding (in float32 some ten, of random sign), and no further off than the modules, which round every step
        assert _rel(got, want) <= (4 if dtype == torch.float32 else 1) * UNIT[dtype]
        assert dtype == torch.float32 or _rel(got, want) <= _rel(modules, want)


@pytest.mark.parametrize("C", [7, 8, 9, 21, 64])
@torch.no_grad()
def test_embedded_rows_of_many_features(device, C):
    """Features whose sum grows with their number: the mean's error must not."""
    from ar_nanotabpfn_amd.glue import embed_context_rows

    e = _model(device, torch.float32, 128, 3).embedder
    g = torch.Generator().manual_seed(C)
    x, y = (torch.randn(2, 200, C, generator=g) + 3).to(device), torch.randn(2, 200, generator=g).to(device)
    want = copy.deepcopy(e).double().embed_context(x.double(), y.double())
    # the mean is rounded once and each later step as in the modules, or not at all: their error at most, of 51200 values with some five
    # roundings of random sign (a share of 1/sqrt(5 x 51200) of it by chance, five times that allowed)
    assert _rel(embed_context_rows(e, x, y), want) <= 1.01 * _rel(e.embed_context(x, y), want)
    wide = torch.cat([x] * 10, dim=-1)
    assert embed_context_rows(e, wide[..., :64], y) is not None and embed_context_rows(e, wide[..., :65], y) is None


@DTYPES
@pytest.mark.parametrize("D,K,B,Nt,shift", [(128, 2, 1, 1, 0.0), (256, 5, 3, 17, 0.0), (512, 20, 2, 40, 0.0), (256, 21, 16, 45, 0.0),
                                            (128, 22, 1, 16, 0.0), (256, 42, 4, 9, 2.0)])
@torch.no_grad()
def test_log_densities(device, dtype, D, K, B, Nt, shift):
    from ar_nanotabpfn_amd.glue import mixture_log_density

    model = _model(device, dtype, D, K)
    g = torch.Generator().manual_seed(Nt)
    rows, y = torch.randn(B, 2 * Nt, D, generator=g).to(device, dtype), torch.randn(Nt, B, generator=g).to(device, dtype).t() + shift
    got = mixture_log_density(model.backbone.norm, model.head, rows[:, Nt:], y)
    wide = copy.deepcopy(model).double()
    want = wide.head.log_likelihood(wide.backbone.norm(rows[:, Nt:].double()), y.double().unsqueeze(-1))
    modules = model.head.log_likelihood(model.backbone.norm(rows[:, Nt:]), y.unsqueeze(-1))
    assert got.shape == (B, Nt) and got.dtype == dtype
    # z and the hidden layer are rounded to the type (float32: sums of up to 512 terms), and the densities' quotient
    # (y - mean) / std carries a part of that many times over
    assert _rel(got, want) <= 6 * UNIT[dtype] + _rel(modules, want) * (0.0 if dtype != torch.float32 else 1.5)
    assert dtype == torch.float32 or _rel(got, want) <= _rel(modules, want)


@torch.no_grad()
def test_values_that_are_not_finite(device):
    from ar_nanotabpfn_amd.glue import mixture_log_density

    model = _model(device, torch.float32, 128, 5)
    rows, y = torch.randn(3, 8, 128, device=device), torch.randn(3, 8, device=device)
    want = model.head.log_likelihood(model.backbone.norm(rows), y.unsqueeze(-1))
    rows[1, 2, 7], y[2, 3], y[0, 1] = float("nan"), float("nan"), float("inf")
    got = mixture_log_density(model.backbone.norm, model.head, rows, y)
    modules = model.head.log_likelihood(model.backbone.norm(rows), y.unsqueeze(-1))
    assert torch.equal(torch.isnan(got), torch.isnan(modules)) and torch.equal(torch.isinf(got), torch.isinf(modules))
    finite = torch.isfinite(modules)
    assert int(finite.sum()) == 21 and torch.allclose(got[finite], want[finite], atol=1e-4)


def test_modules_of_a_program_are_called(device):
    """Hooks, overridden methods, recorded gradients, autocast and tangents: the modules run."""
    import torch.autograd.forward_ad as fwad

    from ar_nanotabpfn_amd.glue import embed_context_rows, mixture_log_density
    from ar_nanotabpfn_amd.inference import ARTabPFNPredictor

    model = _model(device, torch.float32, 128, 3)
    x, y, rows = torch.randn(2, 5, 3, device=device), torch.randn(2, 5, device=device), torch.randn(2, 5, 128, device=device)
    assert embed_context_rows(model.embedder, x, y) is None and mixture_log_density(model.backbone.norm, model.head, rows, y) is None
    with torch.no_grad():
        with torch.autocast("cuda", dtype=torch.bfloat16):
            assert embed_context_rows(model.embedder, x, y) is None
        with fwad.dual_level():
            assert mixture_log_density(model.backbone.norm, model.head, rows, y) is None
        assert embed_context_rows(model.embedder, x, y.half()) is None and embed_context_rows(model.embedder, x, y[:, :4]) is None
        assert mixture_log_density(model.backbone.norm, model.head, rows, y[:1]) is None
    seen = []
    for module in (model.embedder.x_embed, model.head.head[2]):
        module.register_forward_hook(lambda *a: seen.append(a[0]))
    pred = ARTabPFNPredictor.from_trained_model(model, backend="triton_shared_context")
    plain = ARTabPFNPredictor.from_trained_model(_model(device, torch.float32, 128, 3), backend="triton_shared_context")
    data = (x[:1].expand(2, -1, -1), y[:1].expand(2, -1), x + 1, y + 1)
    a, b = pred.evaluate_joint_density(*data), plain.evaluate_joint_density(*data)
    assert len(seen) >= 3 and torch.allclose(a, b, atol=1e-4)


def test_arguments_are_checked():
    from ar_nanotabpfn_amd import _lib

    lib, f32 = _lib.load(), _lib.ARTAB_F32
    a = _lib.ArtabEmbedRowsArgs()
    a.B = a.N = a.C = 1
    a.D = 12
    call = lambda: lib.artab_embed_rows(ctypes.byref(a), f32, None)  # noqa: E731
    assert call() == _lib.ARTAB_ERR_UNSUPPORTED
    a.D = 128
    assert call() == _lib.ARTAB_ERR_NULL_POINTER
    a.B = 2 ** 26
    assert call() == _lib.ARTAB_ERR_BAD_SHAPE
    a.B = 0
    assert call() == 0
    d = _lib.ArtabDensityArgs()
    d.B = d.Nt = d.K = 1
    d.D, d.F = 128, 128
    assert lib.artab_density(ctypes.byref(d), f32, None) == _lib.ARTAB_ERR_UNSUPPORTED
    d.F = 256
    assert lib.artab_density(ctypes.byref(d), f32, None) == _lib.ARTAB_ERR_NULL_POINTER
    assert not lib.artab_density_supported(256, 256, 43) and lib.artab_density_supported(512, 256, 42)
