"""The layer kernels for many rows (ARTAB_TILE_ROWS 33 / 64: one and two blocks of 32 rows per workgroup) against
float64 with the kernels' roundings, against the small-tile kernels' error, and fused against separate launches."""

import pytest
import torch

from .helpers import randn

pytestmark = pytest.mark.gpu


def _norm(D, seed, dtype, device):
    n = torch.nn.LayerNorm(D)
    with torch.no_grad():
        n.weight.copy_(randn((D,), seed, torch.float32) * 0.2 + 1)
        n.bias.copy_(randn((D,), seed + 1, torch.float32) * 0.2)
    return n.to(device, dtype)


def _ln64(x, n):
    return torch.nn.functional.layer_norm(x, x.shape[-1:], n.weight.double().cpu(), n.bias.double().cpu(), n.eps)


# one row; one short of, at and past a block and a tile of two; more tiles than one per XCD
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("tile", [33, 64])
@pytest.mark.parametrize("D,rows", [(128, 1), (128, 95), (256, 31), (256, 64), (256, 65), (256, 700), (512, 33)])
def test_wide_layer_matches_float64(device, tuning, dtype, tile, D, rows):
    from ar_nanotabpfn_amd.glue import layer_post, layer_post_pre, layer_pre, pack_weight

    F = 256
    attn, y = randn((rows, D), 1, dtype), randn((rows, 2 * D), 2, dtype, 1.5).to(device)[:, D:]  # strided residual rows
    w_o, w_fo = randn((D, D), 3, dtype, D ** -0.5), randn((D, D), 4, dtype, D ** -0.5)
    w_qkv = randn((3 * D, D), 5, dtype, D ** -0.5)
    w_1, w_2 = randn((F, D), 6, dtype, D ** -0.5), randn((D, F), 7, dtype, F ** -0.5)
    b_1, b_2 = randn((F,), 8, dtype, 0.3), randn((D,), 9, dtype, 0.3)
    n1, n2, n3 = (_norm(D, s, dtype, device) for s in (10, 12, 14))
    p_o, p_fo, p_qkv, p_1, p_2 = (pack_weight(w.to(device)) for w in (w_o, w_fo, w_qkv, w_1, w_2))
    post = (attn.to(device), y, p_o, n2, p_1, b_1.to(device), p_2, b_2.to(device), n3)

    # float64 on the same bits, rounded where the kernels keep 16 bits
    x1 = _ln64(y.cpu().double() + attn.double() @ w_o.double().t(), n2).to(dtype).double()
    h = torch.nn.functional.gelu(x1 @ w_1.double().t() + b_1.double()).to(dtype).double()
    out_ref = _ln64(x1 + h @ w_2.double().t() + b_2.double(), n3)
    x = out_ref.to(dtype).double()
    y_ref = _ln64(x + x @ w_fo.double().t(), n1)
    qkv_ref = y_ref.to(dtype).double() @ w_qkv.double().t()
    ulp = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11

    @torch.no_grad()
    def run(t):
        tuning(ARTAB_TILE_ROWS=t)
        out = layer_post(*post)
        return out, layer_pre(out, p_fo, n1, p_qkv), layer_post_pre(*post, p_fo, n1, p_qkv)

    def err(a, ref):
        return float((a.cpu().double() - ref).norm() / ref.norm())

    out, (y_sep, qkv_sep), (y_one, qkv_one) = run(tile)
    assert torch.equal(y_sep, y_one) and torch.equal(qkv_sep, qkv_one)
    out_s, (y_s, qkv_s), _ = run(32)
    # the bounds of the small-tile kernels' tests: a rounding or two of the largest entry
    assert float((out.cpu().double() - out_ref).abs().max()) <= 3 * ulp * max(1.0, float(out_ref.abs().max()))
    assert float((y_one.cpu().double() - y_ref).abs().max()) <= 4 * ulp * max(1.0, float(y_ref.abs().max()))
    # no further from float64 than the small tiles: the same roundings, which of them flip is chance (1 % of the sum of
    # some ten thousand of them; single rows 10 %)
    slack = 1.02 if rows * D > 10000 else 1.1
    for a, s, ref in ((out, out_s, out_ref), (y_one, y_s, y_ref), (qkv_one, qkv_s, qkv_ref)):
        assert err(a, ref) <= slack * err(s, ref)


@pytest.mark.parametrize("rows,tile", [(4096, 16), (8192, 32), (8193, 33), (24577, 64)])
def test_rule(device, tuning, rows, tile):
    """Which kernel a row count takes: the bits of the one it should be, and of no other."""
    from ar_nanotabpfn_amd.glue import layer_post, pack_weight

    dtype, D = torch.bfloat16, 256
    g = torch.Generator(device).manual_seed(1)
    attn, y = (torch.randn(rows, D, generator=g, device=device).to(dtype) for _ in range(2))
    p_o, p_1, p_2 = (pack_weight(randn((D, D), s, dtype, D ** -0.5).to(device)) for s in (3, 6, 7))
    n2, n3 = (_norm(D, s, dtype, device) for s in (12, 14))
    results = {}
    for t in (None, 16, 32, 33, 64):
        tuning(ARTAB_TILE_ROWS=t)
        results[t] = layer_post(attn, y, p_o, n2, p_1, None, p_2, None, n3)
    for t in (16, 32, 33, 64):
        assert torch.equal(results[None], results[t]) == (t == tile)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("backend", ["shared_context", "per_dataset"])
# batch entries that end inside a tile and inside its 16-row stores; one row per entry; head sizes 32, 64 and 128
@pytest.mark.parametrize("B,Nc,Nt,D,H,tile", [(1, 77, 5, 128, 4, 33), (3, 17, 5, 256, 8, 64), (5, 33, 1, 256, 4, 33), (2, 65, 31, 512, 4, 33),
                                              (41, 3, 2, 128, 4, 33)])
def test_keys_and_values_go_to_the_caches(device, tuning, monkeypatch, dtype, backend, B, Nc, Nt, D, H, tile):
    """Prefill and teacher forcing as one call, where the layer kernels write keys and values into the caches and the
    attention reads them there, against the layer-by-layer form, which copies them: the same bits."""
    from ar_nanotabpfn_amd.inference import ARTabPFNPredictor
    from ar_nanotabpfn_amd.model import ARTabPFN

    tuning(ARTAB_TILE_ROWS=tile)
    torch.manual_seed(Nc)
    model = ARTabPFN(d_model=D, n_heads=H, n_layers=3, d_ff=256, num_features=2).to(device, dtype).eval()
    g = torch.Generator().manual_seed(Nt)
    xc, xt = (torch.randn(B, n, 2, generator=g).to(device, dtype) for n in (Nc, Nt))
    yc, yt = (torch.randn(B, n, generator=g).to(device, dtype) for n in (Nc, Nt))
    names = ("k_ctx_cache", "v_ctx_cache") if backend == "shared_context" else ("k_cache", "v_cache")

    def run(one_call):
        p = ARTabPFNPredictor.from_trained_model(model, backend=backend)
        stack = p._stack_pass
        monkeypatch.setattr(p, "_stack_pass", lambda *a: stack(*a) if one_call else None)
        out = p.evaluate_joint_density(xc, yc, xt, yt)
        return [out] + [getattr(layer, n).clone() for layer in model.backbone.layers for n in names]

    for a, b in zip(run(True), run(False)):
        assert torch.equal(a, b)
