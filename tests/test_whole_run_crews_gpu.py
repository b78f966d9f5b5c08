"""The whole-run decode of one trajectory per workgroup (two crews of wavefronts) against the step-by-step route with
the same variates: where blocks and groups of keys end, contexts of both kinds, and the line to the one-crew kernel."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu

TOL = {torch.float32: 1e-4, torch.float16: 1e-2, torch.bfloat16: 2e-2}  # of the test of the other kernel: the same rounding


def _rel(a, b):
    a, b = a.double(), b.double()
    return float((a - b).norm() / b.norm().clamp(min=1e-30))


# Nc: one short of, at and past a block of 32 (16 in float32), a group of four, a group of both wavefronts of a head;
# Nt: own rows that begin a new block; 765 and 766 rows lie on either side of the line between the kernels in 16 bits; in
# float32 there is none, and a wavefront of the last two sizes has some tens of groups
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32], ids=["bf16", "f16", "f32"])
@pytest.mark.parametrize("backend", ["triton_shared_context", "flex_attention"], ids=["shared", "own"])
@pytest.mark.parametrize("D,Nc,Nt", [(128, 1, 3), (128, 31, 20), (128, 129, 36), (128, 256, 5), (256, 33, 35), (256, 127, 18),
                                     (256, 128, 3), (256, 765, 6), (256, 766, 6), (128, 2500, 4), (256, 3001, 4)])
def test_crews_equal_step_by_step(device, tuning, dtype, backend, D, Nc, Nt):
    from ar_nanotabpfn_amd.inference import ARTabPFNPredictor
    from ar_nanotabpfn_amd.model import ARTabPFN

    tuning(ARTAB_TRAJECTORY=1)
    B, L = 3, 2
    torch.manual_seed(3)
    model = ARTabPFN(d_model=D, n_heads=D // 32, n_layers=L, d_ff=256, num_features=2, buffer_size=6, num_components=4)
    with torch.no_grad():
        for name, p in model.named_parameters():
            if "norm" in name or name.endswith("bias"):
                p.add_(0.1 * torch.randn_like(p))
        # components that overlap: a draw on the boundary between two of them moves little
        model.head.head[2].weight.mul_(0.02)
        model.head.mean_bias.mul_(0.02)
        model.head.head[2].bias.zero_()
        model.head.std_bias.fill_(math.log(math.expm1(0.5)))
    model = model.eval().to(device, dtype)
    g = torch.Generator().manual_seed(4)
    rows = 1 if backend == "triton_shared_context" else B
    xc = torch.randn(rows, Nc, 2, generator=g).expand(B, -1, -1).to(device, dtype)
    yc = torch.randn(rows, Nc, generator=g).expand(B, -1).to(device, dtype)
    xt = torch.randn(B, Nt, 2, generator=g).to(device, dtype)
    names = ("k_buf_cache", "v_buf_cache") if backend == "triton_shared_context" else ("k_cache", "v_cache")
    results = {}
    for whole in (True, False):
        pred = ARTabPFNPredictor.from_trained_model(model, backend=backend)
        pred.whole_run_decode = whole
        for _ in range(2):  # (a first run of the recorded route draws variates while it records)
            torch.manual_seed(5)
            y = pred.sample_sequence(xc, yc, xt)
        assert (pred._trajectory is not None) == whole and torch.isfinite(y).all()
        results[whole] = y, [getattr(l, n).clone() for l in model.backbone.layers for n in names]
    (y1, c1), (y0, c0) = results[True], results[False]
    assert _rel(y1, y0) <= TOL[dtype]
    for a, b in zip(c1, c0):
        assert _rel(a, b) <= TOL[dtype]
