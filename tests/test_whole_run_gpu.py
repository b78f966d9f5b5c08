"""The whole sampling run as one launch (``ARTabPFNPredictor.whole_run_decode``) against the step-by-step
routes with the same variates: drawn values and the K/V rows left in the caches."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu

TOL = {torch.float32: 1e-4, torch.float16: 1e-2, torch.bfloat16: 2e-2}


def _rel(a, b):
    a, b = a.double(), b.double()
    return float((a - b).norm() / b.norm().clamp(min=1e-30))


# edges: no buffer row at all (Nt = 1), one; contexts shorter than a key block, one key past whole blocks;
# one trajectory, groups that do not divide the batch; two wavefronts per head (D 128), two heads per
# wavefront (D 512); more mixture components than the step tail takes
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32], ids=["bf16", "f16", "f32"])
@pytest.mark.parametrize("backend", ["triton_shared_context", "flex_attention"], ids=["shared", "own"])
@pytest.mark.parametrize("D,L,K,B,Nc,Nt,group", [
    (128, 2, 20, 1, 1, 1, 1), (128, 3, 5, 5, 33, 2, 2), (256, 2, 5, 13, 64, 40, 8), (256, 1, 21, 3, 97, 35, 1),
    (512, 2, 3, 7, 31, 5, 3), (128, 2, 4, 9, 200, 70, 5)])
def test_whole_run_equals_step_by_step(device, tuning, dtype, backend, D, L, K, B, Nc, Nt, group):
    from ar_nanotabpfn_amd.inference import ARTabPFNPredictor
    from ar_nanotabpfn_amd.model import ARTabPFN

    if D == 512 and dtype == torch.float32:
        pytest.skip("D 512 is built for 16-bit types")
    tuning(ARTAB_TRAJECTORY=group)
    torch.manual_seed(3)
    model = ARTabPFN(d_model=D, n_heads=D // 32, n_layers=L, d_ff=256, num_features=2, buffer_size=6, num_components=K)
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
        assert (pred._trajectory is not None) == whole and y.shape == (B, Nt) and torch.isfinite(y).all()
        results[whole] = (y, [getattr(l, n).clone() for l in model.backbone.layers for n in names], pred.seq_len, pred.buffer_len)
    (y1, c1, *s1), (y0, c0, *s0) = results[True], results[False]
    assert s1 == s0
    assert _rel(y1, y0) <= TOL[dtype]
    for a, b in zip(c1, c0):
        assert _rel(a, b) <= TOL[dtype]
