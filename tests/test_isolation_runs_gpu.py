"""A sampling run in one launch: a trajectory that meets a value that is not finite leaves the others of its
workgroup bit for bit as they are without it."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu


# two wavefronts per head, one, two heads per wavefront; groups of all sizes, full and with a remainder; fewer
# and more committed rows than a block of keys
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32], ids=["bf16", "f16", "f32"])
@pytest.mark.parametrize("backend", ["triton_shared_context", "flex_attention"], ids=["shared", "own"])
@pytest.mark.parametrize("D,B,Nc,Nt,group,at,when", [
    (128, 5, 33, 6, 2, 1, 2), (256, 13, 20, 40, 8, 4, 30), (512, 7, 31, 5, 3, 0, 1), (128, 9, 64, 70, 5, 6, 0)])
def test_one_trajectory_not_finite(device, tuning, dtype, backend, D, B, Nc, Nt, group, at, when):
    from ar_nanotabpfn_amd.inference import ARTabPFNPredictor
    from ar_nanotabpfn_amd.model import ARTabPFN

    if D == 512 and dtype == torch.float32:
        pytest.skip("D 512 is built for 16-bit types")
    tuning(ARTAB_TRAJECTORY=group)
    torch.manual_seed(3)
    model = ARTabPFN(d_model=D, n_heads=D // 32, n_layers=2, d_ff=256, num_features=2, buffer_size=6, num_components=4)
    model = model.eval().to(device, dtype)
    g = torch.Generator().manual_seed(4)
    shared = backend == "triton_shared_context"
    rows = 1 if shared else B
    xc = torch.randn(rows, Nc, 2, generator=g).expand(B, -1, -1).to(device, dtype)
    yc = torch.randn(rows, Nc, generator=g).expand(B, -1).to(device, dtype)
    xt = torch.randn(B, Nt, 2, generator=g).to(device, dtype)
    names = ("k_buf_cache", "v_buf_cache") if shared else ("k_cache", "v_cache")
    results = []
    for value in (None, math.inf):
        x = xt.clone()
        if value is not None:
            x[at, when, 0] = value
        pred = ARTabPFNPredictor.from_trained_model(model, backend=backend)
        torch.manual_seed(5)
        y = pred.sample_sequence(xc, yc, x)
        assert pred._trajectory is not None
        results.append((y, [getattr(l, n).clone() for l in model.backbone.layers for n in names]))
    (clean, c0), (got, c1) = results
    others = torch.arange(B, device=device) != at
    assert torch.isfinite(clean).all() and torch.equal(got[others], clean[others])
    assert torch.equal(got[at, :when], clean[at, :when]) and not torch.isfinite(got[at, when:]).any()
    for a, b in zip(c1, c0):
        assert torch.equal(a[others], b[others])
