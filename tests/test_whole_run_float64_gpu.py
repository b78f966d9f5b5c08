"""The whole sampling run as one launch against float64: the rows it leaves in the caches and the values it draws, with
the values it drew as the oracle's buffer values.  Its error is that of the step-by-step routes, not more."""

import numpy as np
import pytest
import torch

from oracle.model_oracle import OracleModel, OraclePredictor

pytestmark = pytest.mark.gpu

# A rounding of an activation is 2^-9, 2^-12, 2^-25 of it at most.  Rows of the second layer have gone through some
# ten of them in 16 bits, which add up as random errors of a third of that each: 2.3 units measured; float32 sums of 128
# to 256 terms: 8.7 units measured.  The bound is four times that.
BOUND = {torch.bfloat16: 10 * 2.0 ** -9, torch.float16: 10 * 2.0 ** -12, torch.float32: 35 * 2.0 ** -25}


def _rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


def _f64(t):
    return t.detach().float().cpu().numpy().astype(np.float64)


@pytest.mark.parametrize("dtype", list(BOUND), ids=["bf16", "f16", "f32"])
@pytest.mark.parametrize("backend", ["triton_shared_context", "flex_attention"], ids=["shared", "own"])
# (d_model 128 with 300 rows, 256 with 150 and 300: a second and a third group of keys to every wavefront of a head)
@pytest.mark.parametrize("D,Nc,group", [(128, 3, 1), (128, 40, 3), (256, 33, 1), (128, 300, 1), (256, 150, 1), (256, 300, 1)])
def test_whole_run_against_float64(device, monkeypatch, tuning, dtype, backend, D, Nc, group):
    from ar_nanotabpfn_amd.glue import TrajectoryDecoder
    from ar_nanotabpfn_amd.inference import ARTabPFNPredictor
    from ar_nanotabpfn_amd.model import ARTabPFN

    tuning(ARTAB_TRAJECTORY=group)
    B, Nt, shared = 12, 20, backend == "triton_shared_context"
    torch.manual_seed(1)
    model = ARTabPFN(d_model=D, n_heads=D // 32, n_layers=2, d_ff=256, num_features=2, buffer_size=6, num_components=4).eval()
    with torch.no_grad():
        for layer in model.backbone.layers:  # scores of some spread
            layer.attn_rows.q_proj.weight.mul_(3)
            layer.attn_rows.k_proj.weight.mul_(3)
        model.head.weight_bias.copy_(torch.tensor([25.0, 0.0, 0.0, 0.0]))  # every draw from component 0
    model = model.to(device, dtype)
    g = torch.Generator().manual_seed(2)
    rows = 1 if shared else B
    xc, yc, xt = (torch.randn(*s, generator=g).to(device, dtype) for s in ((rows, Nc, 2), (rows, Nc), (B, Nt, 2)))
    xc, yc = xc.expand(B, -1, -1), yc.expand(B, -1)
    normals, call = [], TrajectoryDecoder.__call__
    monkeypatch.setattr(TrajectoryDecoder, "__call__", lambda self, *a: normals.append(a[5]) or call(self, *a))

    def run(whole):
        p = ARTabPFNPredictor.from_trained_model(model, backend=backend)
        p.whole_run_decode = whole
        y = p.sample_sequence(xc, yc, xt)
        first = 0 if shared else Nc
        k, v = ("k_buf_cache", "v_buf_cache") if shared else ("k_cache", "v_cache")
        left = [_f64(getattr(layer, n)[:, :, first:first + Nt - 1]) for layer in model.backbone.layers for n in (k, v)]
        oracle = OraclePredictor(OracleModel({n: _f64(t) for n, t in model.state_dict().items()}, D // 32),
                                 "shared" if shared else "per_dataset")
        z = oracle.fixed_buffer_decode(_f64(xc), _f64(yc), _f64(xt), _f64(y))
        want = [t for pair in zip(oracle.k_buf, oracle.v_buf) for t in pair]
        return y, oracle.m.head_parameterize(z), [_rel(a, b) for a, b in zip(left, want)]

    y, (mean, std, _), errors = run(True)
    assert len(normals) == 1
    drawn = mean[:, :, 0, 0] + std[:, :, 0, 0] * _f64(normals[0])[:Nt].T
    errors.append(_rel(_f64(y), drawn))
    _, _, steps = run(False)
    assert max(errors) <= BOUND[dtype], errors
    # (the two routes round at the same places; a tenth for other orders of summation)
    assert all(e <= 1.1 * s for e, s in zip(errors, steps)), (errors, steps)
