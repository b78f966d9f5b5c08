"""Models and predictors that have been used are copied and pickled like new ones, and the copy computes the same."""

import copy
import io

import pytest
import torch

pytestmark = pytest.mark.gpu


def _pickled(x):
    f = io.BytesIO()
    torch.save(x, f)
    f.seek(0)
    return torch.load(f, weights_only=False)


@pytest.mark.parametrize("duplicate", [copy.deepcopy, copy.copy, _pickled], ids=["deepcopy", "copy", "pickle"])
@pytest.mark.parametrize("backend", ["triton_shared_context", "flex_attention"], ids=["shared", "own"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("whole_run", [True, False], ids=["run", "steps"])
def test_copy_of_a_used_predictor(device, duplicate, backend, dtype, whole_run):
    from ar_nanotabpfn_amd.inference import ARTabPFNPredictor
    from ar_nanotabpfn_amd.model import ARTabPFN

    torch.manual_seed(1)
    model = ARTabPFN(d_model=128, n_heads=4, n_layers=2, d_ff=256, num_features=2, buffer_size=6, num_components=4)
    p = ARTabPFNPredictor.from_trained_model(model.eval().to(device, dtype), backend=backend)
    p.whole_run_decode = whole_run
    g = torch.Generator().manual_seed(4)
    xc, yc = (torch.randn(1, 30, *d, generator=g).expand(4, *[-1] * (1 + len(d))).to(device, dtype) for d in ((2,), ()))
    xt = torch.randn(4, 5, 2, generator=g).to(device, dtype)

    def results(p):
        for _ in range(2):  # (a first run of the recorded route draws variates while it records)
            torch.manual_seed(5)
            y = p.sample_sequence(xc, yc, xt)
        return [y, p.evaluate_joint_density(xc, yc, xt, y)]

    want = results(p)
    q = duplicate(p)
    assert q.whole_run_decode == whole_run and q.backend == p.backend and q.seq_len == p.seq_len
    for a, b in zip(results(q), want):
        assert torch.equal(a, b)
    m = duplicate(model)  # (it has prepared weights by now)
    for a, b in zip(results(ARTabPFNPredictor.from_trained_model(m, backend=backend)) if whole_run else [], want):
        assert torch.equal(a, b)
    for a, b in zip(results(p), want):
        assert torch.equal(a, b)
