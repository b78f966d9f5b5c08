"""A model whose parameters are views into one vector, as flat optimisers and ``vector_to_parameters`` leave them: those of the
head lie at addresses that are not multiples of 16 bytes."""

import pytest
import torch
from torch.nn.utils import parameters_to_vector, vector_to_parameters

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("backend", ["triton_shared_context", "flex_attention"], ids=["shared", "own"])
def test_sampling_and_density(device, backend, dtype):
    from ar_nanotabpfn_amd.inference import ARTabPFNPredictor
    from ar_nanotabpfn_amd.model import ARTabPFN

    g = torch.Generator().manual_seed(4)
    xc, yc = (torch.randn(1, 30, *d, generator=g).expand(4, *[-1] * (1 + len(d))).to(device, dtype) for d in ((2,), ()))
    xt = torch.randn(4, 5, 2, generator=g).to(device, dtype)
    results = []
    for flat in (False, True):
        torch.manual_seed(1)
        model = ARTabPFN(d_model=128, n_heads=4, n_layers=2, d_ff=256, num_features=2, buffer_size=6, num_components=5)
        model = model.eval().to(device, dtype)
        if flat:
            vector_to_parameters(parameters_to_vector(model.parameters()), model.parameters())
            assert model.head.head[0].weight.data_ptr() % 16
        p = ARTabPFNPredictor.from_trained_model(model, backend=backend)
        torch.manual_seed(5)
        y = p.sample_sequence(xc, yc, xt)
        results.append([y, p.evaluate_joint_density(xc, yc, xt, results[0][0] if flat else y)])
    for a, b in zip(*results):
        assert torch.equal(a, b)


def test_training(device):
    import ar_nanotabpfn_amd.model as model_mod
    from ar_nanotabpfn_amd.attention import create_dense_mask, create_row_mask

    g = torch.Generator().manual_seed(2)
    mk = lambda *s: torch.randn(*s, generator=g).to(device)  # noqa: E731
    data, y = (mk(3, 17, 2), mk(3, 17), mk(3, 4, 2), mk(3, 4), mk(3, 12, 2)), mk(3, 12)
    losses = []
    for flat in (False, True):
        torch.manual_seed(1)
        model = model_mod.ARTabPFN(d_model=128, n_heads=4, n_layers=2, d_ff=256, num_features=2, buffer_size=4, num_components=5).to(device)
        if flat:  # the first parameter after one of odd size: every layer's lie off 16 bytes
            v = torch.cat([torch.zeros(1, device=device), parameters_to_vector(model.parameters())])
            vector_to_parameters(v[1:], model.parameters())
            assert model.backbone.layers[0].ff[0].weight.data_ptr() % 16
        with torch.autocast("cuda", dtype=torch.bfloat16):
            loss = model(*data, create_dense_mask(1), create_row_mask(33, 17, 4), y_target=y)
        loss.backward()
        assert all(p.grad is not None and torch.isfinite(p.grad).all() for p in model.parameters())
        losses.append(loss.item())
    assert abs(losses[0] - losses[1]) <= 5e-3 * abs(losses[0])
