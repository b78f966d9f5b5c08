"""The float32 layer kernel at its tile heights (4, 8 and 16 rows, by how many rows there are per compute unit): the
edges of the tiles and of the rule, against the library's products around the same attention."""

import pytest
import torch

from ar_nanotabpfn_amd.inference import ARTabPFNPredictor
from ar_nanotabpfn_amd.model import ARTabPFN

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [128, 256, 512])
# rows per compute unit that a launch has, and rows beyond: one row, a ragged tile of 4, the last launch in tiles of 4, the
# first and the last in tiles of 8, the first in tiles of 16
@pytest.mark.parametrize("per_unit,more", [(0, 1), (0, 7), (4, 0), (4, 1), (8, -3), (8, 1)])
def test_layers_of_few_rows(device, monkeypatch, D, per_unit, more):
    rows = per_unit * torch.cuda.get_device_properties(device).multi_processor_count + more
    torch.manual_seed(rows)
    model = ARTabPFN(d_model=D, n_heads=D // 32, n_layers=2, d_ff=256, num_features=2).to(device).eval()
    g = torch.Generator().manual_seed(rows)
    x, y = torch.randn(1, rows, 2, generator=g).to(device), torch.randn(1, rows, generator=g).to(device)

    def run(one_call):
        p = ARTabPFNPredictor.from_trained_model(model, backend="shared_context")
        stack, taken = p._stack_pass, []
        monkeypatch.setattr(p, "_stack_pass", lambda *a: taken.append(stack(*a) if one_call else None) or taken[-1])
        p.init_kv_cache(1, 1, x.device, x.dtype)
        p.prefill_context(x, y)
        assert len(taken) == 1 and (taken[0] is not None) == one_call
        return [getattr(layer, n).clone() for layer in model.backbone.layers for n in ("k_ctx_cache", "v_ctx_cache")]

    # Sums of up to 512 float32 products in another order: each rounds at 2^-24 of its terms; two layers of five
    # products and three norms, whose gain is of order one, stay under 1e-5 of the result's size.  The largest row by
    # itself as well: a tile's last rows must not borrow from their neighbours.
    for a, b in zip(run(True), run(False)):
        a, b = a.double(), b.double()
        assert ((a - b).norm() / b.norm()).item() < 1e-5
        by_row = (a - b).norm(dim=-1) / b.norm(dim=-1)
        assert by_row.max().item() < 1e-4
