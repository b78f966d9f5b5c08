"""The row attention's gradients with one workgroup per (batch entry, head): at the edges of its sizes, and just
beyond them, against the float32-arithmetic kernels (which the float64 oracle checks in test_row_mask_gpu.py)."""

import pytest
import torch

from tests.helpers import randn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize(
    "B,H,D,Nc,Nb,T,A",
    [
        (2, 2, 32, 1, 0, 1, 0),        # one key, one tile of rows for four groups
        (2, 2, 32, 31, 1, 0, 0),       # no targets: nothing to clear
        (3, 4, 32, 64, 32, 512, 8),    # the training configuration: targets that attend and targets that do not
        (1, 4, 32, 96, 32, 70, 1),     # all 128 keys, a ragged last tile
        (65, 4, 32, 33, 8, 100, 2),    # more pairs than compute units: two groups
        (20, 4, 32, 100, 29, 70, 2),   # 129 keys: eight wavefronts, the keys of a dQ piece dealt over two
        (20, 4, 32, 240, 16, 33, 2),   # all 256
        (8, 4, 32, 240, 16, 33, 2),    # as many keys, fewer pairs: the two launches
        (38, 4, 32, 230, 27, 90, 1),   # 257 keys: sixteen wavefronts, the keys of a dQ piece dealt over four
        (38, 4, 32, 500, 12, 20, 1),   # all 512
        (38, 4, 32, 500, 13, 20, 1),   # one more: the two launches
        (2, 3, 64, 65, 16, 65, 2),     # head_dim 64
        (38, 4, 64, 200, 56, 40, 0),
        (65, 4, 32, 240, 16, 33, 2),   # a second round of four pairs: the two launches   # all 256, no target attends
    ],
)
def test_gradients_match_the_float32_kernels(device, dtype, B, H, D, Nc, Nb, T, A):
    import ar_nanotabpfn_amd.attention_kernels as ak

    R = Nc + Nb + T
    # (the layout a layer's projections have: rows of all heads, with room between them)
    q, k, v, dout = (randn((B, R, H, D + 8), s, dtype, 0.8).to(device)[..., :D].transpose(1, 2) for s in (1, 2, 3, 4))
    out, lse = ak._row_mask_forward(q, k, v, Nc, Nb, A, True, want_lse=True)
    got = ak.row_mask_attention_backward(q, k, v, out, dout, lse, Nc, Nb, A)
    again = ak.row_mask_attention_backward(q, k, v, out, dout, lse, Nc, Nb, A)
    ref = ak.row_mask_attention_backward(q, k, v, out, dout, lse, Nc, Nb, A, use_triton=False)
    # the rounded queries, P, dS and the result: four roundings of at most half a unit each, independent of one another
    unit = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    for name, a, b, c in zip(("dq", "dk", "dv"), got, again, ref):
        assert torch.equal(a, b), name
        a, c = a.double(), c.double()
        if R > Nc + Nb and name != "dq":
            assert not a[:, :, Nc + Nb :].any(), name
        if not c.any():  # (one visible key: the softmax is constant)
            assert float(a.abs().max()) <= 2e-2, name
            continue
        assert float((a - c).norm()) <= 1.25 * unit * float(c.norm()) + 1e-3, name
        assert float((a - c).abs().max()) <= 2e-2 * max(1.0, float(c.abs().max())), name
