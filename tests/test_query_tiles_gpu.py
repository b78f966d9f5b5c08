"""Unsplit attention (prefill, teacher forcing, the training row mask) at calls that take query tiles of 256, 128 and 64
rows, on both sides of where the choice changes, against the float32-arithmetic kernels."""

import pytest
import torch

from tests.helpers import max_abs, out_tol, randn, to_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,H,D,Nc,rows", [
    (64, 4, 32, 96, 608),    # 128: less rounding up, few keys
    (64, 4, 32, 700, 256),   # 256: long keys, nothing rounded up
    (64, 4, 32, 700, 257),   # 128: 512 rows against 384
    (8, 4, 32, 40, 30),      # 64: few rows, few keys
    (8, 4, 32, 301, 64),     # 128: few rows, more keys
    (4, 8, 32, 257, 500),    # 128: 64 would fill the chip no better over this many keys
    (4, 8, 32, 256, 500),    # 64
    (16, 8, 64, 200, 516),   # head_dim 64: 128
    (2, 8, 64, 100, 33),     # 64
    (1, 8, 32, 1500, 1999),  # 256: 64 workgroups, long keys
    (2, 4, 32, 900, 1025),   # 128: 40 workgroups of 256 rows, fewer than they are worth there
    (4, 8, 64, 500, 300),    # head_dim 64, half the chip at 128 rows: 64 in bf16
    (8, 8, 64, 400, 440),    # 448 rows against 512: 64 in bf16
])
def test_unsplit_calls(device, dtype, B, H, D, Nc, rows):
    import ar_nanotabpfn_amd.attention_kernels as ak

    half = max(1, rows // 2)
    q, kb, vb = (randn((B, H, n, D), s, dtype, 0.7).to(device) for s, n in ((1, 2 * half), (2, half), (3, half)))
    kc, vc = (randn((B, H, Nc, D), s, dtype, 0.7).to(device) for s in (4, 5))
    calls = [lambda fast: ak.teacher_forcing_attention(q, kc, vc, kb, vb, half, use_triton=fast)]
    x = randn((B, rows, 3, H, D), 6, dtype, 0.7).to(device)
    xq, xk, xv = (x[:, :, i].transpose(1, 2) for i in range(3))
    calls.append(lambda fast: ak.prefill_attention(xq, xk, xv, use_triton=fast))
    if rows > Nc + 8:
        calls.append(lambda fast: ak.row_mask_attention(xq, xk, xv, Nc, 8, 2, use_triton=fast))
    for call in calls:
        assert max_abs(to_np(call(True)), to_np(call(False))) <= 2 * out_tol(dtype)  # (each within out_tol of the exact result)
