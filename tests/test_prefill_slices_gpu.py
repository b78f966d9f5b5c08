"""Prefill with its keys dealt over several workgroups against float64 and against the unsliced launch."""

import pytest
import torch

import ar_nanotabpfn_amd.attention_kernels as ak
from ar_nanotabpfn_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
# first sizes that are sliced, ragged last slices and tiles, one key past a slice of 128, several tables
@pytest.mark.parametrize("B,H,Nc,forced", [(1, 4, 4096, 0), (1, 8, 5001, 0), (2, 8, 2049, 0), (1, 3, 257, 3), (2, 8, 129, 2),
                                           (1, 8, 1000, 7), (3, 5, 640, 2)])
def test_sliced_prefill(dtype, B, H, Nc, forced):
    g = torch.Generator("cuda").manual_seed(Nc)
    q, k, v = (torch.randn(B, Nc, H, 32, generator=g, device="cuda").to(dtype).transpose(1, 2) for _ in range(3))
    kc, vc = (torch.full((B, H, Nc + 3, 32), 7.0, device="cuda", dtype=dtype) for _ in range(2))
    if not forced:
        assert _lib.load().artab_prefill_workspace_bytes(B, H, Nc, 32, _lib.dtype_code(dtype)) > 0
    # float64 is taken of the rows on both sides of every boundary of tiles and of the ends
    rows = sorted({r for t in range(0, Nc, 256) for r in (t, t + 1, t + 127, t + 255) if r < Nc} | {Nc - 1})
    s = torch.matmul(q[:, :, rows].double(), k.double().transpose(-1, -2).contiguous()) * 32 ** -0.5
    ref = torch.matmul(s.softmax(-1), v.double().contiguous())

    def error(slices):
        with _lib.tuning(ARTAB_SPLIT=slices, ARTAB_SMALL=0):
            out = ak.prefill_attention(q, k, v, kc, vc)
        return ((out[:, :, rows].double() - ref).norm() / ref.norm()).item()

    e_one, e_many = error(1), error(forced)
    # the merge is float32: one rounding of the result, as without slices
    assert e_many <= 1.05 * e_one + 1e-5, (e_many, e_one)
    assert e_many <= (4e-3 if dtype == torch.bfloat16 else 6e-4)
    for c, t in ((kc, k), (vc, v)):
        assert torch.equal(c[:, :, :Nc], t) and bool((c[:, :, Nc:] == 7.0).all())
