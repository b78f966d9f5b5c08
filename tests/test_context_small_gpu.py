"""Context attention and prefill with few query rows in one launch, against float64 and the tiled route."""

import pytest
import torch

import ar_nanotabpfn_amd.attention_kernels as ak
from ar_nanotabpfn_amd import _lib

pytestmark = pytest.mark.gpu


def _reference(q, k, v):
    s = torch.matmul(q.double(), k.double().transpose(-1, -2).contiguous()) * q.shape[-1] ** -0.5
    return torch.matmul(s.softmax(-1), v.double().contiguous()), torch.logsumexp(s, -1)


def _check(dtype, got, tiled, ref):
    err = [((t.double() - ref).norm() / ref.norm()).item() for t in (got, tiled)]
    # u: unit roundoff of the model's type.  Both routes round the scaled queries (the same values), the
    # probabilities and the result to it; the probabilities are rounded at other scales (2^s against 2^(s - max)), which
    # moves the result by at most u of the mean of |v| they weight.
    u = 2.0 ** -9 if dtype == torch.bfloat16 else 2.0 ** -12
    assert err[0] <= err[1] + u, err
    # rounded queries move a score of deviation up to 4 by u 4 / sqrt(3); with the other two roundings under 4 u
    assert err[0] <= 4 * u, err


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [32, 64])
# the shortest context, ragged blocks, fewer blocks than wavefronts, the longest; ragged row tiles of one to eight
# heads, rows of several trajectories in a tile; a context of its own per trajectory; the most workgroups
@pytest.mark.parametrize("B,H,Lq,Nc,own", [(1, 1, 1, 64, False), (5, 3, 7, 97, False), (8, 8, 1, 512, False), (33, 8, 2, 1536, False),
                                           (3, 5, 33, 255, True), (7, 2, 1, 641, True), (1024, 8, 1, 300, False)])
def test_context(device, dtype, D, B, H, Lq, Nc, own):
    g = torch.Generator("cuda").manual_seed(Nc)
    q = torch.randn(B, Lq, H, D, generator=g, device=device).to(dtype).transpose(1, 2)  # strided, as projections are
    k, v = (torch.randn(*((B,) if own else ()), H, Nc + 2, D, generator=g, device=device).to(dtype)[..., :Nc, :] for _ in range(2))
    k[..., -1, :] *= 4  # a late maximum
    out, lse = ak.context_attention(q, k, v)
    with _lib.tuning(ARTAB_SMALL=0):
        tiled, _ = ak.context_attention(q, k, v)
    ref, ref_lse = _reference(q, k, v)
    _check(dtype, out, tiled, ref)
    # scores of up to 4 sqrt(D) in 16-bit queries: 2^-9 (bf16) of them
    assert (lse.double() - ref_lse).abs().max().item() < (0.1 if dtype == torch.bfloat16 else 0.02)


def test_context_not_finite(device):
    q = torch.randn(4, 4, 1, 64, device=device, dtype=torch.bfloat16)
    k, v = (torch.randn(4, 100, 64, device=device, dtype=torch.bfloat16) for _ in range(2))
    q[1, 2] = float("nan")
    v[3, 7, 5] = float("inf")
    out, lse = ak.context_attention(q, k, v)
    assert out[1, 2].isnan().all() and lse[1, 2].isnan().all()
    assert (out[[0, 2, 3]][:, :3]).isfinite().all() and lse[[0, 2, 3]].isfinite().all()
    assert (out[:, 3, 0, 5] == float("inf")).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,H,N,D,stored", [(1, 8, 1024, 32, 1), (1, 4, 65, 64, 1), (3, 5, 127, 32, 3), (3, 2, 200, 64, 1)])
def test_prefill(device, dtype, B, H, N, D, stored):
    g = torch.Generator("cuda").manual_seed(N)
    q, k, v = (torch.randn(B, N, H, D, generator=g, device=device).to(dtype).transpose(1, 2) for _ in range(3))
    caches = [torch.full((stored, H, N + 3, D) if B == stored else (H, N + 3, D), 7.0, device=device, dtype=dtype) for _ in range(2)]
    out = ak.prefill_attention(q, k, v, *caches)
    for c, t in zip(caches, (k, v)):
        assert torch.equal(c[..., :N, :], t if B == stored else t[0]) and bool((c[..., N:, :] == 7.0).all())
    with _lib.tuning(ARTAB_SMALL=0):
        tiled = ak.prefill_attention(q, k, v)
    _check(dtype, out, tiled, _reference(q, k, v)[0])
