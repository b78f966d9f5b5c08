"""float32 attention on the matrix cores against float64 products: every form (one tile per wavefront, a tile's
keys dealt over a workgroup, over several workgroups), at the edges of its 32-key blocks and 16-row tiles."""

import pytest
import torch

import ar_nanotabpfn_amd.attention_kernels as ak

pytestmark = pytest.mark.gpu


def _randn(device, *shape, seed=0):
    g = torch.Generator().manual_seed(sum(shape) + seed)
    return torch.randn(*shape, generator=g).to(device)


def _reference(q, k, v, mask=None):
    q, k, v = (t.cpu().double() for t in (q, k, v))
    s = q @ k.transpose(-1, -2).contiguous() * q.shape[-1] ** -0.5
    if mask is not None:
        s = s.masked_fill(~mask.cpu(), float("-inf"))
    return torch.softmax(s, -1) @ v, torch.logsumexp(s, -1)


def _close(a, b):
    assert float((a.cpu().double() - b).abs().max()) <= 2e-5, float((a.cpu().double() - b).abs().max())


@pytest.mark.parametrize("own", [False, True], ids=["shared", "own"])
@pytest.mark.parametrize("B,H,Lq,Nc,D", [
    (1, 1, 1, 1, 32), (3, 4, 5, 31, 32), (2, 3, 17, 33, 64), (1, 2, 16, 4097, 32), (4, 9, 33, 64, 128), (5, 8, 7, 1500, 64),
    (64, 8, 130, 95, 32), (40, 8, 300, 65, 64), (70, 9, 60, 40, 128)])
def test_context(device, own, B, H, Lq, Nc, D):
    q = _randn(device, B, Lq, H, D).transpose(1, 2)
    k, v = (_randn(device, *((B,) if own else ()), H, Nc, D, seed=i) for i in (1, 2))
    out, lse = ak.context_attention(q, k, v)
    ref, ref_lse = _reference(q, k, v)
    _close(out, ref)
    _close(lse, ref_lse)


@pytest.mark.parametrize("own", [False, True], ids=["shared", "own"])
@pytest.mark.parametrize("new", [False, True], ids=["stored", "new"])
@pytest.mark.parametrize("B,H,Lq,Nc,D,n", [
    (1, 1, 1, 1, 32, 0), (7, 4, 2, 33, 64, 1), (9, 3, 2, 4500, 32, 32), (33, 8, 1, 100, 128, 31), (70, 8, 2, 64, 32, 65),
    (1100, 32, 2, 40, 32, 3)])
def test_decode(device, own, new, B, H, Lq, Nc, D, n):
    q = _randn(device, B, Lq, H, D).transpose(1, 2)
    k, v = (_randn(device, *((B,) if own else ()), H, Nc, D, seed=i) for i in (1, 2))
    kb, vb = (_randn(device, B, H, n + 2, D, seed=i) for i in (3, 4))
    kn, vn = (_randn(device, B, H, 1, D, seed=i) if new else None for i in (5, 6))
    want_k, want_v = kb.clone(), vb.clone()
    if new:
        want_k[:, :, n:n + 1], want_v[:, :, n:n + 1] = kn, vn
    m = n + int(new)
    out = ak.decode_attention(q, k, v, kb, vb, n, kn, vn)
    full = [torch.cat([c.expand(B, -1, -1, -1), w[:, :, :m]], 2) for c, w in ((k, want_k), (v, want_v))]
    _close(out, _reference(q, *full)[0])
    assert torch.equal(kb, want_k) and torch.equal(vb, want_v)


@pytest.mark.parametrize("B,H,Nc,Nt,D", [(1, 2, 1, 1, 32), (3, 4, 33, 17, 64), (16, 8, 333, 45, 32), (40, 9, 31, 80, 128)])
def test_teacher_forcing_and_prefill(device, B, H, Nc, Nt, D):
    q = _randn(device, B, 2 * Nt, H, D).transpose(1, 2)
    k, v = (_randn(device, H, Nc, D, seed=i) for i in (1, 2))
    kb, vb = (_randn(device, B, H, Nt, D, seed=i) for i in (3, 4))
    i, j = torch.arange(2 * Nt, device=device)[:, None], torch.arange(Nt, device=device)[None]
    seen = torch.where(i < Nt, j <= i, j < i - Nt)
    mask = torch.cat([torch.ones(2 * Nt, Nc, dtype=torch.bool, device=device), seen], 1)
    full = [torch.cat([c.expand(B, -1, -1, -1), w], 2) for c, w in ((k, kb), (v, vb))]
    out, lse = ak.teacher_forcing_attention(q, k, v, kb, vb, Nt, return_lse=True)
    ref, ref_lse = _reference(q, *full, mask)
    _close(out, ref)
    _close(lse, ref_lse)
    # prefill: the targets' rows as a context of their own, its keys and values written to the cache
    cache = [torch.zeros(B, H, Nt + 1, D, device=device) for _ in range(2)]
    out = ak.prefill_attention(q[:, :, :Nt], kb, vb, *cache)
    _close(out, _reference(q[:, :, :Nt], kb, vb)[0])
    for c, w in zip(cache, (kb, vb)):
        assert torch.equal(c[:, :, :Nt], w) and not c[:, :, Nt:].any()


@pytest.mark.parametrize("B,H,Nc,Nb,Nt,D", [(2, 3, 17, 4, 24, 32), (9, 4, 70, 33, 70, 64)])
def test_row_mask(device, B, H, Nc, Nb, Nt, D):
    R, attend = Nc + Nb + Nt, Nt // (2 * Nb)
    q, k, v = (_randn(device, B, H, R, D, seed=i) for i in range(3))
    from ar_nanotabpfn_amd.attention import RowMask

    mask = RowMask(R, Nc, Nb, attend).dense().to(device)
    _close(ak.row_mask_attention(q, k, v, Nc, Nb, attend), _reference(q, k, v, mask)[0])
