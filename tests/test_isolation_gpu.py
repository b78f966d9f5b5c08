"""A value that is not finite stays with the rows that see it: other trajectories of a call, and rows whose mask
hides the key, give bit for bit what they give without it."""

import math

import pytest
import torch

import ar_nanotabpfn_amd.attention_kernels as ak

pytestmark = pytest.mark.gpu

BAD = [math.nan, math.inf]


def _randn(device, *shape, seed=0):
    g = torch.Generator().manual_seed(sum(shape) + seed)
    return torch.randn(*shape, generator=g).to(device)


# a trajectory in the middle of a block of 16 columns, at its edge, in a second block and in a second tile; a
# buffer of one row, of a whole block of 32 and of one row more; every form of the kernel (heads of 128; keys
# dealt over workgroups at 4500 rows; a tile per wavefront at 1100 x 32)
@pytest.mark.parametrize("bad", BAD, ids=["nan", "inf"])
@pytest.mark.parametrize("where", ["stored", "new"])
@pytest.mark.parametrize("B,H,Lq,Nc,D,n,at", [
    (9, 4, 2, 33, 32, 1, 3), (9, 4, 1, 64, 64, 33, 8), (40, 3, 2, 4500, 32, 32, 7), (21, 8, 2, 100, 128, 31, 16),
    (33, 4, 1, 40, 64, 32, 31), (1100, 32, 2, 40, 32, 3, 17)])
def test_decode_float32(device, bad, where, B, H, Lq, Nc, D, n, at):
    q = _randn(device, B, Lq, H, D).transpose(1, 2)
    k, v = (_randn(device, H, Nc, D, seed=i) for i in (1, 2))
    outs = []
    for value in (None, bad):
        kb, vb = (_randn(device, B, H, n + 1, D, seed=i) for i in (3, 4))
        kn, vn = (_randn(device, B, H, 1, D, seed=i) for i in (5, 6))
        if value is not None:
            (vb if where == "stored" else vn)[at, :, 0, D // 2] = value
        outs.append(ak.decode_attention(q, k, v, kb, vb, n, kn, vn))
    clean, got = outs
    others = torch.arange(B, device=device) != at
    assert torch.equal(got[others], clean[others])
    # the trajectory itself: the dimension that holds it, and no other
    wrong = ~torch.isfinite(got[at])
    assert wrong[..., D // 2].all() and int(wrong.sum()) == H * Lq


@pytest.mark.parametrize("bad", BAD, ids=["nan", "inf"])
@pytest.mark.parametrize("B,H,Nc,Nt,D,row", [(2, 3, 33, 17, 64, 16), (4, 8, 333, 45, 32, 5), (40, 9, 31, 80, 128, 40)])
def test_teacher_forcing_float32(device, bad, B, H, Nc, Nt, D, row):
    q = _randn(device, B, 2 * Nt, H, D).transpose(1, 2)
    k, v = (_randn(device, H, Nc, D, seed=i) for i in (1, 2))
    outs = []
    for value in (None, bad):
        kb, vb = (_randn(device, B, H, Nt, D, seed=i) for i in (3, 4))
        if value is not None:
            vb[1, :, row] = value
        outs.append(ak.teacher_forcing_attention(q, k, v, kb, vb, Nt))
    clean, got = outs
    i = torch.arange(2 * Nt, device=device)
    sees = torch.where(i < Nt, i >= row, i - Nt > row)
    assert torch.equal(got[1][:, ~sees], clean[1][:, ~sees]) and not torch.isfinite(got[1][:, sees]).any()
    assert torch.equal(got[0], clean[0]) and torch.equal(got[2:], clean[2:])


@pytest.mark.parametrize("bad", BAD, ids=["nan", "inf"])
def test_row_mask_float32(device, bad):
    from ar_nanotabpfn_amd.attention import RowMask

    B, H, Nc, Nb, Nt, D, row = 3, 4, 70, 33, 70, 64, 81
    R, attend = Nc + Nb + Nt, Nt // (2 * Nb)
    q, k, v = (_randn(device, B, H, R, D, seed=i) for i in range(3))
    clean = ak.row_mask_attention(q, k, v, Nc, Nb, attend)
    v[1, :, row] = bad
    got = ak.row_mask_attention(q, k, v, Nc, Nb, attend)
    sees = RowMask(R, Nc, Nb, attend).dense().to(device)[:, row]
    assert torch.equal(got[1][:, ~sees], clean[1][:, ~sees]) and not torch.isfinite(got[1][:, sees]).any()
    assert torch.equal(got[0], clean[0]) and torch.equal(got[2], clean[2])
