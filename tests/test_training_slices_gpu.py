"""The weight gradients' tiles and slices of rows: one row beside and on the edges of tiles of 64 and 128 and of slices of
256, slices that get no rows, for the head's launch and for those of a layer's front, back and both."""

import pytest
import torch

from .test_training_head_gpu import _problem

# Written for tiles of 128 rows, which were in the tree when a run of the device tests faulted and have been taken out since.
pytestmark = [pytest.mark.gpu, pytest.mark.skip(reason="part of a run that faulted, cause not shown")]


# a ragged and a whole tile, one row in a second one; one row in a second slice, in a third; 43 of 64 slices with rows
@pytest.mark.parametrize("D,rows", [(128, 127), (128, 128), (256, 129), (128, 257), (256, 513), (128, 16385)])
def test_head(device, D, rows):
    """A sum over rows is the sum of the sums over parts of them, of at most one tile each."""
    from ar_nanotabpfn_amd.training import head_loss

    head, z, y = _problem(device, D, 5, 1, rows)

    def sums(z, y):  # of the rows' gradients, not their mean: the same values for a row whatever is beside it
        with torch.autocast("cuda", torch.bfloat16):
            loss = head_loss(head, z.requires_grad_(), y)
        return torch.autograd.grad(loss, list(head.parameters()), torch.full_like(loss, z.shape[1]))

    parts = [sums(z[:, i:i + 96].clone(), y[:, i:i + 96].clone()) for i in range(0, rows, 96)]
    for whole, *part in zip(sums(z.clone(), y.clone()), *parts):
        exact = torch.stack([p.double() for p in part]).sum(0)
        # the same bfloat16 products in float32 sums of another order: 2^-24 of the terms, whose sum may cancel
        size = torch.stack([p.double().abs() for p in part]).sum(0).norm()
        assert (whole.double() - exact).norm() <= 1e-5 * size, tuple(whole.shape)


# rows of an entry: a whole tile, one row more, one row in a second slice; all of them: ragged slices of two and three
@pytest.mark.parametrize("D,B,Nc,Nb,Nt", [(128, 3, 56, 8, 64), (128, 3, 100, 8, 149), (256, 3, 56, 8, 65), (256, 5, 100, 8, 85)])
def test_stack(device, D, B, Nc, Nb, Nt):
    """The gradient of a batch is the sum of its entries' gradients."""
    from ar_nanotabpfn_amd.attention import create_dense_mask, create_row_mask
    from ar_nanotabpfn_amd.model import ARTabPFN

    torch.manual_seed(4)
    model = ARTabPFN(d_model=D, n_heads=D // 32, n_layers=2, d_ff=256, num_features=2, buffer_size=8, num_components=5).to(device)
    g = torch.Generator().manual_seed(5)
    mk = lambda *s: torch.randn(*s, generator=g).to(device)  # noqa: E731
    data = [mk(B, Nc, 2), mk(B, Nc), mk(B, Nb, 2), mk(B, Nb), mk(B, Nt, 2), mk(B, Nt)]
    masks = create_dense_mask(1), create_row_mask(Nc + Nb + Nt, Nc, Nb)

    def sums(data):
        with torch.autocast("cuda", torch.bfloat16):
            loss = model(*data[:5], *masks, y_target=data[5])
        return torch.autograd.grad(loss, list(model.parameters()), torch.full_like(loss, data[0].shape[0]))

    entries = [sums([t[b:b + 1].clone() for t in data]) for b in range(B)]
    for whole, *part in zip(sums(data), *entries):
        # (the attention deals its keys by the size of the call: roundings to bfloat16, 2^-9, that fall the other way)
        size = torch.stack([p.abs() for p in part]).sum(0).norm()
        assert (whole - torch.stack(part).sum(0)).norm() <= 2.0 ** -9 * 4 * size, tuple(whole.shape)
