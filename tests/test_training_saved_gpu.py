"""What the fused training kernels keep between forward and backward goes through autograd's saved tensors: it is
freed with them, seen by their hooks, and the backward pass reads parameters where they are at that time."""

import pytest
import torch
from torch.utils.checkpoint import checkpoint

import ar_nanotabpfn_amd.model as model_mod
from ar_nanotabpfn_amd.attention import create_dense_mask, create_row_mask

pytestmark = pytest.mark.gpu


def _setup(device, B=16, Nt=300):
    torch.manual_seed(1)
    model = model_mod.ARTabPFN(d_model=128, n_heads=4, n_layers=3, d_ff=256, num_features=2, buffer_size=4, num_components=5).to(device)
    g = torch.Generator().manual_seed(2)
    mk = lambda *s: torch.randn(*s, generator=g).to(device)  # noqa: E731
    data, y = (mk(B, 17, 2), mk(B, 17), mk(B, 4, 2), mk(B, 4), mk(B, Nt, 2)), mk(B, Nt)
    masks = (create_dense_mask(1), create_row_mask(21 + Nt, 17, 4))

    def loss():
        with torch.autocast("cuda", dtype=torch.bfloat16):
            return model(*data, *masks, y_target=y)
    return model, loss


def _grads(model):
    out = [p.grad.clone() for n, p in model.named_parameters() if not n.startswith("head")]  # (the head's sums are a library's)
    model.zero_grad(set_to_none=True)
    return out


def _equal(a, b):
    return len(a) == len(b) and all(torch.equal(x, y) for x, y in zip(a, b))


def test_kept_memory_is_freed_by_the_backward_pass(device):
    model, loss = _setup(device)
    loss().backward()  # (library workspaces, gradients)
    model.zero_grad(set_to_none=False)
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    out = loss()
    kept = torch.cuda.memory_allocated() - before
    out.backward()
    left = torch.cuda.memory_allocated() - before
    # the embedding and the layers keep 42 MB of it; what is left is the loss
    assert kept > 42e6 and left < 1e5, (kept, left)


def test_saved_tensor_hooks_see_all_of_it(device):
    model, loss = _setup(device)
    loss().backward()
    want = _grads(model)
    before = torch.cuda.memory_allocated()
    with torch.autograd.graph.save_on_cpu():
        out = loss()
    assert torch.cuda.memory_allocated() - before < 10e6  # (42 MB otherwise)
    out.backward()
    assert _equal(_grads(model), want)


def test_checkpoint(device):
    model, loss = _setup(device)
    loss().backward()
    want = _grads(model)
    for reentrant in (False, True):
        if reentrant:
            x = torch.zeros(1, device=device, requires_grad=True)
            checkpoint(lambda x: loss() + 0 * x.sum(), x, use_reentrant=True).backward()
        else:
            checkpoint(loss, use_reentrant=False).backward()
        assert _equal(_grads(model), want)


def test_backward_twice(device):
    model, loss = _setup(device)
    out = loss()
    out.backward(retain_graph=True)
    want = _grads(model)
    out.backward()
    assert _equal(_grads(model), want)
    with pytest.raises(RuntimeError):
        out.backward()


def test_parameter_data_exchanged_before_the_backward_pass(device):
    model, loss = _setup(device)
    loss().backward()
    want = _grads(model)
    out = loss()
    for p in model.parameters():
        p.data = p.data.clone()
    # the memory of the old values, taken by somebody else
    others = [torch.full_like(p, float("nan")) for p in model.parameters()]
    out.backward()
    assert _equal(_grads(model), want) and others
    # of another size: refused before anything is launched
    out = loss()
    w = model.backbone.layers[1].ff[0].weight
    w.data = w.data[:128].clone()
    with pytest.raises(RuntimeError, match="another size"):
        out.backward()
    # written to in place: refused by autograd, as ever
    model, loss = _setup(device)
    out = loss()
    with torch.no_grad():
        model.backbone.layers[0].norm1.weight.mul_(2)
    with pytest.raises(RuntimeError, match="inplace"):
        out.backward()
