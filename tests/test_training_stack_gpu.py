"""``ARTabPFN.forward`` under bfloat16 autocast on the fused training kernels (embedding, layer stack) against the
same model as PyTorch modules around the device row attention: loss and every parameter gradient."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def only_modules(monkeypatch):
    """Neither embedding nor stack nor head on the training kernels from here on."""
    import ar_nanotabpfn_amd.model as model_mod

    monkeypatch.setattr(model_mod, "layer_stack_supported", lambda *a: False)
    monkeypatch.setattr(model_mod, "embed_rows", lambda *a: None)
    monkeypatch.setattr(model_mod, "head_loss", lambda *a: None)


# edges: one row tile and one row past it, no whole 64-row piece for the weight gradients, one layer, one buffer row,
# one feature, both widths and head dims, tokens that take no part, the row attention's backward pass in one launch and in two
@pytest.mark.parametrize("D,H,L,B,Nc,Nb,Nt,feat,tokens", [
    (128, 4, 1, 1, 16, 1, 15, 1, 1), (128, 4, 2, 3, 17, 4, 12, 2, 6), (128, 2, 2, 5, 40, 8, 100, 3, 8),
    (256, 8, 2, 2, 33, 5, 61, 10, 32), (256, 4, 1, 7, 64, 16, 129, 2, 16),
    (128, 4, 1, 3, 300, 32, 64, 2, 32),
    # a run of this file and the other training tests once left the GPU faulted, and later a run of all device tests; both had
    # a weight-gradient kernel with twice the bytes on their way, which has been taken out both times.  Which test it was is
    # not known, and no access out of range has been found.  Of the first run's tests these sizes (and the 515 tiles of the
    # many-tiles test) have not run since with the attention's query tiles they take now.
    pytest.param(128, 4, 1, 33, 300, 32, 512, 2, 32, marks=pytest.mark.skip(reason="part of a run that faulted, cause not shown"))])
def test_fused_training_equals_modules(device, monkeypatch, D, H, L, B, Nc, Nb, Nt, feat, tokens):
    import ar_nanotabpfn_amd.model as model_mod
    from ar_nanotabpfn_amd.attention import create_dense_mask, create_row_mask

    torch.manual_seed(1)
    model = model_mod.ARTabPFN(d_model=D, n_heads=H, n_layers=L, d_ff=256, num_features=feat, buffer_size=tokens, num_components=5)
    with torch.no_grad():
        for name, p in model.named_parameters():
            if "norm" in name or name.endswith("bias"):
                p.add_(0.1 * torch.randn_like(p))
    model = model.to(device)
    g = torch.Generator().manual_seed(2)
    mk = lambda *s: torch.randn(*s, generator=g).to(device)  # noqa: E731
    data = (mk(B, Nc, feat), mk(B, Nc), mk(B, Nb, feat), mk(B, Nb), mk(B, Nt, feat))
    y = mk(B, Nt)
    masks = (create_dense_mask(1), create_row_mask(Nc + Nb + Nt, Nc, Nb))

    def step():
        model.zero_grad(set_to_none=True)
        with torch.autocast("cuda", dtype=torch.bfloat16):
            loss = model(*data, *masks, y_target=y)
        loss.backward()
        return loss.item(), {n: p.grad for n, p in model.named_parameters()}

    taken = {}
    for name in ("embed_rows", "layer_stack", "head_loss"):
        monkeypatch.setattr(model_mod, name, lambda *a, f=getattr(model_mod, name), name=name: taken.setdefault(name, f(*a)))
    loss, grads = step()
    assert len(taken) == 3 and all(t is not None for t in taken.values()), "the fused route was not taken"
    taken.clear()
    loss2, grads2 = step()
    assert loss == loss2 and all(torch.equal(grads[n], grads2[n]) for n in grads)
    only_modules(monkeypatch)
    ref_loss, ref = step()
    assert abs(loss - ref_loss) <= 5e-3 * abs(ref_loss)
    for n, r in ref.items():
        assert grads[n].shape == r.shape and torch.isfinite(grads[n]).all()
        # (both sides round every product operand to eight bits: a per cent or two for the smallest gradients)
        assert float((grads[n] - r).norm()) <= 4e-2 * float(r.norm()) + 1e-6, n


@pytest.mark.parametrize("D,H,L,B,Nc,Nb,Nt", [(128, 4, 4, 8, 40, 8, 64), (256, 8, 2, 5, 33, 5, 61)])
def test_both_routes_against_float32(device, monkeypatch, D, H, L, B, Nc, Nb, Nt):
    """The gradients of both routes under autocast against those of the modules in float32: the fused kernels, which keep
    the residual stream and the norms in float32, are not further off than the modules."""
    import ar_nanotabpfn_amd.model as model_mod
    from ar_nanotabpfn_amd.attention import create_dense_mask, create_row_mask

    torch.manual_seed(1)
    model = model_mod.ARTabPFN(d_model=D, n_heads=H, n_layers=L, d_ff=256, num_features=2, buffer_size=Nb, num_components=5).to(device)
    g = torch.Generator().manual_seed(2)
    mk = lambda *s: torch.randn(*s, generator=g).to(device)  # noqa: E731
    data, y = (mk(B, Nc, 2), mk(B, Nc), mk(B, Nb, 2), mk(B, Nb), mk(B, Nt, 2)), mk(B, Nt)
    masks = (create_dense_mask(1), create_row_mask(Nc + Nb + Nt, Nc, Nb))

    def step(autocast):
        model.zero_grad(set_to_none=True)
        with torch.autocast("cuda", dtype=torch.bfloat16, enabled=autocast):
            loss = model(*data, *masks, y_target=y)
        loss.backward()
        return loss.detach().double(), {n: p.grad.double() for n, p in model.named_parameters()}

    fused_loss, fused = step(True)
    only_modules(monkeypatch)
    module_loss, modules = step(True)
    true_loss, true = step(False)

    def error(a, names):
        return float(torch.stack([(a[n] - true[n]).norm() ** 2 for n in names]).sum().sqrt()
                     / torch.stack([true[n].norm() ** 2 for n in names]).sum().sqrt())

    groups = {"all": list(true), "layers": [n for n in true if "layers" in n], "embedding": [n for n in true if "embed" in n or n == "ar_tokens"]}
    report = {g: (error(fused, names), error(modules, names)) for g, names in groups.items()}
    print(report, (fused_loss - true_loss).item(), (module_loss - true_loss).item())
    # products of bf16 operands on both sides: 2^-9 each, some tens of them
    assert all(f <= m and f <= 2e-2 for f, m in report.values()), report
    assert abs(fused_loss - true_loss) <= 2e-3 * abs(true_loss)
