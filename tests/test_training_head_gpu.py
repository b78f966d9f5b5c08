"""The mixture head of a training step and its loss on the device kernels, against the modules in float64."""

import copy
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def _problem(device, D, K, B, T):
    from ar_nanotabpfn_amd.model import MixtureGaussianHead

    torch.manual_seed(3)
    head = MixtureGaussianHead(D, 256, num_components=K)
    with torch.no_grad():
        for p in head.parameters():
            p.add_(0.05 * torch.randn_like(p))
        # deviations about 0.5, as a trained head's: a change of a raw output by e moves the gradient by about e / 0.5 of
        # itself.  (Fresh heads have deviations of 1 / (K - 1), and K - 1 times their roundings in every gradient.)
        head.std_bias.add_(math.log(math.expm1(0.5)) - head.std_bias.mean())
    z, y = torch.randn(B, T, D), 2 * torch.randn(B, T, 1)
    return head.to(device), z.to(device), y.to(device)


def _gradients(loss, z, head):
    return torch.autograd.grad(loss, [z, *head.parameters()])


def _modules_in(dtype, head, z, y, autocast=False):
    h = copy.deepcopy(head).to(dtype)
    z = z.detach().to(dtype).requires_grad_()
    with torch.autocast("cuda", torch.bfloat16, enabled=autocast):
        loss = h(z, y.to(dtype))[0]
    return loss, _gradients(loss, z, h)


def _kernels(head, z, y):
    from ar_nanotabpfn_amd.training import head_loss

    z = z.detach().requires_grad_()
    with torch.autocast("cuda", torch.bfloat16):
        loss = head_loss(head, z, y)
    assert loss is not None
    return loss, _gradients(loss, z, head)


def _loss_of(head_loss, head, z, y):
    z = z.detach().requires_grad_()
    with torch.autocast("cuda", torch.bfloat16):
        return head_loss(head, z, y), z, head


@pytest.mark.parametrize("D,K,B,T", [
    (128, 20, 3, 33),     # 60 raw outputs, a ragged last tile
    (128, 2, 1, 1), (256, 5, 2, 32),
    (128, 21, 5, 13), (256, 22, 1, 70),  # 63 and 66 outputs: the last of the narrow form, the first of the wide one
    (128, 42, 4, 50),     # the most
    (256, 20, 25, 999),   # several tiles to some workgroups, slices of the weight gradients
])
def test_loss_and_gradients(device, D, K, B, T):
    head, z, y = _problem(device, D, K, B, T)
    exact, exact_grads = _modules_in(torch.float64, head, z, y)
    auto, auto_grads = _modules_in(torch.float32, head, z, y, autocast=True)
    loss, grads = _kernels(head, z, y)
    # five roundings of at most 2^-9, of random sign, in raw outputs of the order of one, which enter with 1 / 0.5
    assert abs(loss.item() - exact.item()) <= 5 * 2.0 ** -9 * max(1.0, abs(exact.item()))
    # z, W_1, the hidden layer, W_2, the raw outputs' gradient are rounded as in the modules.  Both errors are those of the few
    # rows whose y lies far out, where a component's t^2 multiplies them, one draw of the roundings each: some ten such rows,
    # whose norms differ by a third from draw to draw; and a rounding where the modules happen to have none (1 or 2 rows)
    for got, ref, module in zip(grads, exact_grads, auto_grads):
        error, theirs = ((g.double() - ref).norm() for g in (got, module))
        assert error <= 1.5 * theirs + 2.0 ** -9 * ref.norm() + 1e-9, (tuple(got.shape), error.item(), theirs.item())
    if B * T >= 1000:  # the ordinary row is not further off than with the modules
        ours, theirs = (((g[0].double() - exact_grads[0]).norm(dim=2) / exact_grads[0].norm(dim=2)).median() for g in (grads, auto_grads))
        assert ours <= theirs


@pytest.mark.parametrize("case", ["far", "nan", "narrow", "inf"])
def test_unusual_values(device, case):
    head, z, y = _problem(device, 128, 5, 2, 40)
    if case == "far":      # likelihoods that underflow: the sums are taken behind the largest exponent
        y[0, 3] = 1e3
    elif case == "nan":
        y[1, 7] = float("nan")
    elif case == "narrow":  # deviations at both ends of their range, weights that vanish
        with torch.no_grad():
            head.std_bias[:2] = torch.tensor([-80.0, 90.0])
            head.weight_bias[3] = -300.0
    else:
        with torch.no_grad():
            head.weight_bias[3] = float("-inf")
    module, module_grads = _modules_in(torch.float32, head, z, y, autocast=True)
    loss, grads = _kernels(head, z, y)
    if case == "nan":
        assert loss.isnan() and module.isnan()
    else:
        assert loss.isfinite() and abs(loss.item() - module.item()) <= 2e-2 * abs(module.item())
    for got, ref in zip(grads, module_grads):
        assert torch.equal(got.isnan(), ref.isnan())
        if case != "nan":
            assert (got - ref).norm() <= 5e-2 * ref.norm() + 1e-6


def test_gradients_of_gradients(device):
    head, z, y = _problem(device, 128, 5, 2, 20)
    from ar_nanotabpfn_amd.training import head_loss

    out = []
    for run in (lambda z: head_loss(head, z, y), lambda z: head(z, y)[0]):
        z = z.detach().requires_grad_()
        with torch.autocast("cuda", torch.bfloat16):
            loss = run(z)
        (g,) = torch.autograd.grad(loss, head.head[0].weight, create_graph=True)
        out.append(torch.autograd.grad(g.square().sum(), z)[0])
    assert (out[0] - out[1]).norm() <= 2e-2 * out[1].norm()


def test_what_the_kernels_are_not_for(device):
    from ar_nanotabpfn_amd.training import head_loss

    head, z, y = _problem(device, 128, 43, 2, 20)
    z.requires_grad_()
    with torch.autocast("cuda", torch.bfloat16):
        assert head_loss(head, z, y) is None                      # 129 raw outputs
        head, *_ = _problem(device, 128, 5, 1, 1)
        assert head_loss(head, z, y.clone().requires_grad_()) is None
        assert head_loss(head, z[:, ::2], y[:, ::2]) is None
        assert head_loss(head, z, y.double()) is None
        head.head[2] = torch.nn.Linear(256, 15, bias=False, device=device)
        assert head_loss(head, z, y) is None and head(z, y)[0].isfinite()
        assert head_loss(head.half(), z, y) is None


def _through_the_model(device):
    """A training step's loss as a function of nothing, and its head."""
    import ar_nanotabpfn_amd.model as model_mod
    from ar_nanotabpfn_amd.attention import create_dense_mask, create_row_mask

    torch.manual_seed(1)
    model = model_mod.ARTabPFN(d_model=128, n_heads=4, n_layers=1, d_ff=256, num_features=2, buffer_size=4, num_components=5).to(device)
    mk = lambda *s: torch.randn(*s, generator=torch.Generator().manual_seed(2)).to(device)  # noqa: E731
    data, y = (mk(3, 17, 2), mk(3, 17), mk(3, 4, 2), mk(3, 4), mk(3, 12, 2)), mk(3, 12)
    masks = (create_dense_mask(1), create_row_mask(33, 17, 4))

    def loss():
        with torch.autocast("cuda", dtype=torch.bfloat16):
            return model(*data, *masks, y_target=y)
    return loss, model.head


def test_tangents_of_head_parameters(device):
    """Forward-mode differentiation in the head's parameters: along a direction, what the gradients give."""
    import torch.autograd.forward_ad as fwad

    loss, head = _through_the_model(device)
    bias = head.mean_bias
    (grad,) = torch.autograd.grad(loss(), bias)
    direction = torch.linspace(-1.0, 2.0, bias.numel(), device=device)
    with fwad.dual_level():
        del head.mean_bias
        head.mean_bias = fwad.make_dual(bias.detach(), direction)
        tangent = fwad.unpack_dual(loss()).tangent
    # (the modules' bf16 products here, the kernels' there: five roundings of at most 2^-9, twice)
    assert abs(float(tangent) - float(grad @ direction)) <= 2 * 5 * 2.0 ** -9 * float(grad.norm() * direction.norm())


def test_batched_gradients_of_head_parameters(device):
    loss, head = _through_the_model(device)
    out, params = loss(), list(head.parameters())
    want = torch.autograd.grad(out, params, retain_graph=True)
    scales = torch.tensor([1.0, -0.5, 3.0], device=device)
    got = torch.autograd.grad(out, params, grad_outputs=scales, is_grads_batched=True)
    for g, w in zip(got, want):  # (the modules' products here, the kernels' there, as above)
        assert g.shape == (3, *w.shape)
        assert float((g - scales.view(-1, *[1] * w.dim()) * w).norm()) <= 2 * 2 * 5 * 2.0 ** -9 * float((scales.norm() * w.norm()))


def test_targets_that_lie_anywhere_and_move_on(device):
    """The values are a table's last columns, at an odd address, and the program puts the next ones in their place before
    the backward pass (the modules keep no reference to them)."""
    from ar_nanotabpfn_amd.training import head_loss

    head, z, y = _problem(device, 128, 5, 1, 33)
    want = _gradients(*_loss_of(head_loss, head, z, y))
    table = torch.cat([torch.zeros(1, 5, 1, device=device), y], dim=1)
    mine = table[:, 5:]
    assert mine.is_contiguous() and mine.data_ptr() % 16
    args = _loss_of(head_loss, head, z, mine)
    table.fill_(float("nan"))
    for got, ref in zip(_gradients(*args), want):
        assert torch.equal(got, ref)
    mine.copy_(y)
    loss, z, _ = _loss_of(head_loss, head, z, mine)
    table.fill_(float("nan"))
    (got,) = torch.autograd.grad(loss, z, create_graph=True)  # (the modules' route, with the kept values)
    assert got.isfinite().all() and (got - want[0]).norm() <= 2 * 5 * 2.0 ** -9 * want[0].norm()
