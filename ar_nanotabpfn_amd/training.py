"""The layer stack of a training step on the device kernels (``artab_train_forward`` / ``_backward``): what
``TwoStageTransformer.forward`` and the final norm record under bfloat16 autocast (model.py:100-147, :317-369;
train.py:289-300), as one differentiable call; the row embeddings in front of it and the mixture head with its loss
behind it as one each.

The residual stream, the norms and every sum stay float32; products take bfloat16 operands, as autocast's do.
"""

from __future__ import annotations

import ctypes

import torch
from torch import Tensor, nn
from torch.autograd import forward_ad

from . import _lib
from . import attention_kernels as ak
from .attention import RowMask

__all__ = ["embed_rows", "layer_stack_supported", "layer_stack", "head_loss"]

# A program that has put callables of its own in their place gets the modules, which call them.
_attention_calls = (ak.row_mask_attention, ak.row_mask_attention_backward)


def _layer_params(layer):
    """The parameters of a layer in the order of ``artab_train_args.params``."""
    mods = layer._modules
    af, ar, ff = mods["attn_features"]._modules, mods["attn_rows"]._modules, mods["ff"]._modules
    one, two = ff["0"]._parameters, ff["2"]._parameters
    n1, n2, n3 = mods["norm1"]._parameters, mods["norm2"]._parameters, mods["norm3"]._parameters
    return (af["v_proj"]._parameters["weight"], af["out_proj"]._parameters["weight"], ar["q_proj"]._parameters["weight"],
            ar["k_proj"]._parameters["weight"], ar["v_proj"]._parameters["weight"], ar["out_proj"]._parameters["weight"],
            one["weight"], one["bias"], two["weight"], two["bias"], n1["weight"], n1["bias"], n2["weight"], n2["bias"],
            n3["weight"], n3["bias"])


def _shapes(D: int, F: int):
    """Their sizes."""
    return ((D, D),) * 6 + ((F, D), (F,), (D, F), (D,)) + ((D,),) * 6


def _args(backbone, B: int, R: int, mask: RowMask, first_row: int) -> "_lib.ArtabTrainArgs":
    layer = backbone.layers[0]
    a = _lib.ArtabTrainArgs()
    a.B, a.R, a.H, a.D, a.F = B, R, layer.attn_rows.n_heads, backbone.d_model, layer.ff[0].out_features
    a.n_layers, a.first_row = len(backbone.layers), first_row
    a.context_len, a.buffer_len, a.attending_chunks = mask.context_len, mask.buffer_len, mask.attending_chunks
    a.eps1, a.eps2, a.eps3, a.eps_out = layer.norm1.eps, layer.norm2.eps, layer.norm3.eps, backbone.norm.eps
    return a


def layer_stack_supported(backbone, x: Tensor, mask, first_row: int) -> bool:
    """True when ``layer_stack`` computes what the modules would: gradients are being recorded under bfloat16
    autocast, float32 parameters, widths the kernels are built for, equal layers."""
    if not (x.is_cuda and x.dtype == torch.float32 and torch.is_grad_enabled() and isinstance(mask, RowMask)
            and torch.is_autocast_enabled("cuda") and torch.get_autocast_dtype("cuda") == torch.bfloat16
            and (ak.row_mask_attention, ak.row_mask_attention_backward) == _attention_calls):
        return False
    layers = list(backbone.layers)
    if not layers or x.shape[1] != mask.num_rows or x.shape[2] != backbone.d_model:
        return False
    first = layers[0]
    D, F, norm = x.shape[2], first.ff[0].out_features, backbone.norm
    shapes, heads = _shapes(D, F), first.attn_rows.n_heads
    constants = [getattr(first, n).eps for n in ("norm1", "norm2", "norm3")]

    def same(layer):
        af, ar = layer._modules["attn_features"], layer._modules["attn_rows"]
        projections = [*af._modules.values(), *ar._modules.values()]
        unused = (af._modules["q_proj"]._parameters["weight"], af._modules["k_proj"]._parameters["weight"])
        return (ar.n_heads == heads and ar.head_dim * heads == D and [layer._modules[n].eps for n in ("norm1", "norm2", "norm3")] == constants
                and _f32(x.device, _layer_params(layer), shapes) and all(m._parameters["bias"] is None for m in projections)
                and all(p.dtype == torch.float32 and p.device == x.device for p in unused))

    return (all(same(layer) for layer in layers) and _f32(x.device, (norm.weight, norm.bias), ((D,), (D,)))
            and (x.requires_grad or any(p.requires_grad for p in backbone.parameters()))
            and _lib.load().artab_train_saved_bytes(ctypes.byref(_args(backbone, x.shape[0], x.shape[1], mask, first_row))) > 0)


def _f32(device, tensors, shapes) -> bool:
    """Float32 tensors of these sizes, as the kernels read them (16-byte pieces, no strides)."""
    return all(t is not None and type(t) in (Tensor, nn.Parameter) and t.dtype == torch.float32 and t.device == device and t.shape == s
               and t.is_contiguous() and t.data_ptr() % 16 == 0 for t, s in zip(tensors, shapes))


def _pieces(t: Tensor) -> Tensor:
    """``t`` without strides, at an address that 16-byte loads can take."""
    t = t.contiguous()
    return t.clone() if t.data_ptr() % 16 else t


class _Embed(torch.autograd.Function):
    @staticmethod
    def forward(ctx, xc, yc, xb, yb, xt, w_x, b_x, w_y, b_y, markers, tokens):
        a = _lib.ArtabTrainEmbedArgs()
        B, a.feat, a.D = xc.shape[0], xc.shape[2], markers.shape[1]
        a.B, a.n_context, a.n_buffer, a.n_target = B, xc.shape[1], xb.shape[1], xt.shape[1]
        R = a.n_context + a.n_buffer + a.n_target
        out = torch.empty((B, R, a.D), device=xc.device, dtype=torch.float32)
        xy = torch.empty((B, R, 2), device=xc.device, dtype=torch.float32)
        for name, t in zip(("x_context", "y_context", "x_buffer", "y_buffer", "x_target", "w_x", "b_x", "w_y", "b_y", "markers",
                            "tokens", "out", "xy"), (xc, yc, xb, yb, xt, w_x, b_x, w_y, b_y, markers, tokens, out, xy)):
            setattr(a, name, t.data_ptr())
        _lib.check(_lib.load().artab_train_embed(ctypes.byref(a), _lib.current_stream(xc.device)))
        # (through save_for_backward: freed when the backward pass is done, seen by saved-tensor hooks)
        ctx.save_for_backward(xy)
        ctx.args, ctx.shapes = a, (w_x.shape, w_y.shape, tokens.shape)
        return out

    @staticmethod
    @torch.autograd.function.once_differentiable
    def backward(ctx, dx):
        lib, a = _lib.load(), _lib.ArtabTrainEmbedArgs.from_buffer_copy(ctx.args)
        (xy,) = ctx.saved_tensors
        dx, xy = _pieces(dx), _pieces(xy)
        D, n = a.D, ctx.shapes[2][0]
        grads = torch.empty((7 + n) * D, device=dx.device, dtype=torch.float32)
        if n > a.n_buffer:  # tokens behind the buffer rows take no part
            grads[(7 + a.n_buffer) * D :].zero_()
        scratch = torch.empty(lib.artab_train_embed_scratch_bytes(ctypes.byref(a)), device=dx.device, dtype=torch.uint8)
        a.out, a.xy, a.grads, a.scratch = dx.data_ptr(), xy.data_ptr(), grads.data_ptr(), scratch.data_ptr()
        _lib.check(lib.artab_train_embed_backward(ctypes.byref(a), _lib.current_stream(dx.device)))
        w_x, b_x, w_y, b_y, markers, tokens = grads.split((D, D, D, D, 3 * D, n * D))
        return (None,) * 5 + (w_x.view(ctx.shapes[0]), b_x, w_y.view(ctx.shapes[1]), b_y, markers.view(3, D), tokens.view(n, D))


def embed_rows(model, x_context, y_context, x_buffer, y_buffer, x_target):
    """The embedded rows ``[B,R,D]`` of ``ARTabPFN.forward``, or None where the kernel does not apply (the data
    itself wants gradients, types or widths it is not built for)."""
    e = model.embedder
    params = (e.x_embed.weight, e.x_embed.bias, e.y_embed.weight, e.y_embed.bias, e.marker_embed.weight, model.ar_tokens)
    data = [t.contiguous() for t in (x_context, y_context, x_buffer, y_buffer, x_target)]
    xs, ys = data[0::2], data[1::2]
    D, (B, feat) = model.d_model, (xs[0].shape[0], xs[0].shape[-1])
    if not (torch.is_autocast_enabled("cuda") and torch.get_autocast_dtype("cuda") == torch.bfloat16 and D in (128, 256)
            and xs[0].is_cuda and all(t.dim() == 3 and t.shape[0] == B and t.shape[2] == feat for t in xs)
            and all(tuple(y.shape) in ((B, x.shape[1]), (B, x.shape[1], 1)) for x, y in zip(xs, ys))
            and not any(t.requires_grad for t in data) and any(p.requires_grad for p in params)
            and xs[0].shape[1] >= 1 and xs[2].shape[1] >= 1 and xs[1].shape[1] <= model.ar_tokens.shape[0]
            and _f32(xs[0].device, data, [t.shape for t in data])
            and _f32(xs[0].device, params, ((D, 1), (D,), (D, 1), (D,), (3, D), (model.ar_tokens.shape[0], D)))
            and B >= 1 and feat >= 1 and B * sum(x.shape[1] for x in xs) < 2 ** 30):
        return None
    return _Embed.apply(*data, *params)


def _set_pointers(a, x: Tensor, params, saved: Tensor):
    """The tensors of a call into its arguments; returns what the arguments point at."""
    n = 16 * a.n_layers
    pointers = (ctypes.c_void_p * n)(*(p.data_ptr() for p in params[:n]))
    a.x, a.params, a.saved = x.data_ptr(), ctypes.cast(pointers, ctypes.c_void_p), saved.data_ptr()
    a.norm_gamma, a.norm_beta = params[n].data_ptr(), params[n + 1].data_ptr()
    return pointers


class _LayerStack(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, backbone, mask, first_row, *params):
        lib = _lib.load()
        B, R, D = x.shape
        x = _pieces(x)
        a = _args(backbone, B, R, mask, first_row)
        saved = torch.empty(lib.artab_train_saved_bytes(ctypes.byref(a)), device=x.device, dtype=torch.uint8)
        z = torch.empty((B, R - first_row, D), device=x.device, dtype=torch.float32)
        ctx.args = _lib.ArtabTrainArgs.from_buffer_copy(a)  # (sizes and constants only)
        pointers = _set_pointers(a, x, params, saved)  # noqa: F841  (alive until the call)
        a.z = z.data_ptr()
        _lib.check(lib.artab_train_forward(ctypes.byref(a), _lib.current_stream(x.device)))
        ctx.save_for_backward(x, saved, *params)
        return z

    @staticmethod
    @torch.autograd.function.once_differentiable
    def backward(ctx, dz):
        lib = _lib.load()
        x, saved, *params = ctx.saved_tensors  # (raises if one of them was changed in place since)
        a = _lib.ArtabTrainArgs.from_buffer_copy(ctx.args)
        D, F, L = a.D, a.F, a.n_layers
        # parameters whose data was exchanged since are read where they now are: they have to be of the same form
        if not (_f32(x.device, (x,), ((a.B, a.R, D),)) and saved.data_ptr() % 16 == 0
                and _f32(x.device, params, _shapes(D, F) * L + ((D,), (D,)))):
            raise RuntimeError("a parameter of the layer stack has another size or type than in the forward pass")
        dz = _pieces(dz.float())
        pointers = _set_pointers(a, x, params, saved)  # noqa: F841  (alive until the call)
        scratch = torch.empty(lib.artab_train_scratch_bytes(ctypes.byref(a)), device=x.device, dtype=torch.uint8)
        dx = torch.empty_like(x)
        sizes = (D * D,) * 5 + (F * D, D * F) + (D,) * 5 + (F,) + (D,) * 2 + (D * D,) * 2
        total = sum(sizes)
        grads = torch.empty(L * total + 2 * D, device=x.device, dtype=torch.float32)
        a.dz, a.dx, a.grads, a.scratch = dz.data_ptr(), dx.data_ptr(), grads.data_ptr(), scratch.data_ptr()
        _lib.check(lib.artab_train_backward(ctypes.byref(a), _lib.current_stream(x.device)))
        out = []
        for i in range(L):
            q, k, v, _, o, w1, w2, g3, b3, bias2, g2, b2, bias1, g1, b1, f_out, f_v = grads[i * total : (i + 1) * total].split(sizes)
            square = lambda t: t.view(D, D)  # noqa: E731
            out += [square(f_v), square(f_out), square(q), square(k), square(v), square(o), w1.view(F, D), bias1, w2.view(D, F), bias2,
                    g1, b1, g2, b2, g3, b3]
        out += [grads[L * total : L * total + D], grads[L * total + D :]]
        return (dx, None, None, None, *out)


def layer_stack(backbone, x: Tensor, mask: RowMask, first_row: int) -> Tensor:
    """``backbone`` on the rows ``x [B,R,D]`` under the training row mask: the final norm's output of rows
    ``first_row`` and on, ``[B, R - first_row, D]``, differentiable in ``x`` and every parameter that takes part.
    The feature attention's q and k projections do not (one key per query: the softmax weight is 1)."""
    params = [p for layer in backbone.layers for p in _layer_params(layer)]
    return _LayerStack.apply(x, backbone, mask, first_row, *params, backbone.norm.weight, backbone.norm.bias)


class _HeadLoss(torch.autograd.Function):
    @staticmethod
    def forward(ctx, z, y, head, *params):
        lib = _lib.load()
        a = _lib.ArtabTrainHeadArgs()
        a.rows, a.D, a.F, a.K, a.std_min = z.shape[0] * z.shape[1], z.shape[2], params[0].shape[0], params[4].shape[0], head.std_min
        saved = torch.empty(lib.artab_train_head_saved_bytes(ctypes.byref(a)), device=z.device, dtype=torch.uint8)
        loss = torch.empty((), device=z.device, dtype=torch.float32)
        ctx.args, ctx.head = _lib.ArtabTrainHeadArgs.from_buffer_copy(a), head  # (sizes and constants only)
        _head_pointers(a, z, y, params, saved)
        a.loss = loss.data_ptr()
        _lib.check(lib.artab_train_head_forward(ctypes.byref(a), _lib.current_stream(z.device)))
        ctx.save_for_backward(z, saved, *params)
        return loss

    @staticmethod
    def backward(ctx, dloss):
        lib = _lib.load()
        z, saved, *params = ctx.saved_tensors  # (raises if one of them was changed in place since)
        create_graph = torch.is_grad_enabled()
        transformed = _transformed(dloss, z, *params)
        if create_graph or transformed:  # gradients that can be differentiated again, or many at once
            wanted = [t for t in (z, *params) if t.requires_grad]
            y = saved[: 4 * ctx.args.rows].view(torch.float32).view(*z.shape[:2], 1)  # (the kernels' copy)
            # (in float32 under a transform: it makes batched products of the modules' products, their right operands transposed
            # views, and those of bfloat16 have faulted the device)
            with torch.enable_grad(), torch.autocast("cuda", torch.bfloat16, enabled=not transformed):
                loss = torch.func.functional_call(ctx.head, dict(zip(_HEAD_PARAMETERS, params)), (z, y))[0]
            grads = iter(torch.autograd.grad(loss, wanted, dloss, create_graph=create_graph))
            dz, *dparams = (next(grads) if t.requires_grad else None for t in (z, *params))
            return (dz, None, None, *dparams)
        a = _lib.ArtabTrainHeadArgs.from_buffer_copy(ctx.args)
        D, F, K = a.D, a.F, a.K
        if not (_f32(z.device, (z,), (z.shape,)) and z.numel() == a.rows * D and saved.data_ptr() % 16 == 0
                and _f32(z.device, params, _head_shapes(D, F, K))):
            raise RuntimeError("a parameter of the head has another size or type than in the forward pass")
        dloss = dloss.float().contiguous()
        _head_pointers(a, z, None, params, saved)
        scratch = torch.empty(lib.artab_train_head_scratch_bytes(ctypes.byref(a)), device=z.device, dtype=torch.uint8)
        dz = torch.empty_like(z)
        grads = torch.empty(F * D + 128 * F + F + 128, device=z.device, dtype=torch.float32)
        a.dloss, a.dz, a.grads, a.scratch = dloss.data_ptr(), dz.data_ptr(), grads.data_ptr(), scratch.data_ptr()
        _lib.check(lib.artab_train_head_backward(ctypes.byref(a), _lib.current_stream(z.device)))
        w1, w2, b1, raw = grads.split((F * D, 128 * F, F, 128))
        per_component = raw[: 3 * K].view(K, 3).t().contiguous()  # a bias added behind b_2 has b_2's gradient
        return (dz, None, None, w1.view(F, D), b1, w2[: 3 * K * F].view(3 * K, F), raw[: 3 * K], *per_component)


def _transformed(*tensors) -> bool:
    """Whether a transform is at work (``vmap`` and its kin), or one of the tensors stands for many (batched gradients) or
    has a tangent."""
    if torch._C._are_functorch_transforms_active() or not all(map(torch._C._has_storage, tensors)):
        return True
    # (outside of every dual level there are no tangents)
    return forward_ad._current_level >= 0 and any(forward_ad.unpack_dual(t).tangent is not None for t in tensors)


_HEAD_PARAMETERS = ("head.0.weight", "head.0.bias", "head.2.weight", "head.2.bias", "mean_bias", "std_bias", "weight_bias")


def _head_shapes(D: int, F: int, K: int):
    return ((F, D), (F,), (3 * K, F), (3 * K,), (K,), (K,), (K,))


def _head_pointers(a, z: Tensor, y, params, saved: Tensor):
    for name, t in zip(("z", "y", "w1", "b1", "w2", "b2", "mean_bias", "std_bias", "weight_bias", "saved"), (z, y, *params, saved)):
        setattr(a, name, None if t is None else t.data_ptr())


def head_loss(head, z: Tensor, y: Tensor):
    """The loss of ``MixtureGaussianHead.forward(z, y)`` for ``z [B,T,D]``, ``y [B,T,1]`` under bfloat16 autocast,
    differentiable in ``z`` and the head's parameters, or None where the kernels do not apply (the data itself wants
    gradients, types or sizes they are not built for, tangents and transforms)."""
    one, two = head.head[0], head.head[2]
    params = (one.weight, one.bias, two.weight, two.bias, head.mean_bias, head.std_bias, head.weight_bias)
    F, K = one.out_features, head.num_components
    if not (torch.is_autocast_enabled("cuda") and torch.get_autocast_dtype("cuda") == torch.bfloat16 and torch.is_grad_enabled()
            and all(p is not None for p in params)  # (a Linear without a bias)
            and z.is_cuda and z.dtype == torch.float32 and z.dim() == 3 and tuple(y.shape) == (z.shape[0], z.shape[1], 1)
            and not y.requires_grad and head.dim_y == 1 and isinstance(K, int) and isinstance(head.std_min, float)
            and z.shape[2] in (128, 256) and F == 256 and 1 <= 3 * K <= 128 and 1 <= z.shape[0] * z.shape[1] < 2 ** 30
            and (z.requires_grad or any(p.requires_grad for p in params)) and not _transformed(z, y, *params)):
        return None
    y = y.contiguous()
    if not (type(z) is Tensor and z.is_contiguous() and z.data_ptr() % 16 == 0 and type(y) is Tensor and y.dtype == torch.float32 and y.device == z.device and _f32(z.device, params, _head_shapes(z.shape[2], F, K))):
        return None
    return _HeadLoss.apply(z, y, head, *params)
