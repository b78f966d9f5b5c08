"""A prefill or teacher-forced pass through the layer stack as one call of the library (``artab_layer_stack``).

A layer is two launches of 15 to 70 us; issued one by one from Python they cost about 100 us of host time, which
is what such passes waited for (12 layers against 5001 rows: 1.2 ms of host time, 0.9 ms of kernels)."""

from __future__ import annotations

import ctypes
from typing import Optional

import torch
from torch import Tensor

from . import _lib
from . import attention_kernels as ak
from .live import Methods, Prepared, Sources, capturing
from .model import TwoStageTransformerLayer

__all__ = ["LAYER_METHODS", "LayerStack"]

# A program that has put callables of its own in their place gets the layer-by-layer form, which calls them.
LAYER_METHODS = Methods(TwoStageTransformerLayer, "fused_weights", "feature_stage", "qkv_heads", "packed_weights", "_fusable", "fused_for",
                        "pre_attention", "finish", "finish_then_pre", "feed_forward")
_attention_calls = (ak.prefill_attention, ak.teacher_forcing_attention, ak.hybrid_teacher_forcing_attention)


def _small_vectors(layer):
    """Parameters that enter unpacked, in the order of ``artab_stack_layer``, the weights that are packed, and the
    constants."""
    mods = layer._modules
    feat, rows, ff = mods["attn_features"]._modules, mods["attn_rows"]._modules, mods["ff"]._modules
    p1, p2 = ff["0"]._parameters, ff["2"]._parameters
    norms = mods["norm1"], mods["norm2"], mods["norm3"]
    n1, n2, n3 = (n._parameters for n in norms)
    return ((p1["bias"], p2["bias"], n1["weight"], n1["bias"], n2["weight"], n2["bias"], n3["weight"], n3["bias"]),
            (feat["v_proj"]._parameters["weight"], feat["out_proj"]._parameters["weight"], rows["q_proj"]._parameters["weight"],
             rows["k_proj"]._parameters["weight"], rows["v_proj"]._parameters["weight"], rows["out_proj"]._parameters["weight"],
             p1["weight"], p2["weight"]),
            (*(n.eps for n in norms), mods["attn_rows"].n_heads))


def _pack_f32(w: Tensor) -> Tensor:
    w = w.detach().contiguous()
    if w.data_ptr() % 16:
        w = w.clone()
    packed = torch.empty_like(w)
    _lib.check(_lib.load().artab_pack_stack_weight_float(w.data_ptr(), packed.data_ptr(), *w.shape, _lib.current_stream(w.device)))
    return packed


def _covered(layer, x: Tensor) -> bool:
    """Whether the call has kernels for this layer's widths and type (``artab_layer_stack``)."""
    if x.dtype == torch.float32:
        return x.shape[-1] in (128, 256, 512) and layer.ff[0].out_features == 256
    return layer.fused_for(x)


class LayerStack:
    """What a pass reads of the layers, collected again whenever a parameter is another tensor or has been
    written to, or a constant is another number; each call looks at all of them."""

    def __init__(self):
        self._sources = self._key = self._layers = self._prepared = None

    def _collect(self, layers, x: Tensor) -> bool:
        """Bring ``self._layers`` up to date; False where the layers are not of the form the call takes."""
        try:
            params = [_small_vectors(layer) for layer in layers]
        except (AttributeError, KeyError):
            return False
        tensors = [p for vectors, weights, _ in params for ps in (vectors, weights) for p in ps]
        if any(p is None for p in tensors):
            return False
        key = (x.dtype, x.device, *[constants for _, _, constants in params])
        if key == self._key and self._sources.unchanged(tensors):
            return self._layers is not None
        if capturing(x.device):  # (what a recording packs exists when it is replayed)
            return False
        self._key, self._sources, self._layers, self._prepared = key, Sources(tensors), None, None
        first = layers[0]
        D, F = x.shape[-1], first.ff[0].out_features
        for layer, (vectors, weights, _) in zip(layers, params):
            sizes = ((F,), (D,)) + ((D,),) * 6 + ((D, D),) * 6 + ((F, D), (D, F))
            if not (layer.attn_rows.n_heads == first.attn_rows.n_heads
                    and all(p.dtype == x.dtype and p.device == x.device and p.is_contiguous() and tuple(p.shape) == s
                            for p, s in zip(vectors + weights, sizes))
                    and all(p.data_ptr() % 16 == 0 for p in vectors)):
                return False
        array, keep = (_lib.ArtabStackLayer * len(layers))(), []
        for a, layer, (v, w, constants) in zip(array, layers, params):
            if x.dtype == torch.float32:
                packed = tuple(_pack_f32(p) for p in (*layer.fused_weights(), *w[5:]))
            else:
                packed = layer.packed_weights()
            a.w_fo, a.w_qkv, a.w_o, a.w_1, a.w_2 = (t.data_ptr() for t in packed)
            a.b_1, a.b_2, a.gamma1, a.beta1, a.gamma2, a.beta2, a.gamma3, a.beta3 = (t.data_ptr() for t in v)
            a.eps1, a.eps2, a.eps3 = constants[:3]
            keep += [*packed, *v]
        self._layers, self._prepared = array, Prepared(keep)
        return True

    @staticmethod
    def applies(layers, shape, dtype, device) -> bool:
        """Whether passes of such rows ``[B,N,D]`` through these layers have kernels and stand for what the layers do."""
        if not (device.type == "cuda" and layers and shape.numel() and (ak.prefill_attention, ak.teacher_forcing_attention,
                                                                        ak.hybrid_teacher_forcing_attention) == _attention_calls
                and LAYER_METHODS.of(*layers)):
            return False
        rows, D = layers[0].attn_rows, shape[-1]
        return rows.head_dim in (32, 64, 128) and rows.n_heads * rows.head_dim == D and _covered(layers[0], torch.empty((0, D), dtype=dtype, device=device))

    def _ready(self, layers, x: Tensor, caches, need: int) -> bool:
        """Whether the library takes passes of ``x [B,N,D]`` through ``layers`` with caches of at least ``need`` rows; their
        weights and caches are then in place."""
        if not self.applies(layers, x.shape, x.dtype, x.device):
            return False
        first = layers[0]
        k0 = caches[0][0]
        H, Dh, rows = first.attn_rows.n_heads, first.attn_rows.head_dim, k0.shape[-2]
        shape = (x.shape[0], H, rows, Dh) if k0.dim() == 4 else (H, rows, Dh)
        if not (rows >= need
                and all(t.shape == shape and t.dtype == x.dtype and t.device == x.device and t.is_contiguous() and t.data_ptr() % 16 == 0
                        for c in caches for t in c)
                and self._collect(layers, x)):
            return False
        for a, (k, v) in zip(self._layers, caches):
            a.k_cache, a.v_cache = k.data_ptr(), v.data_ptr()
        return True

    def _args(self, layers, x: Tensor, caches, num_targets: int, context_len: int, out: Optional[Tensor]):
        first, k0 = layers[0], caches[0][0]
        B, N, D = x.shape
        return _lib.ArtabStackArgs(ctypes.addressof(self._layers), len(layers), B, N, first.attn_rows.n_heads, D,
                                   first.ff[0].out_features, num_targets, context_len, int(k0.dim() == 4), k0.shape[-2], x.data_ptr(),
                                   None if out is None else out.data_ptr(), None)

    def __call__(self, layers, x: Tensor, caches, num_targets: int = 0, context_len: int = 0) -> Optional[Tensor]:
        """``x [B,N,D]`` through ``layers``; ``caches``: ``(k, v)`` of every layer, ``[H,R,Dh]`` or ``[B,H,R,Dh]``.
        ``num_targets`` 0: prefill; else teacher forcing against the first ``context_len`` cached rows.  None, with
        nothing done, where the call does not apply."""
        N, own = x.shape[1], caches[0][0].dim() == 4
        if (num_targets and context_len <= 0) or not self._ready(layers, x, caches, N if num_targets == 0 else context_len + (N if own else 0)):
            return None
        x = _pieces(x)
        self._prepared.use()
        lib, code = _lib.load(), _lib.dtype_code(x.dtype)
        out = torch.empty_like(x)
        args = self._args(layers, x, caches, num_targets, context_len, out)
        scratch = torch.empty(lib.artab_layer_stack_scratch_bytes(ctypes.byref(args), code), device=x.device, dtype=torch.uint8)
        args.scratch = scratch.data_ptr()
        _lib.check(lib.artab_layer_stack(ctypes.byref(args), code, _lib.current_stream(x.device)))
        return out

    def context(self, layers, x: Tensor, caches, targets: Optional[Tensor] = None):
        """A prefill of ``x [B,Nc,D]`` for the caches alone, and with ``targets [B',2 Nt,D]`` the teacher-forced pass over them
        beside it.  True or that pass's output; None, with nothing done, where the call does not apply."""
        N, own = x.shape[1], caches[0][0].dim() == 4
        both = targets is not None
        if both and not (targets.dtype == x.dtype and targets.device == x.device and targets.numel() and targets.shape[1] % 2 == 0
                         and x.shape[0] == (targets.shape[0] if own else 1)):
            return None
        if not self._ready(layers, x, caches, N + (targets.shape[1] if both and own else 0)):
            return None
        x = _pieces(x)
        self._prepared.use()
        lib, code, stream = _lib.load(), _lib.dtype_code(x.dtype), _lib.current_stream(x.device)
        args, second, out = self._args(layers, x, caches, 0, 0, None), None, True
        if both:
            targets = _pieces(targets)
            out = torch.empty_like(targets)
            second = ctypes.byref(self._args(layers, targets, caches, targets.shape[1] // 2, N, out))
        scratch = torch.empty(lib.artab_layer_stack_context_scratch_bytes(ctypes.byref(args), second, code), device=x.device,
                              dtype=torch.uint8)
        args.scratch = scratch.data_ptr()
        _lib.check(lib.artab_layer_stack_context(ctypes.byref(args), second, code, stream))
        return out


def _pieces(x: Tensor) -> Tensor:
    x = x.contiguous()
    return x.clone() if x.data_ptr() % 16 else x
