"""The C entry points that take whole layers refuse a pointer that is missing or off a 16-byte boundary before they
launch anything.  (No call here is one that a device would be given.)"""

import ctypes

import pytest

from ar_nanotabpfn_amd import _lib

AT = 0x10000  # never read: every call is refused
POINTERS = ("w_fo", "w_qkv", "w_o", "w_1", "b_1", "w_2", "b_2", "gamma1", "beta1", "gamma2", "beta2", "gamma3", "beta3", "k_cache", "v_cache")
F32, BF16 = 2, 0


def _stack(layer=None, value=None, **other):
    layers = (_lib.ArtabStackLayer * 3)()
    for i, one in enumerate(layers):
        for name in POINTERS:
            setattr(one, name, value if i == 2 and name == layer else AT)
    a = _lib.ArtabStackArgs(ctypes.addressof(layers), 3, 1, 32, 4, 128, 256, 0, 0, 0, 32, AT, AT, AT)
    for name, v in other.items():
        setattr(a, name, v)
    return a, layers


@pytest.mark.parametrize("dtype", [F32, BF16], ids=["f32", "bf16"])
def test_layer_stack_refuses_addresses_off_16_bytes(dtype):
    lib = _lib.load()
    import torch

    assert _lib.dtype_code(torch.float32 if dtype == F32 else torch.bfloat16) == dtype
    for name in POINTERS:
        a, keep = _stack(name, AT + 4)
        assert lib.artab_layer_stack(ctypes.byref(a), dtype, None) == _lib.ARTAB_ERR_BAD_STRIDE, name
    for name in ("x", "out", "scratch"):
        a, keep = _stack(**{name: AT + 8})
        assert lib.artab_layer_stack(ctypes.byref(a), dtype, None) == _lib.ARTAB_ERR_BAD_STRIDE, name


@pytest.mark.parametrize("dtype", [F32, BF16], ids=["f32", "bf16"])
def test_layer_stack_refuses_missing_pointers(dtype):
    lib = _lib.load()
    for name in POINTERS:
        if name == "b_2" or (name == "b_1" and dtype == BF16):
            continue  # may be NULL
        a, keep = _stack(name, None)
        assert lib.artab_layer_stack(ctypes.byref(a), dtype, None) == _lib.ARTAB_ERR_NULL_POINTER, name


def _train(bad=None, value=AT + 4, param=None):
    a = _lib.ArtabTrainArgs()
    a.B, a.R, a.H, a.D, a.F, a.n_layers = 1, 40, 4, 128, 256, 2
    a.context_len, a.buffer_len, a.attending_chunks, a.first_row = 16, 4, 1, 20
    params = (ctypes.c_void_p * 32)(*[AT] * 32)
    if param is not None:
        params[param] = value
    for name in ("x", "norm_gamma", "norm_beta", "saved", "z", "dz", "dx", "grads", "scratch"):
        setattr(a, name, value if name == bad else AT)
    a.params = ctypes.cast(params, ctypes.c_void_p)
    return a, params


def test_training_refuses_addresses_off_16_bytes():
    lib = _lib.load()
    calls = ((lib.artab_train_forward, ("x", "norm_gamma", "norm_beta", "saved", "z")),
             (lib.artab_train_backward, ("x", "norm_gamma", "norm_beta", "saved", "dz", "dx", "grads", "scratch")))
    for call, names in calls:
        for name in names:
            a, keep = _train(name)
            assert call(ctypes.byref(a), None) == _lib.ARTAB_ERR_BAD_STRIDE, name
        for i in range(32):
            a, keep = _train(param=i)
            assert call(ctypes.byref(a), None) == _lib.ARTAB_ERR_BAD_STRIDE, i
            a, keep = _train(param=i, value=None)
            assert call(ctypes.byref(a), None) == _lib.ARTAB_ERR_NULL_POINTER, i


def test_training_embedding_refuses_addresses_off_16_bytes():
    lib = _lib.load()
    names = ("x_context", "y_context", "x_buffer", "y_buffer", "x_target", "w_x", "b_x", "w_y", "b_y", "markers", "tokens", "out", "xy",
             "grads", "scratch")

    def args(bad):
        a = _lib.ArtabTrainEmbedArgs()
        a.B, a.n_context, a.n_buffer, a.n_target, a.feat, a.D = 1, 16, 4, 20, 2, 128
        for name in names:
            setattr(a, name, AT + 4 if name == bad else AT)
        return ctypes.byref(a)

    for name in ("w_x", "b_x", "w_y", "b_y", "markers", "tokens", "out", "xy"):
        assert lib.artab_train_embed(args(name), None) == _lib.ARTAB_ERR_BAD_STRIDE, name
    for name in ("out", "xy", "grads", "scratch"):
        assert lib.artab_train_embed_backward(args(name), None) == _lib.ARTAB_ERR_BAD_STRIDE, name
