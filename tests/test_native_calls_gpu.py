"""The native form of the small calls (csrc/native_calls.cpp): same results as the path behind it, and everything
that is not the plain case left to that path."""

import pytest
import torch

import ar_nanotabpfn_amd.attention_kernels as ak

pytestmark = pytest.mark.gpu


def _randn(device, dtype, *shape):
    g = torch.Generator().manual_seed(sum(shape))
    return torch.randn(*shape, generator=g).to(device, dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32], ids=["bf16", "f16", "f32"])
@pytest.mark.parametrize("own_context", [False, True], ids=["shared", "own"])
@pytest.mark.parametrize("Lq", [1, 2])
def test_native_calls_equal_the_python_path(device, monkeypatch, dtype, own_context, Lq):
    B, H, Nc, D, cap, n = 5, 4, 70, 32, 9, 6
    # (queries as a projection leaves them: heads inside a row)
    q = _randn(device, dtype, B, Lq, H, D).transpose(1, 2)
    k, v = (_randn(device, dtype, *((B,) if own_context else ()), H, Nc, D + i)[..., :D] for i in (0, 8))
    new = [_randn(device, dtype, B, H, 1, D) for _ in range(2)]
    results = []
    for native in (True, False):
        if not native:
            monkeypatch.setattr(ak, "_call", lambda *a: None)
        buf = [_randn(device, dtype, B, H, cap, D) for _ in range(2)]
        results.append([*ak.context_attention(q, k, v, 0.3), ak.decode_attention(q, k, v, *buf, n, *new), *buf,
                        ak.decode_attention(q, k, v, *buf, n)])
        assert not native or ak._call("context_attention", q, k, v, None, 0) is not None
        assert not native or ak._call("decode_attention", q, k, v, *buf, n, *new, 0) is not None
    for a, b in zip(*results):
        assert torch.equal(a, b) and a.stride() == b.stride()


def test_what_is_not_plain_raises_as_before(device, monkeypatch):
    q, k = _randn(device, torch.float16, 2, 4, 1, 32), _randn(device, torch.float16, 4, 16, 32)
    buf = _randn(device, torch.float16, 2, 4, 3, 32)
    cases = [
        (ValueError, "do not match q", lambda: ak.context_attention(q, k[:3], k[:3])),
        (ValueError, "do not match q", lambda: ak.context_attention(q, k[:, :, :16], k[:, :, :16])),
        (ValueError, "one dtype", lambda: ak.context_attention(q, k.float(), k.float())),
        (ValueError, "needs Nc >= 1", lambda: ak.context_attention(q, k[:, :0], k[:, :0])),
        (ValueError, "head_dim axis must be contiguous", lambda: ak.context_attention(q, k.transpose(1, 2).contiguous().transpose(1, 2), k)),
        (ValueError, "unsupported dtype", lambda: ak.context_attention(q.double(), k.double(), k.double())),
        (RuntimeError, "HIP device only", lambda: ak.context_attention(q.cpu(), k, k)),
        (ValueError, "capacity", lambda: ak.decode_attention(q, k, k, buf, buf, 4)),
        (ValueError, "capacity", lambda: ak.decode_attention(q, k, k, buf, buf, 3, q, q)),  # no room for the new row
        (ValueError, "must be given together", lambda: ak.decode_attention(q, k, k, buf, buf, 1, q)),
        (ValueError, "N=1 .target. or N=2", lambda: ak.decode_attention(q.expand(-1, -1, 3, -1), k, k, buf, buf, 1)),
        (ValueError, "negative buffer length", lambda: ak.decode_attention(q, k, k, buf, buf, -1)),
    ]
    for error, message, call in cases:
        with pytest.raises(error, match=message) as with_native:
            call()
        with monkeypatch.context() as m, pytest.raises(error, match=message) as without:
            m.setattr(ak, "_call", lambda *a: None)
            call()
        assert type(with_native.value) is type(without.value) is error and str(with_native.value) == str(without.value)
