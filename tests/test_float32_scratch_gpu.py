"""float32 context and decode calls use scratch memory of their own: two streams do not share any."""

import pytest
import torch

import ar_nanotabpfn_amd.attention_kernels as ak
from ar_nanotabpfn_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("native", [True, False], ids=["native", "python"])
def test_float32_calls_leave_the_shared_scratch_alone(device, monkeypatch, native):
    if not native:
        monkeypatch.setattr(ak, "_call", lambda *a: None)
    # few queries, many keys: the keys are dealt over workgroups, whose results pass through scratch memory
    B, H, Nc, D = 2, 4, 8192, 32
    assert _lib.load().artab_workspace_bytes(B, H, 2, Nc, D, _lib.dtype_code(torch.float32)) > 0
    g = torch.Generator().manual_seed(0)
    q, k, v = (torch.randn(*s, generator=g).to(device) for s in ((B, H, 2, D), (H, Nc, D), (H, Nc, D)))
    kb, vb = (torch.randn(B, H, 40, D, generator=g).to(device) for _ in range(2))
    with _lib.workspace_tag(4242):
        want = ak.context_attention(q, k, v), ak.decode_attention(q, k, v, kb, vb, 33)
        assert _lib.held_workspace(device) is None
    streams = [torch.cuda.Stream() for _ in range(2)]
    results = [[], []]
    for s in streams:
        s.wait_stream(torch.cuda.current_stream())
    for _ in range(50):
        for s, r in zip(streams, results):
            with torch.cuda.stream(s):
                scaled = q * (1 if s is streams[0] else -1)
                r.append((ak.context_attention(scaled, k, v)[0], ak.decode_attention(scaled, k, v, kb, vb, 33)))
    torch.cuda.synchronize()
    for c, d in results[0]:
        assert torch.equal(c, want[0][0]) and torch.equal(d, want[1])
    for c, d in results[1]:
        assert torch.equal(c, results[1][0][0]) and torch.equal(d, results[1][0][1])
