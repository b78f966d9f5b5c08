"""C++ errors inside the native calls arrive as Python exceptions.  On the CPU: tensors that claim to be on a device
that is not there, so that describing and allocating them fails (each case in a process of its own: an error that
is not converted ends it)."""

import subprocess
import sys

import pytest

_CASE = """
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
from ar_nanotabpfn_amd import _lib
_lib.load()
with FakeTensorMode():
    q, k = torch.empty(2, 4, 1, 32, device="cuda", dtype=torch.float32), torch.empty(4, 16, 32, device="cuda", dtype=torch.float32)
    b = torch.empty(2, 4, 3, 32, device="cuda", dtype=torch.float32)
try:
    print("returned", CALL)
except RuntimeError as err:
    print("raised", type(err).__name__)
"""


@pytest.mark.parametrize("call", ["_lib.native.context_attention(q, k, k, None, 0)",
                                  "_lib.native.decode_attention(q, k, k, b, b, 1, None, None, 0)"], ids=["context", "decode"])
def test_a_cpp_error_is_an_exception(call):
    code = _CASE.replace("CALL", call)
    done = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=300)
    assert done.returncode == 0 and done.stdout.startswith("raised"), (done.returncode, done.stdout, done.stderr[-2000:])


@pytest.mark.gpu
def test_no_memory_for_the_result(device):
    import torch

    import ar_nanotabpfn_amd.attention_kernels as ak

    # 2^18 x 16 x 512 x 128 floats from one row: a terabyte
    q = torch.zeros(1, 1, 1, 128, device=device).expand(2 ** 18, 16, 512, 128)
    k = torch.zeros(16, 8, 128, device=device)
    with pytest.raises(torch.OutOfMemoryError):
        ak.context_attention(q, k, k)
    assert ak.context_attention(q[:1, :, :1], k, k)[0].shape == (1, 16, 1, 128)
