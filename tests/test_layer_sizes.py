"""Weights and vectors of another size are refused before a layer launch.  (On the CPU: the check comes before anything
that needs a device.)"""

import pytest
import torch
from torch import nn

from ar_nanotabpfn_amd import glue

D, F = 128, 256


def _packed(n, k):
    return torch.zeros(n // 32, k // 16, 64, 8, dtype=torch.bfloat16)


def _args():
    norm = nn.LayerNorm(D)
    x = torch.zeros(4, D, dtype=torch.bfloat16)
    pre = {"w_fo": _packed(D, D), "norm1": norm, "w_qkv": _packed(3 * D, D)}
    post = {"w_o": _packed(D, D), "norm2": norm, "w_1": _packed(F, D), "b_1": torch.zeros(F), "w_2": _packed(D, F), "b_2": torch.zeros(D),
            "norm3": norm}
    return x, pre, post


WRONG = [("w_fo", _packed(256, 256)), ("w_qkv", _packed(2 * D, D)), ("norm1", nn.LayerNorm(64)), ("w_o", _packed(D, 64)),
         ("w_1", _packed(F, 64)), ("w_2", _packed(D, 128)), ("b_1", torch.zeros(128)), ("b_2", torch.zeros(64)), ("norm2", nn.LayerNorm(256)),
         ("norm3", nn.LayerNorm(64))]


@pytest.mark.parametrize("name,value", WRONG, ids=[n for n, _ in WRONG])
def test_other_sizes_are_refused(name, value):
    x, pre, post = _args()
    wrong = pre if name in pre else post
    wrong[name] = value
    match = "in a layer of width 128"
    if name in pre:
        with pytest.raises(RuntimeError, match=match):
            glue.layer_pre(x, **pre)
    else:
        with pytest.raises(RuntimeError, match=match):
            glue.layer_post(x, x, **post)
    with pytest.raises(RuntimeError, match=match):
        glue.layer_post_pre(x, x, *post.values(), next_w_fo=pre["w_fo"], next_norm1=pre["norm1"], next_w_qkv=pre["w_qkv"])
