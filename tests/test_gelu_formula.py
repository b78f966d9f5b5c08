"""The formula of the kernels' gelu (``normal_tail`` in csrc/common.h): its constants, taken from the source and evaluated
in float32, against float64."""

import os
import re

import numpy as np
from scipy.special import erfc

SOURCE = open(os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ar_nanotabpfn_amd", "csrc", "common.h")).read()
F = np.float32


def _tail(x):
    body = SOURCE[SOURCE.index("float normal_tail("):]
    body = body[:body.index("return")]
    scale, *p = [F(v) for v in re.findall(r"(-?\d+\.\d{6,})f", body)]
    assert len(p) == 7
    t = F(1) / (scale * np.abs(x) + F(1))
    acc = np.full_like(t, p[0])
    for c in p[1:]:
        acc = (acc.astype(np.float64) * t + c).astype(F)  # fma
    e = np.exp2(((x * x).astype(F) * F(-0.5 * 1.4426950408889634)).astype(F).astype(np.float64)).astype(F)
    return acc * t * e


def test_gelu_is_as_good_as_its_rounding():
    x = np.linspace(-9.9, 9.9, 400001).astype(F)
    tail, d = _tail(x), x.astype(np.float64)
    true = 0.5 * d * erfc(-d / np.sqrt(2))
    # the polynomial 4.4e-7; float32's exponent x^2 / 2 log2 e < 128, rounded twice to half of 2^-17, times ln 2; p t e
    assert np.abs(tail.astype(np.float64) / (0.5 * erfc(np.abs(d) / np.sqrt(2))) - 1).max() <= 4.4e-7 + 2 * 2 ** -18 * 0.7 + 3e-7
    gelu = x * np.where(x > 0, F(1) - tail, tail)
    # half a unit in the last place from rounding to f16, and a hundredth of one from the formula
    unit = np.maximum(2.0 ** (np.floor(np.log2(np.abs(true) + 1e-300)) - 10), 2.0 ** -24)
    assert (np.abs(gelu.astype(np.float16).astype(np.float64) - true) / unit).max() <= 0.51
