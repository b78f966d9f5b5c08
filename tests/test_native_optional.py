"""The native call module is an aid, not a condition: without it, or with one built for another torch, the library
still loads and the calls take their Python form."""

import importlib
import types

import pytest

from ar_nanotabpfn_amd import _lib
from ar_nanotabpfn_amd import attention_kernels as ak


def _missing(name, package=None):
    raise ImportError("no such file")


def _other_torch(name, package=None):
    return types.SimpleNamespace(torch_version="1.0.0", bind=lambda *a: pytest.fail("used"))


@pytest.mark.parametrize("load", [_missing, _other_torch], ids=["missing", "other_torch"])
def test_the_library_loads_without_it(monkeypatch, load):
    for name, value in (("_lib", None), ("_product_lib", None), ("native", None), ("_native_missing", False)):
        monkeypatch.setattr(_lib, name, value)
    monkeypatch.setattr(importlib, "import_module", load)
    with pytest.warns(RuntimeWarning, match="_native.so is not used"):
        assert _lib.load().artab_version() == _lib.ABI_VERSION
    assert _lib.native is None and ak._call("context_attention", None, None, None, None, 0) is None
    with _lib.benchmark_library() as lib:  # no second warning, no second attempt
        assert lib.artab_version() == _lib.ABI_VERSION


def test_it_is_used_where_it_fits():
    _lib.load()
    assert _lib.native is not None
