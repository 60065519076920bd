"""A library built from older sources is refused with the reason, whether its version or an entry is missing."""
import ctypes
from importlib import import_module

import pytest


class _Fn:
    def __init__(self, value):
        self.value = value

    def __call__(self, *a):
        return self.value


@pytest.mark.parametrize("missing,version,match", [("saf3r_pack_qkv_typed", 13, "saf3r_pack_qkv_typed.*build"),
                                                   (None, 12, "ABI 12"), ("saf3r_pack_qkv_typed", 12, "ABI 12")])
def test_older_library_is_refused(pkg, monkeypatch, missing, version, match):
    L = import_module(pkg.__name__ + "._lib")

    class Lib:
        def __getattr__(self, name):
            if name == missing:
                raise AttributeError(f"undefined symbol: {name}")
            fn = _Fn(version)
            setattr(self, name, fn)
            return fn

    monkeypatch.setattr(L, "_lib", None)
    monkeypatch.setattr(ctypes, "CDLL", lambda path: Lib())
    with pytest.raises(RuntimeError, match=match):
        L.load()
    assert L._lib is None
