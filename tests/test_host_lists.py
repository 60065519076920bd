"""Host lists that the ops hand to the C entries, on the CPU: values that do not fit are refused, and an array is
never one that was made from other values."""
from importlib import import_module

import pytest


@pytest.fixture(scope="module")
def ops(pkg):
    return import_module(pkg.__name__ + ".ops")


@pytest.mark.parametrize("bad", [2 ** 31, -2 ** 31 - 1, 2 ** 32 + 4])
def test_int32_lists_refuse_what_does_not_fit(ops, pkg, bad):
    assert list(ops._i32_array([2 ** 31 - 1, -2 ** 31])) == [2 ** 31 - 1, -2 ** 31]
    with pytest.raises(RuntimeError, match="int32"):
        ops._i32_array([1, bad])
    if bad > 0:  # a stride or k of a key set (2^32 + 4 would be a stride of 4 in 32 bits)
        geom = pkg.Geometry(2, 20, 5)
        with pytest.raises(RuntimeError, match="int32"):
            ops.keyset_build([ops.KeySetSpec(0, ops.KEYSET_STRIDE, bad)], geom, None, "cpu")
