"""Which heads of a launch run split (host computation, CPU): every case of tests/split_cases.py takes the route that
test_gpu_split_kinds.py means to run, and the query refuses what the launch refuses."""
import ctypes
from importlib import import_module

import pytest

from tests.split_cases import CASES, case, split_heads


@pytest.fixture(scope="module")
def mods(pkg):
    return import_module(pkg.__name__ + ".ops"), import_module(pkg.__name__ + "._lib").load()


@pytest.mark.parametrize("c", CASES, ids=[c[0] for c in CASES])
def test_split_route(mods, pkg, c):
    ops, lib = mods
    geom, patterns, layouts, want = case(ops, pkg, *c)
    assert split_heads(lib, geom, patterns, layouts) == want


def test_split_route_of_a_small_chip(mods, pkg):
    """No idle work-groups to split into."""
    ops, lib = mods
    geom, patterns, layouts, want = case(ops, pkg, *next(c for c in CASES if c[0] == "s128"))
    assert want and split_heads(lib, geom, patterns, layouts, compute_units=4) == []


def test_split_query_refuses(mods):
    _, lib = mods
    q, mask = lib.saf3r_sparse_attn_split_heads, ctypes.c_uint64(0)
    one, out = (ctypes.c_int32 * 1)(0), ctypes.byref(mask)
    assert q(2, 100, 5, 1, one, 0, 0, None, 256, out) == 0 and mask.value == 0
    for bad in ((0, 100, 5, 1, one, 0, 0, None, 256, out), (2, 100, 5, 65, one, 0, 0, None, 256, out),
                (2, 100, 5, 1, None, 0, 0, None, 256, out), (2, 100, 5, 1, one, 0, 0, None, 256, None),
                (2, 100, 5, 1, (ctypes.c_int32 * 1)(10), 0, 0, None, 256, out),
                (2, 100, 5, 1, one, 0, 0, (ctypes.c_uint8 * 1)(2), 256, out),
                (2, 100, 5, 1, one, 0, 0, None, -1, out)):
        assert q(*bad) == 1 and lib.saf3r_last_error()
