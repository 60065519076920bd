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


def test_lists_of_tensors_are_read_each_time(ops):
    """Elements that can change under the same identity (0-dim tensors) are read in every call, and not held."""
    import torch
    t = torch.tensor([3, 1])
    vals = [t[0], t[1]]
    assert list(ops._i32_array(vals)) == [3, 1]
    assert list(ops._u8_flags(vals, 2)) == [1, 1]
    assert list(ops._u8_layouts([t[1], t[1]], 2)) == [1, 1]
    same = [vals[1], vals[1]]
    assert list(ops._u8_layouts(same, 2)) == [1, 1]
    t[0], t[1] = 5, 0
    assert list(ops._i32_array(vals)) == [5, 0]
    assert list(ops._u8_flags(vals, 2)) == [1, 0]
    assert list(ops._u8_layouts(same, 2)) == [0, 0]


def test_lists_of_other_numbers(ops):
    """Whatever int() or bool() takes counts by its value."""
    import numpy as np
    import torch
    assert list(ops._i32_array([1.0, np.int64(2), np.float32(3), True, torch.tensor(4.0), torch.tensor(True)])) \
        == [1, 2, 3, 1, 4, 1]
    assert list(ops._i32_array(np.array([7, 8]))) == [7, 8] and list(ops._i32_array(iter([5, 6]))) == [5, 6]
    some = [2, -1, 0, 0.5, None, "x", 256, np.bool_(True), np.array(True), torch.tensor(0.0), torch.tensor(False)]
    assert list(ops._u8_flags(some, len(some))) == [1, 1, 0, 1, 0, 1, 1, 1, 1, 0, 0]
    assert list(ops._u8_flags(np.array([0, 3]), 2)) == [0, 1] and list(ops._u8_flags(torch.tensor([2, 0]), 2)) == [1, 0]
    assert list(ops._u8_layouts([1.0, True, np.int32(0), torch.tensor(1)], 4)) == [1, 1, 0, 1]
    for bad in (-1, 3, 256, 300.0):
        with pytest.raises(ValueError, match="layout"):
            ops._u8_layouts([0, bad], 2)
    for fn in (ops._u8_flags, ops._u8_layouts):
        with pytest.raises(ValueError, match="heads"):
            fn([1, 1, 1], 2)


def test_pattern_tensors_are_read_each_time(ops, pkg, monkeypatch):
    """The head counts that ``sparse_attn_fwd`` checks come from the patterns of the call."""
    import torch
    geom = pkg.Geometry(1, 20, 5)
    qp, kp, vp = ops.packed_buffers(geom, 1, "cpu")
    monkeypatch.setattr(ops, "_need_cuda", lambda *a: None)
    t = torch.tensor([ops.DENSE])
    pat = [t[0]]
    ops._pattern_counts.cache_clear()
    for p, what in ((ops.BLOCK_DYNAMIC, "selection list"), (ops.KEYSET, "key-set heads"), (ops.BROADCAST, "BROADCAST")):
        t[0] = p
        with pytest.raises(ValueError, match=what):
            ops.sparse_attn_fwd(qp, kp, vp, geom, pat)


def test_geometry_of_one_type_is_not_kept_for_another(pkg):
    """Geometries are shared by size; sizes of another type (which the C entries refuse) must not become those of a
    later call with the same integers."""
    a = pkg.Geometry.from_tokens(2 * 1043.0, 1043.0)
    b = pkg.Geometry.from_tokens(2 * 1043, 1043)
    c = pkg.Geometry.from_tokens(2 * 1043, 1043, True)
    d = pkg.Geometry.from_tokens(2 * 1043, 1043, 1)
    assert isinstance(a.frames, float) and c.num_special is True
    assert [type(x) for g in (b, d) for x in (g.frames, g.tokens_per_frame, g.num_special, g.slots)] == [int] * 8
    assert b is pkg.Geometry.from_tokens(2 * 1043, 1043)


def test_probe_scores_checks_its_rows_and_output(ops, monkeypatch):
    """Output rows, one per slot and inside ``out``, are checked before anything is launched."""
    import torch
    monkeypatch.setattr(ops, "_need_cuda", lambda *a: None)
    qk32, out = torch.zeros(3, 2, 10, 64), torch.zeros(4, 10)

    def refused(match, **kw):
        with pytest.raises(ValueError, match=match):
            ops.probe_scores(qk32, [2, 0], **kw)
    refused("rows", out=out, rows=[1])          # the kernels read a row per slot
    refused("rows", out=out, rows=[1, 2, 3])
    refused("rows", out=out, rows=[1, -1])
    refused("rows", rows=[-1, 0])
    refused("rows", out=out, rows=[1, 4])
    refused("rows", out=torch.zeros(1, 10))     # no rows given: 0 and 1
    refused("out", out=torch.zeros(4, 10, device="meta"), rows=[0, 1])  # another device's memory
    refused("out", out=out.t().contiguous().t(), rows=[0, 1])
    refused("out", out=torch.zeros(4, 9), rows=[0, 1])
    for slots in ([0, 3], [-1, 0]):
        with pytest.raises(ValueError, match="slots"):
            ops.probe_scores(qk32, slots)


def test_probe_scores_checks_its_zero_rows(ops, monkeypatch):
    """Rows to clear are rows of ``out``."""
    import torch
    monkeypatch.setattr(ops, "_need_cuda", lambda *a: None)
    qk32, out = torch.zeros(3, 2, 10, 64), torch.zeros(4, 10)
    for kw in ({}, {"out": out, "zero_rows": [4]}, {"out": out, "zero_rows": [-1]}):
        with pytest.raises(ValueError, match="zero rows"):
            ops.probe_scores(qk32, [2, 0], **{"zero_rows": [1], **kw})


def test_probe_entry_takes_zero_rows_behind_the_heads(pkg):
    """Refused before any launch: negative slots other than -1, and a head behind a row of zeros."""
    import ctypes
    lib = import_module(pkg.__name__ + "._lib").load()
    for slots, message in (([-2], b"negative"), ([0, -1, 1], b"behind"), ([-1, 0], b"behind")):
        n = len(slots)
        rc = lib.saf3r_probe_scores_host(16, 16, 640, 10, (ctypes.c_int32 * n)(*slots), (ctypes.c_int32 * n)(), n, None, 0,
                                         1.0, 16, 16, 16, 10, None)
        assert rc == 1 and message in lib.saf3r_last_error(), slots


def test_topk_key_sets_need_scores(ops, pkg):
    """Refused on the host: the kernel reads a score row for every top-k head."""
    geom = pkg.Geometry(2, 20, 5)
    stride = ops.KeySetSpec(0, ops.KEYSET_STRIDE, 3)
    for specs in ([ops.KeySetSpec(0, ops.KEYSET_TOPK, 3)], [stride, ops.KeySetSpec(1, ops.KEYSET_TOPK, 3)],
                  [stride] * 70 + [ops.KeySetSpec(1, ops.KEYSET_TOPK, 3)]):
        with pytest.raises(ValueError, match="scores"):
            ops.keyset_build(specs, geom, None, "cpu")
