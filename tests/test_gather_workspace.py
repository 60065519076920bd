"""The sliced gather's workspace, on the CPU with a stand-in for the library: calls that may run at the same time
(streams, threads) never share one, and none is kept for a later call, whose stream can be another."""
import weakref
from importlib import import_module

import pytest
import torch


@pytest.mark.parametrize("other", [1 << 15, 1 << 14])
def test_overlapping_calls_have_workspaces_of_their_own(pkg, monkeypatch, other):
    ops = import_module(pkg.__name__ + ".ops")
    L = import_module(pkg.__name__ + "._lib")
    held, made = [], []
    empty = torch.empty

    def track(*a, **k):
        t = empty(*a, **k)
        made.append(weakref.ref(t))
        return t

    class Lib:
        def saf3r_gather_attn_workspace_bytes(self, n, topk):
            return 64 * n

        def saf3r_gather_attn_fwd_sliced(self, *a):
            ptr, nbytes = a[11], a[12]
            held.append((ptr, nbytes))
            if len(held) == 1:  # a second call while the first one's kernels are in flight
                call(other)
            return 0

    monkeypatch.setattr(L, "load", lambda: Lib())
    monkeypatch.setattr(L, "stream_ptr", lambda *a: None)
    monkeypatch.setattr(torch, "empty", track)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: "cpu")
    r = L.Rows(16, 64, 0, 1 << 40, 0)

    def call(n):
        idx = torch.zeros(n, 1, dtype=torch.int32)
        ops.gather_attn_rows(r, r, r, idx, 1, n, 1, 4, None, r, sliced=True)

    call(1 << 15)
    (a, na), (b, nb) = held
    assert na == 64 << 15 and nb == 64 * other
    assert a + na <= b or b + nb <= a  # both are held until their calls return
    assert len(made) == 2 and all(t() is None for t in made)
