"""``saf3r_frame_topk_scores`` at the line between the per-lane lists (k <= 4) and the threshold search, at the edges
of their word counts and of the candidate window: random and tied scores, frames that start at odd keys, with
and without the cap; bit-exact with the oracle."""
from importlib import import_module

import numpy as np
import pytest
import torch

from oracle import selection as OS

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P", [1, 2, 3, 5, 63, 127, 253, 254, 255, 382, 383, 637, 639, 893, 895, 1149, 1151, 1405, 1407,
                               1408, 1409])
@pytest.mark.parametrize("k", [1, 2, 3, 4, 5])
def test_list_edges(pkg, P, k):
    ops = import_module(pkg.__name__ + ".ops")
    g = np.random.default_rng(P + k)
    F, rows = 5, 9
    n = F * P
    bits = g.integers(0, 1 << 16, (rows, -(-n // 8) * 8)).astype(np.uint16)  # NaNs and infinities among them
    bits[4:, :n] = (0xC000 - 0x4000 * g.integers(0, 2, (rows - 4, n))).astype(np.uint16) + g.integers(0, 3, (rows - 4, n)).astype(np.uint16)
    bits[6, :n] = 0xFFFF  # the lowest key alone
    bits[7, :n] = 0x7FFF
    dev = torch.from_numpy(bits.view(np.int16)).cuda().view(torch.bfloat16)
    want = OS.token_topk_from_scores(bits[:, :n].copy(), F, P, k)
    out = torch.full((rows, want.shape[1] + 3), -7, dtype=torch.int32, device="cuda")
    ops.frame_topk_scores(dev, F, P, k, out=out[:, :want.shape[1]])
    got = out.cpu().numpy()
    assert np.array_equal(got[:, :-3], want) and (got[:, -3:] == -7).all()
    cap = max(1, want.shape[1] // 2)
    got = ops.frame_topk_scores(dev, F, P, k, exclude_first=True, first_stride=2, cap=cap).cpu().numpy()
    assert np.array_equal(got, OS.token_topk_from_scores(bits[:, :n].copy(), F, P, k, exclude_first=True, first_stride=2,
                                                         cap=cap))


@pytest.mark.parametrize("P,k", [(129, 64), (129, 65), (272, 64), (272, 65), (273, 65), (512, 80), (512, 81),
                                 (1024, 112), (1024, 113), (1036, 112), (1036, 127), (1036, 128)])
def test_window_edges(pkg, P, k):
    ops = import_module(pkg.__name__ + ".ops")
    g = np.random.default_rng(P + k)
    F, rows = 3, 8
    n = F * P
    x = torch.from_numpy(g.standard_normal((rows, -(-n // 8) * 8)).astype(np.float32)).to(torch.bfloat16)
    x[4:] = (x[4:] * 2).round()
    bits = x.view(torch.int16).numpy().view(np.uint16)
    got = ops.frame_topk_scores(x.cuda(), F, P, k).cpu().numpy()
    assert np.array_equal(got, OS.token_topk_from_scores(bits[:, :n].copy(), F, P, k))
