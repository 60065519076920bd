"""``saf3r_frame_topk_scores`` on frames of equal and nearly equal scores, whose counts jump over the candidate
window: bit-exact with the oracle. The lowest order key (bits 0xFFFF, -NaN) and the highest (0x7FFF) among them."""
from importlib import import_module

import numpy as np
import pytest
import torch

from oracle import selection as OS

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P", [64, 128, 129, 130, 257, 1036, 1369, 4096])
@pytest.mark.parametrize("k", [1, 4, 63, 64, 65, 128, 129])
def test_tied_frames(pkg, P, k):
    ops = import_module(pkg.__name__ + ".ops")
    g = np.random.default_rng(P + k)
    F, rows = 3, 12
    n = F * P
    bits = np.zeros((rows, -(-n // 8) * 8), dtype=np.uint16)
    for r, base in enumerate((0x0000, 0x3F80, 0xBF80, 0x7FFF, 0xFFFF, 0xFF80)):
        bits[r, :n] = base
    bits[6, :n] = np.where(np.arange(n) % 2, 0x0000, 0x8000)         # +0 and -0
    bits[7, :n] = 0x3F80 + g.integers(0, 3, n)                       # three neighbouring values
    bits[8, :n] = np.where(g.random(n) < 0.02, 0x4000, 0x3F80)       # some above a mass tie
    bits[9, :n] = np.where(g.random(n) < 0.98, 0x4000, 0x3F80)       # some below
    bits[10, :n] = np.where(g.random(n) < 0.03, 0x3F80, 0xFFFF)      # fewer than k above the lowest key
    bits[11, :n] = np.where(g.random(n) < 0.5, 0x7FFF, 0xFFFF)
    dev = torch.from_numpy(bits.view(np.int16)).cuda().view(torch.bfloat16)
    got = ops.frame_topk_scores(dev, F, P, k).cpu().numpy()
    assert np.array_equal(got, OS.token_topk_from_scores(bits[:, :n].copy(), F, P, k))
