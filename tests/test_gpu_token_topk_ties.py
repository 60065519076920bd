"""Token top-k over frames of equal, few and far-apart scores, whose counts jump over the candidate window or close
in on it slowly. Scores are small integers times powers of two or infinite, exact in any summation order: the indices
must equal the oracle's."""
from importlib import import_module

import numpy as np
import pytest
import torch

from oracle import selection as OS

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _scores(kind, frames, P, g):
    """Key scores [frames, P]."""
    n = (frames, P)
    if kind == "equal":
        return np.full(n, 3.0)
    if kind == "zeros":
        return np.zeros(n)
    if kind == "few":
        return g.integers(-2, 3, n).astype(np.float64)
    if kind == "few_above":  # fewer than k above a mass of equal scores
        return np.where(g.random(n) < 0.02, 5.0, 1.0)
    if kind == "few_below":
        return np.where(g.random(n) < 0.98, 5.0, 1.0)
    if kind == "outliers":  # three far above integers that differ
        s = g.permuted(np.tile(np.arange(P) % 128, (frames, 1)), axis=1).astype(np.float64)
        s[:, [0, P // 2, P - 1]] = [2.0 ** 100, 2.0 ** 60, 2.0 ** 100]
        return s
    if kind == "spread":  # every power of two from 2^-60 to 2^60
        return 2.0 ** (g.integers(-60, 61, n).astype(np.float64))
    if kind == "lowest":  # fewer than k finite scores
        return np.where(g.random(n) < 0.01, 2.0, -np.inf)
    s = g.integers(0, 100, n).astype(np.float64)  # "infinite": both, over a hundred values
    s[:, :2], s[:, P // 3] = np.inf, -np.inf
    return s


@pytest.mark.parametrize("P", [20, 64, 65, 129, 300, 1036, 1369, 1600, 4096])
@pytest.mark.parametrize("k", [4, 17, 32, 33, 64, 65, 128])
def test_tied_scores(pkg, P, k):
    ops = import_module(pkg.__name__ + ".ops")
    g = np.random.default_rng(P + k)
    frames, nq = 2, 19
    for kind in ("equal", "zeros", "few", "few_above", "few_below", "outliers", "spread", "lowest", "infinite"):
        sign = np.where(np.arange(nq) % 3 == 2, -1.0, 1.0)  # of the finite scores
        ks = _scores(kind, frames, P, g).reshape(-1)
        fin = np.isfinite(ks)
        q, key = torch.zeros(nq, 64), torch.zeros(frames * P, 64)
        q[:, 0], q[:, 1] = torch.from_numpy(sign), 1.0
        key[:, 0] = torch.from_numpy(np.where(fin, ks, 0.0))
        key[:, 1] = torch.from_numpy(np.where(fin, 0.0, ks))
        s = np.where(fin, sign[:, None] * np.where(fin, ks, 0.0), ks).astype(np.float32) + np.float32(0.0)
        got = ops.token_topk(q.to(torch.bfloat16).to(DEV), key.to(torch.bfloat16).to(DEV), frames, P, k).cpu().numpy()
        want = OS.frame_topk(s, frames, k)
        assert np.array_equal(got, want), f"{kind}: {(got != want).mean():.3%} of the indices differ"
