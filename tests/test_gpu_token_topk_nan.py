"""Token top-k over scores that hold NaNs of both signs and infinities. The order is that of the sortable key:
+NaN above +inf, -NaN below -inf, equal bits by the lower index. Scores are distinct integers (or, with ties, small
ones), exact in any summation order, but for the keys that carry a NaN or an infinity in a feature of their own:
the indices must equal the oracle's.
"""
import numpy as np
import pytest
import torch

from oracle import selection as OS

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
NAN_BITS = {"+": 0x7FC0, "-": 0xFFC0}  # bf16


@pytest.fixture(scope="module")
def ops(pkg):
    from importlib import import_module
    return import_module(pkg.__name__ + ".ops")


def _special(bits, n):
    return torch.full((n,), bits, dtype=torch.int32).to(torch.uint16).view(torch.bfloat16)


def _topk(ops, q, k, frames, P, topk):
    return ops.token_topk(q.to(DEV), k.to(DEV), frames, P, topk).cpu().numpy()


def _handed_on(ops, sign, frames, nq, P):
    """Sign of the score that a key holding a NaN of ``sign`` gets: in a list of all P keys of a frame it stands
    first or last."""
    q = torch.zeros(nq, 64)
    q[:, 0] = q[:, 1] = 1.0
    k = torch.zeros(frames * P, 64)
    k[:, 0] = torch.arange(frames * P) % 8
    k = k.to(torch.bfloat16)
    k[3::P, 1] = _special(NAN_BITS[sign], frames)
    got = _topk(ops, q.to(torch.bfloat16), k, frames, P, P)
    assert got[0, 0] == 3 or got[0, P - 1] == 3
    return "+" if got[0, 0] == 3 else "-"


# the small launches of k <= 16 and k > 16 take the LDS score rows, the larger launch of k <= 8 the two passes
@pytest.mark.parametrize("frames,nq,P,topk,small", [(2, 40, 1036, 64, 20), (2, 40, 1036, 20, 20), (2, 40, 200, 128, 20),
                                                    (2, 40, 60, 20, 20), (2, 40, 1600, 64, 20), (2, 40, 4096, 128, 20),
                                                    (2, 40, 1036, 8, 8), (14, 2005, 300, 8, 8)])
@pytest.mark.parametrize("nans", [1, 10, 40, 100])
@pytest.mark.parametrize("sign", ["+", "-"])
@pytest.mark.parametrize("ties", [False, True])
def test_nan_scores(ops, frames, nq, P, topk, small, nans, sign, ties):
    nans = min(nans, P - 3)
    g = torch.Generator().manual_seed(P + topk + nans)
    q, k = torch.zeros(nq, 64), torch.zeros(frames * P, 64)
    if ties:
        q, k = (torch.randint(-4, 5, t.shape, generator=g).float() for t in (q, k))
    else:  # every key of a frame a score of its own, up to the sign of the query
        rank = torch.cat([torch.randperm(P, generator=g) for _ in range(frames)]).float()
        q[:, 0], q[:, 1] = 64.0, 1.0
        q *= torch.randint(0, 2, (nq, 1), generator=g) * 2.0 - 1.0
        k[:, 0], k[:, 1] = rank // 64, rank % 64
    q[:, 7] = 1.0  # the feature of the special values
    k[:, 7] = 0.0
    s = q.double() @ k.double().T
    k = k.to(torch.bfloat16)
    s = s.float().numpy()
    seen = _handed_on(ops, sign, frames, nq, small)
    nan_score = np.array([0x7FC00000 if seen == "+" else 0xFFC00000], dtype=np.uint32).view(np.float32)
    for f in range(frames):
        at = f * P + torch.randperm(P, generator=g)
        nan, pos, neg = at[:nans], at[nans:nans + 1], at[nans + 1:nans + 3]
        k[nan, 7] = _special(NAN_BITS[sign], nans)
        if not ties:  # (the infinities go with the ties: a row that holds one takes no score window)
            s[:, nan.numpy()] = nan_score
            continue
        k[pos, 7], k[neg, 7] = float("inf"), float("-inf")
        s[:, nan.numpy()] = nan_score
        s[:, pos.numpy()], s[:, neg.numpy()] = np.inf, -np.inf
    got = _topk(ops, q.to(torch.bfloat16), k, frames, P, topk)
    want = OS.frame_topk(s, frames, topk)
    print(f"NaN {sign} handed on as {seen}: {(got != want).mean():.4%} of the indices differ", flush=True)
    assert np.array_equal(got, want)
