"""Token top-k from LDS score rows (``saf3r_token_topk`` for 16 < k <= 128): frame lengths at the edges of
its tiles and register counts, query counts at the edges of its work-groups, both row maps.

The inputs are small integers (or powers of two), so every score is exact in fp32 in any summation order and
the selected indices must equal the oracle's, ties included.
"""
import numpy as np
import pytest
import torch

from oracle import selection as OS

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops(pkg):
    from importlib import import_module
    return import_module(pkg.__name__ + ".ops")


def _check(ops, q, k, frames, P, topk, **kw):
    q, k = q.to(torch.bfloat16), k.to(torch.bfloat16)
    got = ops.token_topk(q.to(DEV), k.to(DEV), frames, P, topk, **kw).cpu().numpy()
    with np.errstate(over="ignore"):
        s = (q.double() @ k.double().T).float().numpy()
    assert np.array_equal(got, OS.frame_topk(s, frames, topk))


# frame lengths around the tile (16), register (64, then pairs of 64 to 1536) and window (64, 128) edges,
# and the lengths of the longer forms (1536 / 1537, 2048 / 2049, 3073, 4096)
@pytest.mark.parametrize("P", [17, 63, 64, 65, 128, 129, 257, 639, 1036, 1369, 1408, 1409, 1536, 1537, 2049, 3073, 4096])
@pytest.mark.parametrize("topk", [17, 32, 33, 64, 65, 128])
def test_rows_exact(ops, P, topk):
    if min(topk, P) <= 16:
        pytest.skip("another kernel")
    g = torch.Generator().manual_seed(1000 * topk + P)
    frames, nq = 3, 33
    q = torch.randint(-8, 9, (nq, 64), generator=g).float()
    k = torch.randint(-8, 9, (frames * P, 64), generator=g).float()
    _check(ops, q, k, frames, P, topk)


@pytest.mark.parametrize("nq", [1, 15, 16, 17, 250])
@pytest.mark.parametrize("frames", [1, 2, 37])
def test_rows_queries_and_frames(ops, nq, frames):
    g = torch.Generator().manual_seed(nq + frames)
    q = torch.randint(-8, 9, (nq, 64), generator=g).float()
    k = torch.randint(-8, 9, (frames * 200, 64), generator=g).float()
    _check(ops, q, k, frames, 200, 40)


@pytest.mark.parametrize("topk", [20, 64, 100])
def test_rows_ties_wide_ranges_and_infinities(ops, topk):
    """Mass ties (the exact threshold), scores over many octaves of both signs (the 64-bit sort), rows with
    infinite scores, and rows of equal scores."""
    g = torch.Generator().manual_seed(topk)
    frames, P, nq = 2, 700, 40
    q = torch.zeros(nq, 64)
    q[:, 0] = 1.0
    q[10:20, 0] = 2.0 ** 100
    q[30:, 0] = 0.0  # every score 0
    k = torch.zeros(frames * P, 64)
    e = torch.randint(-40, 41, (frames * P,), generator=g).float()
    sign = torch.randint(0, 2, (frames * P,), generator=g).float() * 2 - 1
    k[:, 0] = sign * torch.exp2(e)  # 162 distinct values in 1400 keys
    _check(ops, q, k, frames, P, topk)
    ties = torch.randint(0, 3, (frames * P,), generator=g).float() - 1.0
    k[:, 0] = ties
    _check(ops, q, k, frames, P, topk)


def test_rows_general_row_map(ops):
    """Two key frames per stored frame, junk rows between: the general row map."""
    g = torch.Generator().manual_seed(3)
    frames, pad = 4, 3
    for P, topk in ((100, 40), (1036, 64), (1600, 33), (2100, 128)):
        q = torch.randint(-8, 9, (20, 64), generator=g).to(torch.bfloat16)
        k = torch.randint(-8, 9, (frames * P, 64), generator=g).to(torch.bfloat16)
        store = torch.randint(-8, 9, (2, pad + 2 * P, 64), generator=g).to(torch.bfloat16)
        store[:, pad:] = k.view(2, 2 * P, 64)
        store = store.to(DEV)
        kr = ops.rows(store.view(-1, 64), base_row=pad, rows_per_frame=2 * P, frame_row_stride=pad + 2 * P)
        got = ops.token_topk(q.to(DEV), None, frames, P, topk, krows=kr).cpu().numpy()
        assert np.array_equal(got, OS.frame_topk((q.double() @ k.double().T).float().numpy(), frames, topk))


@pytest.mark.parametrize("P", [40, 64, 100, 256, 627])
@pytest.mark.parametrize("topk", [1, 2, 4, 8, 16])
def test_two_pass_exact(ops, P, topk):
    """k <= 16 with enough queries and frames for the two-pass kernel (and, for k > 8 on short frames, the
    rows), the last work-group partly filled; integer scores with many ties: the buffers of its second pass
    overflow and frames are scanned again."""
    g = torch.Generator().manual_seed(7 * P + topk)
    frames, nq = 14, 2005
    q = torch.randint(-2, 3, (nq, 64), generator=g).float()
    k = torch.randint(-2, 3, (frames * P, 64), generator=g).float()
    _check(ops, q, k, frames, P, topk)
    k[:, 8:] = 0.0  # a few dozen distinct scores
    _check(ops, q, k, frames, P, topk)


@pytest.mark.parametrize("topk", [3, 7, 16])
def test_small_launches_take_rows(ops, topk):
    """k <= 16 below the line between the two kernels, and just above it with the same inputs."""
    g = torch.Generator().manual_seed(topk)
    for frames, nq, P in ((1, 1, 20), (2, 500, 1036), (7, 1200, 130), (14, 1200, 130)):
        q = torch.randint(-4, 5, (nq, 64), generator=g).float()
        k = torch.randint(-4, 5, (frames * P, 64), generator=g).float()
        _check(ops, q, k, frames, P, topk)
