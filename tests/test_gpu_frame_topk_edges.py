"""``saf3r_frame_topk_scores`` at the edges of its frame stage: frame lengths around its register counts and word
alignment, list lengths around its candidate window, many and few distinct scores; bit-exact with the oracle."""
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


@pytest.mark.parametrize("P", [1, 2, 63, 127, 128, 129, 254, 255, 256, 382, 383, 639, 895, 896, 1036, 1151, 1369, 1407,
                               1408, 2175, 2176, 3199, 4095, 4096])
@pytest.mark.parametrize("k", [1, 4, 16, 64, 65, 127, 128, 129, 300])
def test_frame_stage(ops, P, k):
    g = torch.Generator().manual_seed(31 * P + k)
    F, rows = 3, 3
    width = -(-F * P // 8) * 8
    for x in (torch.randn(rows, width, generator=g), torch.randint(-3, 4, (rows, width), generator=g).float(),
              torch.nn.functional.normalize(torch.randn(rows, width, generator=g), dim=-1).abs()):
        x = x.to(torch.bfloat16)
        x[:, 5::17] = -0.0
        x[1, ::3] = float("inf")
        x[2, 1::2] = -float("inf")
        got = ops.frame_topk_scores(x.to(DEV), F, P, k)
        want = OS.token_topk_from_scores(x[:, :F * P].contiguous().view(torch.int16).numpy().view(np.uint16), F, P, k)
        assert np.array_equal(got.cpu().numpy(), want)


def test_frame_stage_into_a_wider_output(ops):
    """``out`` rows wider apart than the list, and a capped list (the candidates' order keys)."""
    g = torch.Generator().manual_seed(2)
    F, P, k, rows = 4, 333, 20, 9
    x = torch.randn(rows, 1336, generator=g).to(torch.bfloat16)
    bits = x[:, :F * P].contiguous().view(torch.int16).numpy().view(np.uint16)
    big = torch.full((rows, 100), -7, dtype=torch.int32, device=DEV)
    ops.frame_topk_scores(x.to(DEV), F, P, k, out=big[:, 10:90])
    assert np.array_equal(big[:, 10:90].cpu().numpy(), OS.token_topk_from_scores(bits, F, P, k))
    assert (big[:, :10] == -7).all() and (big[:, 90:] == -7).all()
    got = ops.frame_topk_scores(x.to(DEV), F, P, k, cap=33)
    assert np.array_equal(got.cpu().numpy(), OS.token_topk_from_scores(bits, F, P, k, cap=33))
