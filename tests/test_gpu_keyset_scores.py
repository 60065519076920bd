"""Probe scores that a layer keeps (``last_keysets.scores``): one row per key-set head, in head order; rows of
stride heads, which have no scores, are zeros."""
import importlib

import pytest
import torch

from tests.layer_check import make_stack

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("ratios", [(1.0, 1.0), (1.0, 0.5)])
def test_scores_of_stride_heads_are_zero(pkg, ratios, monkeypatch):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    plug, vggt, synth = (importlib.import_module(pkg.__name__ + m) for m in (".patch", ".vggt", ".synth"))
    ph, pw, frames, H = 7, 9, 3, 4
    m = make_stack(vggt, 1, 64 * H, H).to(DEV).to(torch.bfloat16)
    cfg = {"patch_module": {"type": "headsparse", "topk_mode": "token", "lazy_dino_topk": True, "topk": 3,
                            "block_topk": 2},
           "sparse_config": {"0": [{"mode": "stride", "head_ids": [0], "stride": 4},
                                   {"mode": "q_probe_topk", "head_ids": [1], "stride": 4, "q_sample_ratio": ratios[0]},
                                   {"mode": "q_probe_topk", "head_ids": [2], "stride": 4, "q_sample_ratio": ratios[1]},
                                   {"mode": "stride", "head_ids": [3], "stride": 3}]}}
    plug.patch_model(m, "vggt", cfg)
    plug.update_args_per_forward(m, "vggt", ph * 14, pw * 14)
    N = frames * (ph * pw + 5)
    g = torch.Generator().manual_seed(4)
    x = torch.randn(1, N, 64 * H, generator=g).to(torch.bfloat16).to(DEV)
    pos = synth.vggt_positions(frames, ph, pw).to(DEV)[None]
    w = m.aggregator.global_blocks[0].attn
    assert w.keyset_heads == [0, 1, 2, 3]
    empty = torch.empty
    monkeypatch.setattr(torch, "empty", lambda *a, **k: empty(*a, **k).fill_(7))  # memory that holds no zeros
    with torch.no_grad():
        w(x, pos)
    scores = w.last_keysets.scores.cpu()
    print(f"stride rows: max |score| {scores[[0, 3]].abs().max().item()}", flush=True)
    assert (scores[[0, 3]] == 0).all() and (scores[[1, 2]] != 0).any(dim=1).all()


def test_cleared_rows_of_a_wider_output(pkg):
    """``zero_rows`` beside scored rows: each written over its N scores, every other value left alone, the scored rows
    those of a call without them."""
    ops = importlib.import_module(pkg.__name__ + ".ops")
    N = 1300
    g = torch.Generator().manual_seed(9)
    qk32 = torch.randn(3, 2, N, 64, generator=g).to(DEV)
    out = torch.full((7, N + 4), 7.0, device=DEV)
    qbar, _ = ops.probe_scores(qk32, [2, 0], out=out, rows=[5, 1], zero_rows=[0, 6, 3])
    ref_bar, ref = ops.probe_scores(qk32, [2, 0])
    assert torch.equal(qbar, ref_bar) and torch.equal(out[[5, 1], :N], ref)
    assert (out[[0, 6, 3], :N] == 0).all() and (out[[2, 4]] == 7).all() and (out[:, N:] == 7).all()
