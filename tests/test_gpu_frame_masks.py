"""Frame-relative heads in the packed layout (frames whose special tokens do not fit the padding of the last
patch tile): the keys a row may see, at the sizes where the mask of a special tile can go wrong, against
the oracle on the inputs the kernels consumed (the bars of the other attention tests). Frames whose
specials straddle two tiles, exactly fill one, are more than one tile, and the last frame's at the end of
a full tile; one frame, and frames of a single patch tile.
"""
import importlib

import pytest
import torch

from oracle import attention as OA

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
ATOL_MAX, ATOL_MEAN = 2e-2, 2e-3


@pytest.mark.parametrize("prescaled", [False, True])
@pytest.mark.parametrize("F,T,ns", [(13, 69, 5), (30, 69, 5), (64, 65, 1), (4, 80, 16), (2, 128, 64), (2, 193, 128),
                                    (1, 133, 5), (5, 261, 5), (3, 129, 65), (3, 200, 70), (4, 130, 66)])
def test_packed_frame_relative(pkg, F, T, ns, prescaled):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    ops = importlib.import_module(pkg.__name__ + ".ops")
    geom, og = pkg.Geometry(F, T, ns), OA.Geometry(F, T, ns)
    patterns = [ops.FRAME_LOCAL, ops.ANCHOR_LOCAL, ops.ANCHOR, ops.DENSE]
    H, N = len(patterns), geom.tokens
    g = torch.Generator().manual_seed(F * 31 + T)
    q, k, v = [(1.5 * torch.randn(H, N, 64, generator=g)).to(torch.bfloat16) for _ in range(3)]
    flags = [prescaled] * H
    packed = [ops.LAYOUT_PACKED] * H
    qp, kp, vp = ops.pack_heads(q.to(DEV), k.to(DEV), v.to(DEV), geom, token_order=packed, q_scaled=flags)
    out = ops.sparse_attn_fwd(qp, kp, vp, geom, patterns, token_order=packed, q_scaled=flags)
    torch.cuda.synchronize()
    c = ops.prescale_factor()
    qu = (q.float() * c).to(torch.bfloat16).float() / c if prescaled else q.float()
    got = out.float().cpu().reshape(N, H, 64).permute(1, 0, 2)
    for h, pat in enumerate(patterns):
        ref = OA.sparse_attention_gathered(qu[h], k[h].float(), v[h].float(), pat, og, None, dtype=torch.float64)
        e = (got[h] - ref.float()).abs()
        print(f"F{F} T{T} ns{ns} pattern {pat}: max {e.max().item():.3g} mean {e.mean().item():.3g}", flush=True)
        assert torch.isfinite(got[h]).all() and e.max().item() <= ATOL_MAX and e.mean().item() <= ATOL_MEAN
