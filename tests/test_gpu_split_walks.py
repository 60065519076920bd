"""Short attention launches of mixed heads, some of whose long single-range walks run one query tile per
work-group, the key tiles split over its four waves, against the oracle on the inputs the kernels consumed
(bf16 inputs, fp64 oracle; the bars of the other attention tests, which bound the bf16 rounding of P and of
the output). Which heads split depends on the mix: ANCHOR_LOCAL alone, DENSE and KEYSET, or none where a
packed frame-relative head has the longest walk. Each kind on the split route: test_gpu_split_kinds.py.
"""
import importlib

import pytest
import torch

from oracle import attention as OA

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
ATOL_MAX, ATOL_MEAN = 2e-2, 2e-3


@pytest.fixture(scope="module")
def ops(pkg):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return importlib.import_module(pkg.__name__ + ".ops")


def _check(got, ref, what):
    e = (got - ref.float()).abs()
    print(f"{what}: max {e.max().item():.3g} mean {e.mean().item():.3g}", flush=True)
    assert torch.isfinite(got).all() and e.max().item() <= ATOL_MAX and e.mean().item() <= ATOL_MEAN, what


def _inputs(H, N, outliers, seed):
    g = torch.Generator().manual_seed(seed)
    if not outliers:
        return [(1.5 * torch.randn(H, N, 64, generator=g)).to(torch.bfloat16) for _ in range(3)]
    # two keys 69 and 173 log2 units above the rest, met late: prescaled items are marked and walked again
    q = (0.5 + 0.1 * torch.randn(H, N, 64, generator=g)).to(torch.bfloat16)
    k = (0.3 * torch.randn(H, N, 64, generator=g)).to(torch.bfloat16)
    k[:, 40], k[:, N - 8] = 12.0, 30.0
    return q, k, torch.randn(H, N, 64, generator=g).to(torch.bfloat16)


@pytest.mark.parametrize("order", ["fixed", "paced"])
@pytest.mark.parametrize("prescaled,outliers", [(False, False), (True, False), (False, True), (True, True)])
@pytest.mark.parametrize("F,T,ns", [(4, 450, 5), (2, 1041, 5), (27, 65, 1), (25, 64, 0), (1, 1601, 5), (2, 1700, 5)])
def test_split_walks(ops, pkg, F, T, ns, prescaled, outliers, order):
    geom, og = pkg.Geometry(F, T, ns), OA.Geometry(F, T, ns)
    N = geom.tokens
    patterns = [ops.DENSE, ops.DENSE, ops.KEYSET, ops.BLOCK_DYNAMIC, ops.FRAME_LOCAL, ops.ANCHOR_LOCAL, ops.ANCHOR]
    H = len(patterns)
    tord = ops.token_order_heads(patterns, geom)
    tord = [ops.LAYOUT_PACKED if h == 1 else t for h, t in enumerate(tord)]  # head 1: dense, packed layout
    q, k, v = _inputs(H, N, outliers, F * 7 + T)
    flags = [prescaled] * H
    qp, kp, vp = ops.pack_heads(q.to(DEV), k.to(DEV), v.to(DEV), geom, token_order=tord, q_scaled=flags)
    sel = ops.block_select(*ops.block_pool(qp, kp, geom, [3]), geom.frames, geom.blocks_per_frame, 2)
    specs = [ops.KeySetSpec(2, ops.KEYSET_STRIDE, 1, 0, True)]
    idx, count = ops.keyset_build(specs, geom, None, DEV)
    ks = ops.keyset_gather(kp, geom, specs, v.permute(1, 0, 2).contiguous().to(DEV), H * 64, 64, idx, count)
    out = torch.full((N, H * 64 + 64), 7.0, dtype=torch.bfloat16, device=DEV)
    ops.sparse_attn_fwd(qp, kp, vp, geom, patterns, sel, out=out, keysets=ks, token_order=tord, q_scaled=flags,
                        order=order)
    torch.cuda.synchronize()
    assert (out[:, H * 64:] == 7).all()
    c = ops.prescale_factor()
    qu = (q.float() * c).to(torch.bfloat16).float() / c if prescaled else q.float()
    got = out[:, :H * 64].float().cpu().reshape(N, H, 64).permute(1, 0, 2)
    for h, pat in enumerate(patterns):
        extra = sel[0].cpu() if h == 3 else idx[0, :int(count[0])].cpu() if h == 2 else None
        ref = OA.sparse_attention_gathered(qu[h], k[h].float(), v[h].float(), pat, og, extra, dtype=torch.float64)
        _check(got[h], ref, f"F{F} T{T} ns{ns} head {h} pattern {pat} layout {tord[h]}")


@pytest.mark.parametrize("pattern", ["KEYSET", "TOKEN_DYNAMIC_KEYSET"])
@pytest.mark.parametrize("count", [1, 63, 64, 65, 257])
def test_split_small_keysets(ops, pkg, pattern, count):
    """Key sets far below their capacity, which is what the choice of the route sees: waves without a tile."""
    F, T, ns = 4, 450, 5
    geom, og = pkg.Geometry(F, T, ns), OA.Geometry(F, T, ns)
    N = geom.tokens
    patterns = [getattr(ops, pattern), getattr(ops, pattern)]
    q, k, v = _inputs(2, N, False, count)
    qp, kp, vp = ops.pack_heads(q.to(DEV), k.to(DEV), v.to(DEV), geom)
    specs = [ops.KeySetSpec(h, ops.KEYSET_STRIDE, 1, 0, True) for h in range(2)]
    idx, cnt = ops.keyset_build(specs, geom, None, DEV)
    cnt[0] = count
    ks = ops.keyset_gather(kp, geom, specs, v.permute(1, 0, 2).contiguous().to(DEV), 2 * 64, 64, idx, cnt)
    out = torch.zeros(N, 2 * 64, dtype=torch.bfloat16, device=DEV)
    ops.sparse_attn_fwd(qp, kp, vp, geom, patterns, out=out, keysets=ks)
    torch.cuda.synchronize()
    got = out.float().cpu().reshape(N, 2, 64).permute(1, 0, 2)
    rows = torch.tensor([f * T + s for f in range(F) for s in range(ns)]) if pattern != "KEYSET" else torch.arange(N)
    for h in range(2):
        keys = idx[h, :int(cnt[h])].cpu()
        ref = OA.sparse_attention_gathered(q[h].float(), k[h].float(), v[h].float(), ops.KEYSET, og, keys,
                                           dtype=torch.float64)
        _check(got[h][rows], ref[rows], f"{pattern} {int(cnt[h])} keys")
