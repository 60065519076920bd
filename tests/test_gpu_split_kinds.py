"""Every kind of walk on the split route (tests/split_cases.py), with the route asserted: against the oracle on the
inputs the kernels consumed, with plain and prescaled Q, and with outliers that send prescaled items to the
exact walk (the bars of the other attention tests)."""
import importlib

import pytest
import torch

from oracle import attention as OA
from tests.split_cases import CASES, capacity, case, list_width, split_heads
from tests.test_gpu_split_walks import DEV, _check, _inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order", ["fixed", "paced"])
@pytest.mark.parametrize("prescaled,outliers", [(False, False), (True, False), (False, True), (True, True)])
@pytest.mark.parametrize("c", [c for c in CASES if c[-1] != []], ids=[c[0] for c in CASES if c[-1] != []])
def test_split_kinds(pkg, c, prescaled, outliers, order):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    ops = importlib.import_module(pkg.__name__ + ".ops")
    lib = importlib.import_module(pkg.__name__ + "._lib").load()
    geom, patterns, layouts, want = case(ops, pkg, *c)
    og = OA.Geometry(geom.frames, geom.tokens_per_frame, geom.num_special)
    assert split_heads(lib, geom, patterns, layouts, compute_units=0) == want
    N, H = geom.tokens, len(patterns)
    q, k, v = _inputs(H, N, outliers, 3 * N + H)
    flags = [prescaled] * H
    qp, kp, vp = ops.pack_heads(q.to(DEV), k.to(DEV), v.to(DEV), geom, token_order=layouts, q_scaled=flags)
    sel = ks = idx = None
    dyn = [h for h, p in enumerate(patterns) if p == ops.BLOCK_DYNAMIC]
    if dyn:
        sel = ops.block_select(*ops.block_pool(qp, kp, geom, dyn), geom.frames, geom.blocks_per_frame, 2)
        assert sel.shape[-1] == list_width(geom)
    keyed = [h for h, p in enumerate(patterns) if p in ops.KEYSET_PATTERNS]
    if keyed:  # sets of every token
        specs = [ops.KeySetSpec(h, ops.KEYSET_STRIDE, 1, 0, True) for h in keyed]
        idx, count = ops.keyset_build(specs, geom, None, DEV)
        ks = ops.keyset_gather(kp, geom, specs, v.permute(1, 0, 2).contiguous().to(DEV), H * 64, 64, idx, count)
        assert ks.capacity == capacity(geom)
    out = torch.full((N, H * 64 + 64), 7.0, dtype=torch.bfloat16, device=DEV)
    ops.sparse_attn_fwd(qp, kp, vp, geom, patterns, sel, out=out, keysets=ks, token_order=layouts, q_scaled=flags,
                        order=order)
    torch.cuda.synchronize()
    assert (out[:, H * 64:] == 7).all()
    got = out[:, :H * 64].float().cpu().reshape(N, H, 64).permute(1, 0, 2)
    f = ops.prescale_factor()
    qu = (q.float() * f).to(torch.bfloat16).float() / f if prescaled else q.float()
    special = torch.arange(N) % geom.tokens_per_frame < geom.num_special
    for h, pat in enumerate(patterns):
        lists_only = pat in ops.TOKEN_PATTERNS  # their patch rows are the gather's
        rows = special if lists_only else torch.ones(N, dtype=torch.bool)
        extra = sel[dyn.index(h)].cpu() if h in dyn else None
        ref = OA.sparse_attention_gathered(qu[h], k[h].float(), v[h].float(),
                                           ops.DENSE if lists_only or pat == ops.KEYSET else pat, og, extra,
                                           dtype=torch.float64)
        _check(got[h][rows], ref[rows], f"{c[0]} head {h} {c[4][h]}")
        if lists_only:
            assert (got[h][~special] == 7).all()
