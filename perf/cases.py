"""Workloads of the head-wise sparse global attention, measured through the package's public entry points.

Kinds
-----
layer     one patched global-attention layer (``patch_model`` -> ``global_blocks[0].attn(x, pos)``): qkv
          projection, QK-LayerNorm, RoPE-2D, head-wise sparse attention, output projection; bf16. Its head
          table is either a seeded mix of block patterns or a layer of the VGGT ETH3D head profile.
stack     the 24 patched layers of VGGT-1B with the whole head profile and lazy token lists, in residual form.
gather    ``fused_sparse_topk_attention``: gather attention over per-query key lists.
topk      ``compute_qk_topk_indices_fused``: per-frame token top-k of q.k.
features  ``compute_qk_topk_indices_batched``: per-frame top-k of L2-normalised patch features.

Tokens, features and queries are spatially smooth fields with per-token and per-frame noise, as patch tokens
of neighbouring views are: a token has near matches around its own place in every frame.
"""
from __future__ import annotations

import importlib
import json
import math
import os

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROFILE_PATH = os.path.join(ROOT, "tests", "golden", "vggt_eth3d_profile.json")
NS = 5  # camera and register tokens of a frame
PATCH = 14
HEAD_DIM = 64
LAYER_SCALE = 0.25  # of a block's residual branch (a power of two: exact in bf16)
# image sizes of the configurations (518 x 518, 392 x 518, 504 x 504) and smaller ones, in patches
GRIDS = ((37, 37), (28, 37), (36, 36), (37, 28), (24, 32), (21, 37), (16, 16), (19, 33))
# layers of the head profile that need no lists from an earlier layer
PROFILE_LAYERS = (0, 3, 5, 7, 9, 10, 11, 12, 16, 18, 20, 21)


def _sub(name):
    import __graft_entry__
    return importlib.import_module(__graft_entry__.package().__name__ + "." + name)


def listed():
    return [
        # two views of a scene: the smallest call of the plugin, bound by launches and latency
        {"name": "layer_blocks_2x1041", "kind": "layer", "table": "blocks", "frames": 2, "h": 28, "w": 37, "heads": 16,
         "topk": 4, "mix": 1},
        # one layer over a short clip of 518 x 518 frames, 16 heads
        {"name": "layer_blocks_32x1374", "kind": "layer", "table": "blocks", "frames": 32, "h": 37, "w": 37,
         "heads": 16, "topk": 4, "mix": 1},
        # the benchmark's layer: VGGT-1B, 128 frames of 518 x 518
        {"name": "layer_blocks_128x1374", "kind": "layer", "table": "blocks", "frames": 128, "h": 37, "w": 37,
         "heads": 16, "topk": 4, "mix": 2},
        # a layer of the 24-head shape (504 x 504 frames, top-8 blocks)
        {"name": "layer_blocks24_48x1301", "kind": "layer", "table": "blocks", "frames": 48, "h": 36, "w": 36,
         "heads": 24, "topk": 8, "mix": 3},
        # an early layer of the head profile (anchor, strided and probe key sets) on eight 392 x 518 views
        {"name": "layer_profile7_8x1041", "kind": "layer", "table": "profile", "layer": 7, "frames": 8, "h": 28,
         "w": 37},
        # the profile layer that computes the lazy token lists (top-4) and uses them, at 32 frames
        {"name": "layer_profile11_32x1374", "kind": "layer", "table": "profile", "layer": 11, "frames": 32, "h": 37,
         "w": 37},
        # the whole patched stack, as a forward runs it, on four 392 x 518 views
        {"name": "stack_profile_4x1041", "kind": "stack", "frames": 4, "h": 28, "w": 37},
        # gather attention over top-64 lists of four views, bf16 rows
        {"name": "gather_bf16_4x1036_top64", "kind": "gather", "frames": 4, "h": 28, "w": 37, "topk": 64,
         "dtype": "bfloat16"},
        # gather attention over top-4 lists of 64 views, fp32 rows (as under autocast)
        {"name": "gather_fp32_64x1036_top4", "kind": "gather", "frames": 64, "h": 28, "w": 37, "topk": 4,
         "dtype": "float32"},
        # lazy token selection at the default top-4
        {"name": "topk4_48x1369", "kind": "topk", "frames": 48, "h": 37, "w": 37, "topk": 4},
        # the same at top-64, the list length of the feature-based setting
        {"name": "topk64_16x1036", "kind": "topk", "frames": 16, "h": 28, "w": 37, "topk": 64},
        # lists from DINO patch features, top-64 per frame with the cap of 8192 keys
        {"name": "features64_32x1036", "kind": "features", "frames": 32, "h": 28, "w": 37, "dim": 1024, "topk": 64,
         "max_topk": 8192},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("layer", "layer", "layer", "layer", "stack", "gather", "gather", "topk", "topk", "features"))
    h, w = rng.choice(GRIDS)
    if kind == "layer":
        if rng.random() < 0.5:
            heads = rng.choice((16, 16, 24))
            return {"kind": "layer", "table": "blocks", "frames": _log_int(rng, 2, 128 if heads == 16 else 64), "h": h,
                    "w": w, "heads": heads, "topk": rng.choice((2, 4, 4, 8)), "mix": rng.randint(1, 24)}
        return {"kind": "layer", "table": "profile", "layer": rng.choice(PROFILE_LAYERS),
                "frames": _log_int(rng, 2, 64), "h": h, "w": w}
    if kind == "stack":
        return {"kind": "stack", "frames": _log_int(rng, 2, 6), "h": h, "w": w}
    if kind == "gather":
        topk = rng.choice((1, 4, 4, 8, 16, 64))
        return {"kind": "gather", "frames": _log_int(rng, 2, 64 if topk <= 8 else 16), "h": h, "w": w, "topk": topk,
                "dtype": rng.choice(("bfloat16", "float32"))}
    if kind == "topk":
        topk = rng.choice((1, 4, 4, 8, 16, 32, 64))
        return {"kind": "topk", "frames": _log_int(rng, 2, 64 if topk <= 8 else 16), "h": h, "w": w, "topk": topk}
    return {"kind": "features", "frames": _log_int(rng, 2, 32), "h": h, "w": w, "dim": 1024,
            "topk": rng.choice((4, 16, 64)), "max_topk": rng.choice((1024, 8192))}


# ---- inputs ---------------------------------------------------------------------------------------------

def _field(g, frames, h, w, channels, noise=0.3):
    """[frames, h * w, channels] fp32 of unit variance: a smooth field over the patch grid plus per-token detail,
    shared by the frames, and noise of each frame's own."""
    low = torch.randn(1, channels, max(2, h // 4), max(2, w // 4), generator=g, device="cuda")
    smooth = torch.nn.functional.interpolate(low, size=(h, w), mode="bilinear", align_corners=True)[0]
    base = smooth.reshape(channels, h * w).t() + 0.6 * torch.randn(h * w, channels, generator=g, device="cuda")
    base = base / base.std()
    x = torch.empty(frames, h * w, channels, device="cuda")
    for f in range(frames):
        x[f] = base + noise * torch.randn(h * w, channels, generator=g, device="cuda")
    return x.mul_(1.0 / math.sqrt(1.0 + noise * noise))


def _tokens(g, frames, h, w, channels):
    """bf16 [1, frames * (NS + h * w), channels]: special tokens, then the patch field, per frame."""
    special = torch.randn(1, NS, channels, generator=g, device="cuda") \
        + 0.3 * torch.randn(frames, NS, channels, generator=g, device="cuda")
    x = torch.cat([special.to(torch.bfloat16), _field(g, frames, h, w, channels).to(torch.bfloat16)], dim=1)
    return x.reshape(1, frames * (NS + h * w), channels)


def _positions(frames, h, w):
    yy, xx = torch.meshgrid(torch.arange(h, device="cuda"), torch.arange(w, device="cuda"), indexing="ij")
    patch = torch.stack([yy.flatten(), xx.flatten()], dim=-1) + 1
    frame = torch.cat([torch.zeros(NS, 2, dtype=patch.dtype, device="cuda"), patch], dim=0)
    return frame.repeat(frames, 1)[None]


def _weights(model, g, dim):
    """Random weights whose k projection shares part of the q projection, as correspondence heads' do."""
    with torch.no_grad():
        for blk in model.aggregator.global_blocks:
            a = blk.attn
            wq, wk, wv, wo = (torch.randn(dim, dim, generator=g, device="cuda") / math.sqrt(dim) for _ in range(4))
            a.qkv.weight.copy_(torch.cat([wq, 0.6 * wq + 0.8 * wk, wv]))
            a.proj.weight.copy_(wo)
            for b in (a.qkv.bias, a.proj.bias):
                b.copy_(0.02 * torch.randn(b.shape, generator=g, device="cuda"))
            for n in (a.q_norm, a.k_norm):
                n.weight.copy_(1.0 + 0.1 * torch.randn(HEAD_DIM, generator=g, device="cuda"))
                n.bias.copy_(0.05 * torch.randn(HEAD_DIM, generator=g, device="cuda"))


def _profile():
    with open(PROFILE_PATH) as f:
        return json.load(f)


def _tables(case):
    """{layer: [group, ...]} of a layer or stack case, in the head-profile format."""
    if case["kind"] == "stack":
        return _profile()
    if case["table"] == "profile":
        return {"0": _profile()[str(case["layer"])]}
    synth, ops = _sub("synth"), _sub("ops")
    table = (synth.seeded_patterns if case["heads"] == 16 else synth.da3_patterns)(case["heads"], seed=case["mix"])
    names = {ops.BLOCK_DYNAMIC: "block_topk", ops.FRAME_LOCAL: "frame_local", ops.ANCHOR_LOCAL: "anchor_local",
             ops.DENSE: "dense"}
    groups = {}
    for head, p in enumerate(table):
        groups.setdefault(names[p], []).append(head)
    return {"0": [{"mode": m, "head_ids": ids} for m, ids in groups.items()]}


def _heads(case):
    return case.get("heads", 16)


def _model(case, g):
    heads = _heads(case)
    depth = 24 if case["kind"] == "stack" else 1
    with torch.device("cuda"):
        model = _sub("vggt").GlobalAttentionStack(depth=depth, dim=HEAD_DIM * heads, num_heads=heads)
    _weights(model, g, HEAD_DIM * heads)
    return model.to(torch.bfloat16).eval()


def _gather_lists(g, frames, h, w, topk):
    """int32 [frames * h * w, frames * topk]: in every frame the topk places nearest to the query's own place moved
    by a few patches (frame-major, distinct within a frame)."""
    n, P = frames * h * w, h * w
    yy, xx = torch.meshgrid(torch.arange(h), torch.arange(w), indexing="ij")
    dy, dx = yy.flatten() - h // 2, xx.flatten() - w // 2
    near = torch.argsort(dy * dy + dx * dx, stable=True)[:topk]
    dy, dx = dy[near].cuda(), dx[near].cuda()
    place = torch.arange(n, device="cuda") % P
    idx = torch.empty(n, frames, topk, dtype=torch.int32, device="cuda")
    for f in range(frames):
        oy, ox = (2.0 * torch.randn(2, n, generator=g, device="cuda")).round().long()
        y = (place // w + oy)[:, None] + dy
        x = (place % w + ox)[:, None] + dx
        idx[:, f] = (f * P + (y % h) * w + x % w).to(torch.int32)
    return idx.reshape(n, frames * topk)


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    frames, h, w = case["frames"], case["h"], case["w"]
    kind = case["kind"]
    if kind in ("layer", "stack"):
        plug = _sub("patch")
        model = _model(case, g)
        cfg = {"sparse_config": _tables(case),
               "patch_module": {"type": "headsparse", "topk_mode": "token", "lazy_dino_topk": True, "topk": 4,
                                "block_topk": case.get("topk", 4)}}
        plug.patch_model(model, "vggt", cfg)
        return {"kind": kind, "model": model, "plug": plug, "H": h * PATCH, "W": w * PATCH,
                "x": _tokens(g, frames, h, w, HEAD_DIM * _heads(case)), "pos": _positions(frames, h, w)}
    n = frames * h * w
    if kind == "features":
        f = torch.nn.functional.normalize(_field(g, frames, h, w, case["dim"]).reshape(1, n, case["dim"]), dim=-1)
        return {"kind": kind, "call": _sub("patch.utils").compute_qk_topk_indices_batched, "f": f,
                "topk": case["topk"], "P": h * w, "max_topk": case["max_topk"]}
    # q and k rows of one head: the same field seen with noise of their own (logits of a few units)
    base = _field(g, frames, h, w, HEAD_DIM)
    q = (math.sqrt(3.0) * (base + 0.3 * torch.randn(base.shape, generator=g, device="cuda"))).reshape(n, HEAD_DIM)
    k = (math.sqrt(3.0) * (base + 0.3 * torch.randn(base.shape, generator=g, device="cuda"))).reshape(n, HEAD_DIM)
    binding = _sub("kernel_binding")
    if kind == "topk":
        return {"kind": kind, "call": binding.compute_qk_topk_indices_fused, "q": q[None].to(torch.bfloat16),
                "k": k[None].to(torch.bfloat16), "topk": case["topk"], "P": h * w}
    dtype = getattr(torch, case["dtype"])
    v = torch.randn(n, HEAD_DIM, generator=g, device="cuda")
    return {"kind": kind, "call": binding.fused_sparse_topk_attention, "q": q.to(dtype), "k": k.to(dtype),
            "v": v.to(dtype), "idx": _gather_lists(g, frames, h, w, case["topk"])}


def run(state):
    kind = state["kind"]
    if kind == "gather":
        return state["call"](state["q"], state["k"], state["v"], state["idx"])
    if kind == "topk":
        return state["call"](state["q"], state["k"], state["topk"], state["P"])
    if kind == "features":
        return state["call"](state["f"], state["f"], state["topk"], per_frame=True, num_toks_per_img=state["P"],
                             max_topk=state["max_topk"])
    model = state["model"]
    blocks = model.aggregator.global_blocks
    with torch.no_grad():
        state["plug"].update_args_per_forward(model, "vggt", state["H"], state["W"])
        if kind == "layer":
            return blocks[0].attn(state["x"], state["pos"])
        x = state["x"]
        for blk in blocks:
            x = x + LAYER_SCALE * blk.attn(torch.nn.functional.layer_norm(x, x.shape[-1:]), state["pos"])
        return x


# ---- what a pass cannot do without ----------------------------------------------------------------------

def _stride_members(frames, T, stride, include):
    n = frames * T
    members = -(-n // stride)
    if include:
        members += sum(1 for t in range(T) if t % stride)
        members += sum(1 for f in range(1, frames) for s in range(NS) if (f * T + s) % stride)
    return members


def _layer_flops(groups, frames, h, w, topk):
    """FLOP of the attention and selection of one layer's heads."""
    P = h * w
    T = NS + P
    n, img, special = frames * T, frames * P, frames * NS
    blocks = -(-P // 64)
    total = 0.0
    for gr in groups:
        mode, heads, extra = gr["mode"], len(gr["head_ids"]), 0.0
        if mode == "dense":
            pairs = n * n
        elif mode in ("frame_local", "global_to_frame", "all_to_first"):
            pairs = n * T
        elif mode == "anchor_local":
            pairs = n * 2 * T - T * T
        elif mode == "block_topk":
            k = min(topk, blocks)
            pairs = special * n + img * frames * k * P / blocks
            extra = 2.0 * 64 * (frames * blocks) ** 2
        elif mode == "stride":
            pairs = n * _stride_members(frames, T, gr["stride"], gr.get("include_as", True))
        elif mode == "q_probe_topk":
            pairs = n * max(1, n // gr["stride"])
            extra = 2.0 * 64 * n
        else:  # dino_topk, lists of 4 keys per frame
            pairs = special * n + img * frames * 4
            if gr.get("is_first_dino"):
                extra = 2.0 * 64 * img * img
        total += heads * 4.0 * 64 * pairs + (extra if mode == "dino_topk" else heads * extra)
    return total


def work(case):
    frames, h, w, kind = case["frames"], case["h"], case["w"], case["kind"]
    n_img = frames * h * w
    if kind in ("layer", "stack"):
        dim = HEAD_DIM * _heads(case)
        n = frames * (NS + h * w)
        tables = _tables(case)
        flops = sum(_layer_flops(gr, frames, h, w, case.get("topk", 4)) + 8.0 * n * dim * dim for gr in tables.values())
        return {"bytes": 2.0 * 2 * n * dim + len(tables) * 4 * dim * dim * 2 + n * 16, "flops": flops}
    if kind == "features":
        width = min(frames * min(case["topk"], h * w), case["max_topk"])
        return {"bytes": n_img * case["dim"] * 4.0 + n_img * width * 4.0, "flops": 2.0 * case["dim"] * n_img * n_img}
    if kind == "topk":
        return {"bytes": 2.0 * n_img * 128 + n_img * frames * case["topk"] * 4.0, "flops": 2.0 * 64 * n_img * n_img}
    size = 2 if case["dtype"] == "bfloat16" else 4
    keys = n_img * frames * case["topk"]
    return {"bytes": 4.0 * n_img * 64 * size + keys * 4.0, "flops": 4.0 * 64 * keys}


def tolerance(case):
    """About four times what the path is off against ``exact`` (or, for key indices, against a stable sort of the
    64-bit scores; there a swap at a near tie changes two values, a moved threshold up to a frame's list)."""
    kind = case["kind"]
    if kind == "layer":  # bf16 q, k, v, P and output: 0.0025 to 0.0028
        return {"rel": 1e-2, "max": 0.1}
    if kind == "stack":  # 24 such layers on a bf16 residual stream
        return {"rel": 2.5e-2, "max": 0.3}
    if kind == "gather":  # bf16 output 0.0017, fp32 8e-7
        return {"rel": 7e-3, "max": 0.04} if case["dtype"] == "bfloat16" else {"rel": 4e-6, "max": 1e-4}
    values = case["frames"] ** 2 * case["h"] * case["w"] * min(case["topk"], case["h"] * case["w"])
    if kind == "topk":  # fp32 sums of bf16 products: 5.5e-6 of the indices at near ties
        return {"rel": 0.0, "differ": min(0.01, 2.5e-5 + 8 / values)}
    return {"rel": 0.0, "differ": min(0.01, 2.5e-5 + 128 / values)}  # scores rounded to bf16: 2.6e-6


# ---- the same in 64 bits --------------------------------------------------------------------------------

def _softmax_rows(q, k, v, out, rows, keys=None, step=4096):
    """out[rows] = softmax(q[rows] k[keys]^T / 8) v[keys] in fp64; ``rows`` / ``keys`` are slices or index tensors."""
    kt = (k if keys is None else k[keys]).t().contiguous()
    vv = v if keys is None else v[keys]
    rows = torch.arange(q.shape[0], device=q.device)[rows] if isinstance(rows, slice) else rows
    for r in rows.split(step):
        s = torch.mm(q[r], kt).mul_(0.125)
        out[r] = torch.mm(torch.softmax(s, dim=-1), vv)


def _norm_rope(x, weight, bias, eps, pos):
    """LayerNorm over head_dim, then RoPE-2D (base 100; y on features 0..31, x on 32..63); x [n, H, 64] fp64."""
    x = torch.nn.functional.layer_norm(x, (HEAD_DIM,), weight.double(), bias.double(), eps)
    inv = 1.0 / (100.0 ** (torch.arange(0, 32, 2, dtype=torch.float64, device=x.device) / 32))
    parts = []
    for axis in (0, 1):
        part = x[..., 32 * axis:32 * axis + 32]
        ang = (pos[:, axis].double()[:, None] * inv)[:, None, :]
        a, b = part[..., :16], part[..., 16:]
        parts += [a * ang.cos() - b * ang.sin(), b * ang.cos() + a * ang.sin()]
    return torch.cat(parts, dim=-1)


def _bf16(x):
    return x.to(torch.bfloat16).double()


def _block_head(q, k, v, out, frames, P, topk):
    """Patch rows over the topk key blocks of every frame by block-mean score (means of the bf16 rows)."""
    T, nb = NS + P, -(-P // 64)
    dev = q.device
    pad = torch.arange(nb * 64, device=dev)
    tok = (torch.arange(frames, device=dev)[:, None] * T + NS + pad.clamp(max=P - 1)).reshape(frames * nb, 64)
    valid = (pad < P).repeat(frames).reshape(frames * nb, 64)
    count = valid.sum(1, keepdim=True).double()
    mq, mk = ((_bf16(t)[tok] * valid[..., None]).sum(1) / count for t in (q, k))
    s = torch.mm(mq, mk.t().contiguous()).reshape(frames * nb, frames, nb)
    sel = s.topk(min(topk, nb), dim=-1).indices + (torch.arange(frames, device=dev) * nb)[None, :, None]
    sel = sel.reshape(frames * nb, -1)
    kb, vb = k[tok], v[tok]
    step = max(1, min(64, (1 << 21) // (sel.shape[1] * 64)))
    for i in range(0, frames * nb, step):
        li = sel[i:i + step]
        c = li.shape[0]
        kk = kb[li].reshape(c, -1, HEAD_DIM).transpose(1, 2).contiguous()
        p = torch.bmm(q[tok[i:i + c]], kk).mul_(0.125)
        p.masked_fill_(~valid[li].reshape(c, 1, -1), -math.inf)
        o = torch.bmm(torch.softmax(p, dim=-1), vb[li].reshape(c, -1, HEAD_DIM))
        ok = valid[i:i + c]
        out[tok[i:i + c][ok]] = o[ok]


def _list_attention(q, k, v, idx):
    out = torch.empty_like(q)
    step = max(1, (1 << 22) // idx.shape[1])
    for i in range(0, q.shape[0], step):
        li = idx[i:i + step].long()
        p = torch.softmax((q[i:i + step, None] * k[li]).sum(-1) * 0.125, dim=-1)
        out[i:i + step] = (p[..., None] * v[li]).sum(1)
    return out


def _token_lists(q, k, frames, P, topk):
    """Per-frame top-k of the bf16 rows' products."""
    kt = _bf16(k).t().contiguous()
    base = (torch.arange(frames, device=q.device) * P)[None, :, None]
    return torch.cat([(torch.mm(_bf16(r), kt).reshape(-1, frames, P).topk(topk, dim=-1).indices + base).reshape(
        r.shape[0], -1) for r in q.split(2048)])


def _layer_exact(attn, groups, x, pos, frames, h, w, topk, lists):
    """One layer in fp64 (x [n, dim] fp64); the selections read bf16 rows, as they are defined to. ``lists`` holds
    the token lists of the correspondence heads once a layer has computed them."""
    P = h * w
    T = NS + P
    n, dim = x.shape
    heads = dim // HEAD_DIM
    dev = x.device
    qkv = _bf16(torch.addmm(attn.qkv.bias.double(), x, attn.qkv.weight.double().t().contiguous()))
    qkv = qkv.reshape(n, 3, heads, HEAD_DIM)
    q = _norm_rope(qkv[:, 0], attn.q_norm.weight, attn.q_norm.bias, attn.q_norm.eps, pos).permute(1, 0, 2).contiguous()
    k = _norm_rope(qkv[:, 1], attn.k_norm.weight, attn.k_norm.bias, attn.k_norm.eps, pos).permute(1, 0, 2).contiguous()
    v = qkv[:, 2].permute(1, 0, 2).contiguous()
    token = torch.arange(n, device=dev)
    special = token[token % T < NS]
    image = token[token % T >= NS]
    out = torch.zeros(n, heads, HEAD_DIM, dtype=torch.float64, device=dev)
    every = slice(None)
    for gr in sorted(groups, key=lambda gr: not gr.get("is_first_dino", False)):
        for hd in gr["head_ids"]:
            mode = gr["mode"]
            qh, kh, vh, oh = q[hd], k[hd], v[hd], torch.zeros(n, HEAD_DIM, dtype=torch.float64, device=dev)
            if mode == "dense":
                _softmax_rows(qh, kh, vh, oh, every)
            elif mode in ("frame_local", "global_to_frame", "anchor_local"):
                for f in range(frames):
                    own = token[f * T:(f + 1) * T]
                    keys = own if mode != "anchor_local" or f == 0 else torch.cat([token[:T], own])
                    _softmax_rows(qh, kh, vh, oh, own, keys)
            elif mode == "all_to_first":
                _softmax_rows(qh, kh, vh, oh, every, token[:T])
            elif mode == "block_topk":
                _softmax_rows(qh, kh, vh, oh, special)
                _block_head(qh, kh, vh, oh, frames, P, topk)
            elif mode == "stride":
                m = token % gr["stride"] == 0
                if gr.get("include_as", True):
                    m |= (token < T) | (token % T < NS)
                _softmax_rows(qh, kh, vh, oh, every, token[m])
            elif mode == "q_probe_topk":
                best = torch.mv(kh, qh.mean(0)).topk(max(1, n // gr["stride"])).indices
                _softmax_rows(qh, kh, vh, oh, every, best)
            else:
                if gr.get("is_first_dino") and "idx" not in lists:
                    lists["idx"] = _token_lists(qh[image], kh[image], frames, P, 4)
                _softmax_rows(qh, kh, vh, oh, special)
                oh[image] = _list_attention(qh[image], kh[image], vh[image], lists["idx"])
            out[:, hd] = oh
    return torch.addmm(attn.proj.bias.double(), out.reshape(n, dim), attn.proj.weight.double().t().contiguous())


@torch.no_grad()
def exact(case, seed):
    kind, frames, h, w = case["kind"], case["frames"], case["h"], case["w"]
    if kind in ("topk", "features"):
        return None  # key indices
    if kind == "gather":
        s = prepare(case, seed)
        return _list_attention(s["q"].double(), s["k"].double(), s["v"].double(), s["idx"])
    g = torch.Generator(device="cuda").manual_seed(seed)
    model = _model(case, g)
    x = _tokens(g, frames, h, w, HEAD_DIM * _heads(case))[0].double()
    pos = _positions(frames, h, w)[0]
    tables, lists = _tables(case), {}
    blocks = model.aggregator.global_blocks
    if kind == "layer":
        return _layer_exact(blocks[0].attn, tables["0"], x, pos, frames, h, w, case.get("topk", 4), lists)[None]
    for i, blk in enumerate(blocks):
        y = torch.nn.functional.layer_norm(x, x.shape[-1:])
        x = x + LAYER_SCALE * _layer_exact(blk.attn, tables[str(i)], y, pos, frames, h, w, 4, lists)
    return x[None]
