"""Row addressing of the gather attention: the narrow form (24-bit rows and strides on uniform bases) and the
general one give the same results, for plain and frame-mapped rows, in one pass and sliced."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops(pkg):
    from importlib import import_module
    return import_module(pkg.__name__ + ".ops")


@pytest.mark.parametrize("flags", range(8))  # q / k, v and out in fp32 or bf16
@pytest.mark.parametrize("mapped", [False, True])
@pytest.mark.parametrize("sliced", [False, True])
def test_narrow_and_general_rows(ops, flags, mapped, sliced):
    g = torch.Generator().manual_seed(flags)
    frames, P, T = 3, 37, 42
    n, nk, topk = 101, frames * P, 130
    qk = torch.float32 if flags & 1 else torch.bfloat16
    vt = torch.float32 if flags & 2 else torch.bfloat16
    ot = torch.float32 if flags & 4 else torch.bfloat16
    q = torch.randn(n, 64, generator=g).to(qk)
    k = torch.randn(frames * T, 64, generator=g).to(qk)
    v = torch.randn(frames * T, 128, generator=g).to(vt)  # rows 128 apart
    idx = torch.randint(-2, nk + 3, (n, topk), generator=g, dtype=torch.int32)  # some out of range
    rpf, base, frs = (P, 5, T) if mapped else (None, 2, 0)
    ref_rows = torch.arange(nk) + base + (torch.arange(nk) // P * (T - P) if mapped else 0)
    kk, vv = k[ref_rows].double(), v[ref_rows, 64:].double()
    ok = (idx >= 0) & (idx < nk)
    li = idx.clamp(0, nk - 1).long()
    s = ((q.double()[:, None] * kk[li]).sum(-1) * 0.125).masked_fill(~ok, -torch.inf)
    want = (torch.softmax(s, -1)[..., None] * vv[li]).sum(1)
    qd, kd, vd, idxd = q.to(DEV), k.to(DEV), v.to(DEV), idx.to(DEV)
    outs = []
    # the general form: V through a map of its own (another frame stride, or frames where K has none)
    wide = torch.zeros(frames * (T + 3), 128, dtype=vt, device=DEV)
    wide.view(frames, T + 3, 128)[:, :T] = vd.view(frames, T, 128)
    for general in (False, True):
        out = torch.full((n, 64), float("nan"), dtype=ot, device=DEV)
        kr = ops.rows(kd, base_row=base, rows_per_frame=rpf, frame_row_stride=frs)
        vr = ops.rows(vd, base_row=base, rows_per_frame=rpf, frame_row_stride=frs, offset=64)
        if general and mapped:
            vr = ops.rows(wide, base_row=base, rows_per_frame=P, frame_row_stride=T + 3, offset=64)
        elif general:
            vr = ops.rows(vd, base_row=base, rows_per_frame=nk, frame_row_stride=nk, offset=64)
        ops.gather_attn_rows(ops.rows(qd), kr, vr, idxd, topk, n, topk, nk, None, ops.rows(out), dtype_flags=flags,
                             sliced=sliced)
        outs.append(out.cpu())
    assert torch.equal(outs[0], outs[1])
    # fp32 out: fp32 sums of 64 and 130 terms; bf16 out: one rounding more (2^-9 relative)
    tol = 2e-5 if flags & 4 else 2 ** -8
    assert (outs[0].double() - want).abs().max() <= tol * want.abs().max()
