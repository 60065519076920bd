"""Entries that take parameters as a caller holds them: bf16 LayerNorm parameters and int64 positions in the pack,
head lists from host memory in the key-set entries; each bit-identical to the converted / device-list form."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def mods(pkg):
    from importlib import import_module
    return import_module(pkg.__name__ + ".ops"), import_module(pkg.__name__ + "._lib")


@pytest.mark.parametrize("misaligned", [False, True])
def test_pack_bf16_layernorm_and_int64_positions(mods, pkg, misaligned):
    ops, _ = mods
    g = torch.Generator().manual_seed(1)
    geom = pkg.Geometry(2, 70, 5)
    qkv = torch.randn(geom.tokens, 3 * 128, generator=g).to(torch.bfloat16).to(DEV)
    buf = torch.randn(4, 72, generator=g).to(torch.bfloat16).to(DEV)
    off = 1 if misaligned else 0  # parameters off their 16-byte alignment take fp32 copies
    ln = [buf[i, off:off + 64] for i in range(4)]
    pos = torch.randint(0, 9, (geom.tokens, 2), generator=g).to(DEV)
    assert pos.dtype == torch.int64

    def pack(ln, pos):
        return ops.pack_qkv(qkv, qkv[:, 128:], qkv[:, 256:], 384, 64, geom, 2, ln_q=ln[:2], ln_k=ln[2:], pos=pos,
                            rope_base=100.0, rope_positions=9, fp32_heads=[True, False])
    for a, b in zip(pack(ln, pos), pack([t.float() for t in ln], pos.int())):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))


def test_key_sets_from_host_lists(mods, pkg):
    ops, L = mods
    lib = L.load()
    g = torch.Generator().manual_seed(2)
    geom = pkg.Geometry(3, 155, 5)
    N = geom.tokens
    qk32 = torch.randn(3, 2, N, 64, generator=g).to(DEV)
    _, want = ops.probe_scores(qk32, [2, 0], noalloc=True)  # device lists
    out = torch.full((4, N), -1.0, device=DEV)
    ops.probe_scores(qk32, [2, 0], out=out, rows=[3, 1])
    assert torch.equal(out[[3, 1]], want) and (out[[0, 2]] == -1).all()
    specs = [ops.KeySetSpec(1, ops.KEYSET_STRIDE, 7, 3, True), ops.KeySetSpec(0, ops.KEYSET_TOPK, 40),
             ops.KeySetSpec(2, ops.KEYSET_STRIDE, 4), ops.KeySetSpec(1, ops.KEYSET_TOPK, 11, 0, True)]
    idx, count = ops.keyset_build(specs, geom, out, DEV)
    arr = torch.tensor([[s.mode for s in specs], [s.param for s in specs], [s.start for s in specs],
                        [int(s.include) for s in specs]], dtype=torch.int32, device=DEV)
    idx2, count2 = torch.empty_like(idx), torch.empty_like(count)
    L.check(lib.saf3r_keyset_build(out.data_ptr(), N, 4, *[arr[i].data_ptr() for i in range(4)], 3, 155, 5,
                                   idx2.data_ptr(), N, count2.data_ptr(), L.stream_ptr()))
    assert torch.equal(count, count2)
    for a, b, n in zip(idx, idx2, count.tolist()):
        assert torch.equal(a[:n], b[:n])
    many = (ctypes.c_int32 * 65)(*([0] * 65))
    assert lib.saf3r_keyset_build_host(out.data_ptr(), N, 65, many, many, many, many, 3, 155, 5, idx2.data_ptr(), N,
                                       count2.data_ptr(), L.stream_ptr()) == 2
