"""Attention launches (512 resident work-groups) in which the walks of every head, or the named ones, run split:
(name, F, T, ns, patterns, split heads). P tiles and special tiles at their partial and full sizes."""
ALL = None
CASES = [
    # framed heads, frames of 24 tiles: 33, 64 (no specials), 1 and 6 valid keys in a frame's last tile
    ("frame_local", 3, 1505, 5, ["FRAME_LOCAL"], ALL),
    ("frame_local_full", 2, 1536, 0, ["FRAME_LOCAL"], ALL),
    ("anchor_one_key", 3, 1473, 0, ["ANCHOR"], ALL),
    ("anchor_local", 3, 1478, 5, ["ANCHOR_LOCAL"], ALL),
    ("frame_local_anchor", 2, 1505, 5, ["FRAME_LOCAL", "ANCHOR"], ALL),
    ("anchor_local_of_three", 2, 1505, 5, ["FRAME_LOCAL", "ANCHOR_LOCAL", "ANCHOR"], ["ANCHOR_LOCAL"]),
    # one special token a frame; S = 70 (two special tiles, the second partial) and S = 128 (two full ones)
    ("ns1", 27, 65, 1, ["DENSE", "DENSE_PACKED", "KEYSET", "BLOCK_DYNAMIC"], ALL),
    ("s70", 14, 133, 5, ["DENSE", "DENSE_PACKED", "KEYSET", "BLOCK_DYNAMIC"], ALL),
    ("s128", 2, 900, 64, ["DENSE", "DENSE_PACKED", "KEYSET", "BLOCK_DYNAMIC"], ALL),
    ("no_specials", 25, 64, 0, ["DENSE", "DENSE_PACKED", "KEYSET"], ALL),
    ("block_dynamic", 5, 453, 3, ["BLOCK_DYNAMIC", "BLOCK_DYNAMIC"], ALL),
    # the special rows of the token-list heads: S = 20, S = 70, one of each frame
    ("token_dynamic", 4, 450, 5, ["TOKEN_DYNAMIC"], ALL),
    ("token_dynamic_s70", 14, 133, 5, ["TOKEN_DYNAMIC", "TOKEN_DYNAMIC_KEYSET"], ALL),
    ("token_dynamic_ns1", 30, 60, 1, ["TOKEN_DYNAMIC", "TOKEN_DYNAMIC_KEYSET"], ALL),
    # launches that fill the chip, and walks beyond the longest that splits (256 tiles), split nothing
    ("full", 4, 1041, 5, ["DENSE"] * 40, []),
    ("long", 13, 1374, 5, ["DENSE"], []),
    ("short", 2, 300, 5, ["DENSE", "KEYSET", "FRAME_LOCAL", "ANCHOR_LOCAL", "BLOCK_DYNAMIC"], []),
]


def case(ops, pkg, name, F, T, ns, kinds, split):
    """(geometry, pattern ids, layouts, expected split heads) of a case."""
    geom = pkg.Geometry(F, T, ns)
    patterns = [ops.DENSE if k == "DENSE_PACKED" else getattr(ops, k) for k in kinds]
    layouts = [ops.LAYOUT_PACKED if k == "DENSE_PACKED" else lay
               for k, lay in zip(kinds, ops.token_order_heads(patterns, geom))]
    want = [h for h, k in enumerate(kinds) if split is None or k in split]
    return geom, patterns, layouts, want


def capacity(geom):
    """Of a key set of every token."""
    return -(-geom.tokens // 64) * 64


def list_width(geom):
    """Of the block lists: two blocks a frame, or its only one."""
    return geom.frames * min(2, geom.blocks_per_frame)


def split_heads(lib, geom, patterns, layouts, compute_units=256):
    import ctypes
    n = len(patterns)
    mask = ctypes.c_uint64(0)
    rc = lib.saf3r_sparse_attn_split_heads(geom.frames, geom.tokens_per_frame, geom.num_special, n,
                                           (ctypes.c_int32 * n)(*patterns), list_width(geom), capacity(geom),
                                           (ctypes.c_uint8 * n)(*layouts), compute_units, ctypes.byref(mask))
    assert rc == 0, lib.saf3r_last_error()
    return [h for h in range(n) if mask.value >> h & 1]
