"""Which kernel an attention launch gets, asked of the library itself: on both sides of every line between workgroups of four and
eight waves at head_dim 128, and where query tiles are cut into pieces.  Needs no GPU."""
import ctypes
import os

import pytest


def plan(which, B, H, Sq, Sk, causal, q_offset, D=128, Hkv=None):
    """(waves per workgroup, waves that share 32 queries, key tiles of a piece)"""
    from picotron_amd import _lib
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("library not built here (python -m picotron_amd.build)")
    d = _lib.AttnDesc()
    d.B, d.Hq, d.Hkv, d.Sq, d.Sk, d.D, d.causal, d.q_offset, d.sm_scale = B, H, Hkv or H, Sq, Sk, D, int(causal), q_offset, D ** -0.5
    out = (ctypes.c_int32 * 3)()
    lib = _lib.lib()
    _lib.check((lib.pico_attn_fwd_plan if which == "fwd" else lib.pico_attn_dq_plan)(ctypes.byref(d), 1, out))
    return tuple(out)


def dkdv_plan(B, H, Sq, Sk, causal, q_offset, D=128, Hkv=None, chunks=1):
    """(keys of a key tile, key tiles of a workgroup, trips of a piece)"""
    from picotron_amd import _lib
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("library not built here (python -m picotron_amd.build)")
    d = _lib.AttnDesc()
    d.B, d.Hq, d.Hkv, d.Sq, d.Sk, d.D, d.causal, d.q_offset, d.sm_scale = B, H, Hkv or H, Sq, Sk, D, int(causal), q_offset, D ** -0.5
    out = (ctypes.c_int32 * 3)()
    _lib.check(_lib.lib().pico_attn_dkdv_plan(ctypes.byref(d), chunks, out))
    return tuple(out)


# (B, H, Sq, Sk, causal, q_offset), workgroups of 256 queries and of 128, waves of the forward, waves of dQ
LINES = [
    ((1, 32, 1792, 1792, True, 0), 224, 448, 4, 4),         # under one round
    ((1, 32, 2048, 2048, True, 0), 256, 512, 4, 4),         # one round, of unequal length
    ((1, 32, 2048, 2048, False, 0), 256, 512, 8, 8),        # one round of equal ones
    ((1, 32, 2048, 4096, True, 2048), 256, 512, 8, 8),
    ((1, 33, 2048, 2048, False, 0), 264, 528, 4, 4),
    ((1, 44, 2048, 2048, True, 0), 352, 704, 4, 4),         # the forward's line behind one round ...
    ((1, 353, 256, 256, True, 0), 353, 706, 8, 4),
    ((1, 48, 2048, 2048, True, 0), 384, 768, 8, 4),         # ... and dQ's
    ((1, 385, 256, 256, True, 0), 385, 770, 8, 8),
    ((1, 64, 2048, 2048, False, 0), 512, 1024, 8, 8),       # two rounds
    ((1, 513, 256, 256, False, 0), 513, 1026, 4, 4),        # just over two: equal ones in the forward, all in dQ
    ((1, 513, 256, 256, True, 0), 513, 1026, 8, 4),
    ((1, 180, 768, 768, False, 0), 540, 1080, 4, 4),
    ((1, 180, 768, 768, True, 0), 540, 1080, 8, 4),
    ((1, 180, 768, 1536, True, 768), 540, 1080, 4, 4),
    ((1, 160, 1024, 1024, False, 0), 640, 1280, 4, 4),
    ((1, 641, 256, 256, False, 0), 641, 1282, 8, 8),
    ((1, 341, 300, 300, True, 0), 682, 1023, 4, 4),         # a tenth of the queries of 256 are not there ...
    ((1, 342, 300, 300, True, 0), 684, 1026, 8, 8),         # ... in many workgroups
    ((1, 100, 1153, 1153, True, 0), 500, 1000, 8, 8),       # narrow = 2 wide: none missing
    ((1, 100, 1100, 1100, True, 0), 500, 900, 4, 4),
    ((33, 32, 128, 128, True, 0), 1056, 1056, 4, 4),        # one workgroup to a head either way
    ((64, 32, 16, 512, True, 496), 2048, 2048, 4, 4),
    ((33, 32, 128, 9000, False, 0), 1056, 1056, 4, 4),
    ((33, 32, 129, 129, True, 0), 1056, 2112, 8, 8),
    ((1, 9, 8192, 8192, True, 0), 288, 576, 4, 4),          # keys past which the tiles' traffic counts
    ((1, 9, 8192, 8193, True, 0), 288, 576, 8, 8),
    ((1, 180, 768, 8193, False, 0), 540, 1080, 8, 8),
    ((1, 8, 4096, 32768, True, 28672), 128, 256, 4, 4),     # (not under one round)
]


@pytest.mark.parametrize("sizes,wide,narrow,fwd,dq", LINES)
def test_waves_at_head_dim_128(sizes, wide, narrow, fwd, dq):
    B, H, Sq = sizes[:3]
    assert (B * H * -(-Sq // 256), B * H * -(-Sq // 128)) == (wide, narrow)
    assert plan("fwd", *sizes)[:2] == (fwd, 1) and plan("dq", *sizes)[:2] == (dq, 1)


@pytest.mark.parametrize("sizes,piece", [
    ((2, 4, 1168, 1168, True, 0), 6),       # us whole and cut: 25.2, 19.0
    ((4, 2, 480, 960, True, 480), 4),       # 20.9, 16.9
    ((1, 4, 877, 877, True, 0), 4),         # 20.2, 17.0
    ((1, 4, 903, 903, False, 0), 6),        # 20.8, 17.4
    ((2, 4, 620, 620, True, 0), 0),         # a walk too short for it
    ((1, 9, 890, 890, True, 0), 0),         # 19.7, 21.2
])
def test_short_walks_of_dq_in_pieces(sizes, piece):
    assert plan("dq", *sizes) == (4, 1, piece)


def test_a_descriptor_without_a_launch_has_no_plan():
    for which in ("fwd", "dq"):
        for sizes in ((0, 4, 64, 64, True, 0), (1, 4, 0, 64, True, 0), (1, 4, 64, 0, True, 0)):
            with pytest.raises(RuntimeError, match="no launch"):
                plan(which, *sizes)
        with pytest.raises(RuntimeError, match="no launch"):
            plan(which, 1, 4, 64, 64, True, 0, D=96)


@pytest.mark.parametrize("sizes,kv_heads,want", [   # us of key tiles of 128 (as planned without the other kernel) and of 256
    ((1, 32, 2048, 2048, False, 0), 32, (256, 1, 0)),       # 129, 111: one round of equal ones
    ((1, 32, 2048, 2048, True, 0), 32, (128, 2, 0)),        # 72, 93: of unequal ones
    ((1, 32, 4096, 4096, True, 0), 32, (256, 1, 0)),        # 243, 220
    ((3, 32, 777, 777, True, 0), 32, (256, 1, 0)),          # 64, 44
    ((1, 32, 1024, 1024, False, 0), 32, (128, 1, 0)),       # 36, 50: half a round
    ((2, 32, 1531, 1531, True, 0), 8, (128, 1, 48)),        # 90, 95 uncut: few workgroups
    ((3, 16, 2769, 2769, False, 0), 16, (128, 1, 0)),       # 383, 396: just over two rounds
    ((4, 32, 1281, 1281, True, 0), 32, (256, 1, 0)),       # (as drawn: 0.85 of the time)
])
def test_key_tiles_at_head_dim_128(sizes, kv_heads, want):
    assert dkdv_plan(*sizes, Hkv=kv_heads) == want


def test_key_tiles_of_128_where_the_estimates_are_close():
    """Both just above the line (0.844): one that the other kernel would slow down, 263 -> 269 us, and one that is compared bit for bit with
    its halves as paired and single key tiles of one kernel."""
    assert dkdv_plan(8, 6, 2057, 2057, False, 0, Hkv=2) == (128, 1, 48)
    assert dkdv_plan(4, 16, 1100, 1100, True, 0) == (128, 2, 0)
    assert dkdv_plan(2, 16, 1100, 1100, True, 0) == (128, 1, 0)
