"""Attention where the launch cuts a tile's walk into pieces (fp32 partial accumulators, summed by a second kernel), and over
chunk lists whose chunks end inside a key tile: against an fp32 reference, in every form the epilogues have (plain, merged
into a running result, accumulated into fp32 sums, rounded totals)."""
import ctypes
import math

import pytest
import torch

from oracle import layers as OL
from test_attention_plans import dkdv_plan, plan
from test_gpu_sweep import reference, rel_l2

pytestmark = pytest.mark.gpu


def inputs(device, B, Hq, Hkv, Sq, Sk, D):
    g = torch.Generator(device="cuda").manual_seed(Sq + 7 * Sk + D)
    make = lambda *s: torch.randn(*s, generator=g, device=device).to(torch.bfloat16)  # noqa: E731
    return make(B, Hq, Sq, D), make(B, Hkv, Sk, D), make(B, Hkv, Sk, D), make(B, Hq, Sq, D)


def check(got, want, what):
    out, lse, dq, dk, dv = got
    w_out, w_lse, w_dq, w_dk, w_dv = want
    assert (out.float() - w_out).abs().max().item() <= 2e-2, what
    assert torch.equal(torch.isinf(lse), torch.isinf(w_lse)), what
    assert (lse - w_lse).masked_fill(torch.isinf(w_lse), 0.0).abs().max().item() <= 1e-3, what
    for a, b, name in ((dq, w_dq, "dq"), (dk, w_dk, "dk"), (dv, w_dv, "dv")):
        assert rel_l2(a, b) <= 1e-2, (what, name)


# B, Hq, Hkv, Sq, Sk, D, causal, q_offset, cut (forward, backward): whether the launches are expected to cut
CASES = [
    (1, 1, 1, 4000, 4000, 64, True, 0, (True, True)),       # one head, ragged
    (1, 8, 2, 2048, 2048, 64, True, 0, (False, True)),       # GQA
    (2, 9, 3, 1057, 1057, 64, True, 0, (False, True)),
    (2, 32, 8, 1531, 1531, 128, True, 0, (False, True)),     # head_dim 128, ragged, GQA
    (1, 12, 4, 3000, 3000, 128, True, 0, (True, True)),
    (1, 2, 2, 300, 5001, 64, False, 0, (True, True)),       # few queries, many keys, no mask
    (1, 2, 1, 5001, 300, 128, False, 0, (False, True)),      # the other way round
    (1, 2, 2, 2100, 2500, 128, True, 400, (True, True)),    # shifted diagonal
    (1, 2, 2, 5100, 3500, 64, True, 0, (True, True)),       # keys end before the last queries
    (1, 2, 2, 40, 40, 64, True, 0, (False, False)),         # one tile: nothing to cut
]


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Sk,D,causal,q_offset,cut", CASES)
def test_attention_in_pieces(device, B, Hq, Hkv, Sq, Sk, D, causal, q_offset, cut):
    from picotron_amd import _lib, ops
    q, k, v, do = inputs(device, B, Hq, Hkv, Sq, Sk, D)
    scale = 1 / math.sqrt(D)
    d = ops._desc(q, k, v, q, scale, causal, q_offset)
    for need, expected in zip((_lib.lib().pico_attn_fwd_workspace_bytes(ctypes.byref(d), 1),
                               _lib.lib().pico_attn_bwd_workspace_bytes(ctypes.byref(d), 1)), cut):
        assert (need > 0) == expected
    want = reference(q, k, v, scale, q_offset, causal, do)

    out, lse = ops.attn_fwd(q, k, v, scale, causal, q_offset)
    dq, dk, dv = (torch.empty_like(t) for t in (q, k, v))
    ops.attn_bwd(do, q, k, v, lse, None, scale, causal, q_offset, dq=dq, dk=dk, dv=dv, out=out)
    check((out, lse, dq, dk, dv), want, "bf16 results")

    # a second half of the keys merged into the first half's running result; sums accumulated in fp32
    if not causal:
        h = Sk // 2
        o32, l32 = ops.attn_fwd(q, k[:, :, :h].contiguous(), v[:, :, :h].contiguous(), scale, False, out_dtype=torch.float32)
        ops.attn_fwd(q, k[:, :, h:].contiguous(), v[:, :, h:].contiguous(), scale, False, out=o32, lse=l32, merge=True)
        assert (o32 - want[0]).abs().max().item() <= 2e-2 and (l32 - want[1]).abs().max().item() <= 1e-3
    base = [torch.randn(t.shape, device=device, generator=torch.Generator(device="cuda").manual_seed(5)) for t in (q, k, v)]
    sums = [t.clone() for t in base]
    ops.attn_bwd(do, q, k, v, lse, None, scale, causal, q_offset, dq=sums[0], dk=sums[1], dv=sums[2], dq_accumulate=True,
                 dkv_accumulate=True, out=out)
    check((out, lse, *(s - b for s, b in zip(sums, base))), want, "accumulated")
    # the launches of one call on two inputs in a row share nothing: same inputs, same bits
    again, lse2 = ops.attn_fwd(q, k, v, scale, causal, q_offset)
    assert torch.equal(out, again) and torch.equal(lse, lse2)


# B, Hq, Hkv, chunks, chunk length, D, causal
RAGGED = [(1, 4, 2, 3, 65, 64, True), (1, 2, 2, 4, 113, 128, True), (2, 4, 4, 2, 174, 64, False), (1, 2, 1, 16, 200, 128, True),
          (1, 8, 2, 4, 1000, 64, True), (1, 2, 2, 5, 127, 64, True), (2, 32, 32, 3, 129, 64, True)]


@pytest.mark.parametrize("B,Hq,Hkv,W,Sc,D,causal", RAGGED)
def test_ragged_chunk_lists(device, B, Hq, Hkv, W, Sc, D, causal):
    """The last rank of a ring whose chunk length is no multiple of a key tile, RoPE inside, dk / dv both as accumulated fp32
    sums and as totals rounded to bf16."""
    from picotron_amd import ops
    S, off, scale = W * Sc, (W - 1) * Sc, 1 / math.sqrt(D)
    _, k, v, _ = inputs(device, B, Hq, Hkv, Sc, S, D)
    q, _, _, do = inputs(device, B, Hq, Hkv, Sc, Sc, D)
    cos, sin = (t.to(device) for t in OL.get_cos_sin(S, D, 10000.0, torch.float32))
    k_rot = ops.rope(k, cos, sin)
    q_rot_want = ops.rope(q, cos, sin, pos_offset=off)
    w_out, w_lse, w_dq, w_dk, w_dv = reference(q_rot_want, k_rot, v, scale, off, causal, do)
    turn_back = lambda t, o: ops.rope(t.to(torch.bfloat16), cos, -sin, pos_offset=o).float()  # noqa: E731
    want = (w_out, w_lse, turn_back(w_dq, off), turn_back(w_dk, 0), w_dv)

    ks, vs = ([c.contiguous() for c in t.chunk(W, dim=2)] for t in (k_rot, v))
    assert ops.chunks_fit_one_launch(ks, vs)
    out, lse, q_rot = ops.attn_fwd_chunks(q, ks, vs, scale, causal, off, rope=(cos, sin), q_pos_offset=off, want_q_rot=True)
    assert rel_l2(q_rot.float(), q_rot_want.float()) <= 2e-3
    base = [torch.randn(B, Hkv, Sc, D, device=device) for _ in range(2 * W)]
    sums = [t.clone() for t in base]
    finals = [torch.empty(B, Hkv, Sc, D, dtype=torch.bfloat16, device=device) for _ in range(2 * W)]
    dq = torch.empty(q.shape, dtype=torch.float32, device=device)
    for final in (None, finals):             # the second call adds the block once more to the sums the first one left
        ops.attn_bwd_chunks(do, q_rot, ks, vs, lse, scale, causal, off, dq, sums[:W], sums[W:], dkv_accumulate=[True] * W, out=out,
                            rope=(cos, sin), q_pos_offset=off, dk_finals=final and final[:W], dv_finals=final and final[W:])
    added = [s - b for s, b in zip(sums, base)]
    check((out, lse, dq, torch.cat(added[:W], 2), torch.cat(added[W:], 2)), want, "accumulated")
    totals = [2 * w + torch.cat(b, 2) for w, b in ((want[3], base[:W]), (want[4], base[W:]))]
    for got, total in zip((torch.cat(finals[:W], 2), torch.cat(finals[W:], 2)), totals):
        assert rel_l2(got.float(), total) <= 1e-2


# B, Hq, Hkv, Sq, Sk, causal, q_offset: edges of the 64-key tiles and 128-query trips that launches of few workgroups take
@pytest.mark.parametrize("B,Hq,Hkv,Sq,Sk,causal,q_offset", [(1, 9, 3, 1, 1, True, 0), (1, 4, 2, 63, 65, False, 0), (2, 9, 3, 128, 128, True, 0),
                                                            (1, 4, 2, 129, 257, True, 128), (1, 2, 2, 300, 100, True, 0),
                                                            (1, 3, 1, 127, 64, False, 0), (4, 32, 32, 96, 96, True, 0)])
def test_short_chains(device, B, Hq, Hkv, Sq, Sk, causal, q_offset):
    test_attention_in_pieces(device, B, Hq, Hkv, Sq, Sk, 64, causal, q_offset, (False, False))


# the backward kernels' orders of work: masked and unmasked trips, offsets of the diagonal that are no multiple of a tile, no mask at all
@pytest.mark.parametrize("B,Hq,Hkv,Sq,Sk,D,causal,q_offset", [
    (2, 9, 3, 256, 256, 64, False, 0),       # few workgroups, every key visible
    (1, 4, 4, 97, 161, 64, True, 31),        # few workgroups, queries behind the keys' start
    (1, 4, 4, 130, 700, 64, True, 570),      # split keys: all tiles but the last unmasked
    (2, 6, 2, 333, 333, 64, True, 0),
    (1, 4, 2, 200, 641, 128, True, 441),
    (1, 4, 2, 289, 400, 128, True, 111),     # diagonal through tiles, keys that end inside one
    (1, 2, 2, 500, 300, 128, True, 0),       # queries past all keys
    (1, 3, 3, 65, 193, 128, False, 0),
])
def test_backward_masked_and_unmasked_trips(device, B, Hq, Hkv, Sq, Sk, D, causal, q_offset):
    from picotron_amd import ops
    q, k, v, do = inputs(device, B, Hq, Hkv, Sq, Sk, D)
    scale = 1 / math.sqrt(D)
    want = reference(q, k, v, scale, q_offset, causal, do)
    out, lse = ops.attn_fwd(q, k, v, scale, causal, q_offset)
    dq, dk, dv = (torch.empty_like(t) for t in (q, k, v))
    ops.attn_bwd(do, q, k, v, lse, None, scale, causal, q_offset, dq=dq, dk=dk, dv=dv, out=out)
    check((out, lse, dq, dk, dv), want, "bf16 results")   # (bf16 operands and probabilities: the bounds of the tests above)


# chunks of several whole key tiles and a partial one: dQ's masked and unmasked trips follow each other chunk after chunk, in every kernel
@pytest.mark.parametrize("B,Hq,Hkv,Sq,W,Sc,D,causal,q_offset", [
    (1, 4, 2, 300, 3, 449, 64, False, 0),       # split keys, four waves, cut
    (1, 4, 2, 300, 3, 449, 64, True, 700),
    (2, 32, 8, 512, 2, 833, 64, True, 1154),    # split keys, eight waves
    (8, 32, 32, 768, 3, 257, 64, True, 3),      # four waves
    (4, 32, 32, 1024, 2, 577, 64, True, 130),   # eight waves
    (1, 4, 2, 300, 3, 449, 128, True, 1047),    # four waves, cut
    (1, 4, 2, 300, 4, 191, 128, False, 0),
    (8, 32, 8, 512, 2, 353, 128, True, 194),    # eight waves
])
def test_backward_over_chunks_that_end_inside_tiles(device, B, Hq, Hkv, Sq, W, Sc, D, causal, q_offset):
    from picotron_amd import ops
    q, k, v, do = inputs(device, B, Hq, Hkv, Sq, W * Sc, D)
    scale = 1 / math.sqrt(D)
    ks, vs = ([c.contiguous() for c in t.chunk(W, dim=2)] for t in (k, v))
    out, lse, _ = ops.attn_fwd_chunks(q, ks, vs, scale, causal, q_offset)
    dq, dks, dvs = torch.empty_like(q), [torch.empty_like(t) for t in ks], [torch.empty_like(t) for t in vs]
    ops.attn_bwd_chunks(do, q, ks, vs, lse, scale, causal, q_offset, dq=dq, dks=dks, dvs=dvs, out=out)
    for b in range(0, B, 5):
        for h in range(0, Hkv, 7):
            part, kv = slice(h * Hq // Hkv, (h + 1) * Hq // Hkv), slice(h, h + 1)
            got = (out[b:b + 1, part], lse[b:b + 1, part], dq[b:b + 1, part], torch.cat(dks, 2)[b:b + 1, kv], torch.cat(dvs, 2)[b:b + 1, kv])
            check(got, reference(q[b:b + 1, part], k[b:b + 1, kv], v[b:b + 1, kv], scale, q_offset, causal, do[b:b + 1, part]), (b, h))


# head_dim 128: workgroups of four waves below, at and above the lines to those of eight (in workgroups of 256 queries)
@pytest.mark.parametrize("B,Hq,Hkv,Sq,Sk,causal,q_offset,waves", [
    (1, 32, 8, 2048, 2048, True, 0, 4),      # 256, causal
    (1, 32, 8, 2048, 2048, False, 0, 8),     # 256 equal ones
    (8, 32, 8, 257, 257, True, 0, 4),        # 512, nearly half of them padding
    (8, 11, 11, 901, 901, True, 0, 4),       # 352
    (8, 32, 8, 385, 385, True, 0, 8),        # 512 without padding
    (6, 30, 10, 640, 1280, True, 640, 4),    # 540 equal ones, a sixth of them padding
    (6, 30, 10, 768, 1536, True, 768, 4),    # 540 equal ones without padding
    (6, 30, 10, 768, 768, True, 0, 8),       # 540
    (33, 32, 8, 100, 100, True, 0, 4),       # one workgroup to a head either way
])
def test_forward_on_both_sides_of_the_lines_at_head_dim_128(device, B, Hq, Hkv, Sq, Sk, causal, q_offset, waves):
    """The whole launch equals launches of one batch and kv head at a time (always four waves) element by element to the rounding of
    bf16, and the fp32 reference in every 64 rows."""
    from picotron_amd import ops
    assert plan("fwd", B, Hq, Sq, Sk, causal, q_offset, Hkv=Hkv)[0] == waves
    q, k, v, do = inputs(device, B, Hq, Hkv, Sq, Sk, 128)
    scale, group = 1 / math.sqrt(128), Hq // Hkv
    out, lse = ops.attn_fwd(q, k, v, scale, causal, q_offset)
    for b in range(0, B, 5):
        for h in range(0, Hkv, 7):
            part = slice(h * group, (h + 1) * group)
            o, l = ops.attn_fwd(q[b:b + 1, part], k[b:b + 1, h:h + 1], v[b:b + 1, h:h + 1], scale, causal, q_offset)
            whole = out[b:b + 1, part]
            # one unit in the last place of bf16 (2^-7 of the value at most); a launch that is cut rounds its probabilities against another
            # maximum: 2^-9 / sqrt(3) of the row's root mean square on each side, 1.6e-3 together, of which 2^-6 is ten times
            a, b_ = o.float(), whole.float()
            assert ((a - b_).abs() <= 2 ** -7 * torch.maximum(a.abs(), b_.abs()) + 2 ** -6 * b_.square().mean(-1, keepdim=True).sqrt()).all(), (b, h)
            assert (l - lse[b:b + 1, part]).abs().max().item() <= 1e-5 * max(1.0, lse.abs().max().item())
            # rounded probabilities and rounded results, each 1.1e-3 of a row's norm
            want = reference(q[b:b + 1, part], k[b:b + 1, h:h + 1], v[b:b + 1, h:h + 1], scale, q_offset, causal, do[b:b + 1, part])[0]
            for r in range(0, Sq, 64):
                assert rel_l2(whole[:, :, r:r + 64], want[:, :, r:r + 64]) <= 4e-3, (b, h, r)


# dQ at head_dim 128 on both sides of its lines (in workgroups of 256 queries), alone: no other gradient is asked for
@pytest.mark.parametrize("B,Hq,Hkv,Sq,Sk,causal,q_offset,waves", [
    (1, 32, 8, 2048, 2048, False, 0, 8),     # 256 equal ones
    (8, 32, 8, 257, 257, True, 0, 4),        # 512, nearly half of them padding
    (8, 24, 8, 511, 511, True, 0, 4),        # 384
    (7, 29, 29, 385, 385, True, 0, 8),       # 406
    (6, 32, 8, 640, 900, True, 130, 4),      # 576, a sixth of them padding
    (6, 30, 10, 768, 900, True, 130, 4),     # 540 without padding
    (33, 32, 8, 100, 100, True, 0, 4),       # one workgroup to a head either way
])
def test_dq_on_both_sides_of_the_lines_at_head_dim_128(device, B, Hq, Hkv, Sq, Sk, causal, q_offset, waves):
    """Against the fp32 reference of a batch and kv head at a time, with the bound of bf16 operands that the tests above have."""
    from picotron_amd import ops
    assert plan("dq", B, Hq, Sq, Sk, causal, q_offset, Hkv=Hkv)[0] == waves
    q, k, v, do = inputs(device, B, Hq, Hkv, Sq, Sk, 128)
    scale, group = 1 / math.sqrt(128), Hq // Hkv
    out, lse = ops.attn_fwd(q, k, v, scale, causal, q_offset)
    dq = torch.empty_like(q)
    ops.attn_bwd_chunks(do, q, [k], [v], lse, scale, causal, q_offset, dq=dq, dks=[None], dvs=[None], out=out)
    for b in range(0, B, 5):
        for h in range(0, Hkv, 7):
            part = slice(h * group, (h + 1) * group)
            want = reference(q[b:b + 1, part], k[b:b + 1, h:h + 1], v[b:b + 1, h:h + 1], scale, q_offset, causal, do[b:b + 1, part])
            assert rel_l2(dq[b:b + 1, part], want[2]) <= 1e-2, (b, h)


# head_dim 128: gradients of rotated q and k, added to what is there, of eight and of four waves
@pytest.mark.parametrize("B,Hq,Hkv,S,waves", [(8, 16, 16, 1000, 8), (11, 32, 16, 417, 8), (1, 4, 2, 300, 4)])
def test_gradients_leave_unrotated_and_added_at_head_dim_128(device, B, Hq, Hkv, S, waves):
    """The rotation's backward and the sum in the kernels' epilogues equal the two on their fp32 results: eight roundings of products of
    two elements of a pair, and the sum's."""
    from picotron_amd import ops
    assert plan("dq", B, Hq, S, S, True, 0, Hkv=Hkv)[0] == waves
    q, k, v, do = inputs(device, B, Hq, Hkv, S, S, 128)
    scale = 1 / math.sqrt(128)
    cos, sin = (t.to(device) for t in OL.get_cos_sin(S + 5, 128, 10000.0, torch.float32))
    out, lse = ops.attn_fwd(q, k, v, scale, True, 0)
    plain = ops.attn_bwd(do, q, k, v, lse, None, scale, True, 0, out=out)
    g = torch.Generator(device="cuda").manual_seed(3)
    bases = [torch.randn(t.shape, generator=g, device=device) for t in plain]
    got = [t.clone() for t in bases]
    ops.attn_bwd_rope(do, q, k, v, out, lse, cos, sin, scale, True, *got, 0, q_pos_offset=5, k_pos_offset=5, dq_accumulate=True, dkv_accumulate=True)
    c, s = cos[5:5 + S, :64], sin[5:5 + S, :64]
    for i, (a, b, base) in enumerate(zip(got, plain, bases)):
        lo, hi = b[..., :64], b[..., 64:]
        turned = b if i == 2 else torch.cat((lo * c + hi * s, hi * c - lo * s), -1)
        size = (lo.abs() + hi.abs()).repeat(1, 1, 1, 2) + base.abs()
        assert ((a - (base + turned)).abs() <= 9 * 2 ** -24 * size).all(), i


# dK/dV at head_dim 128 in key tiles of 256, whose waves have dV or dK of 64 keys, 16 of every 64
@pytest.mark.parametrize("B,Hq,Hkv,Sq,W,Sc,causal,q_offset", [
    (8, 32, 32, 97, 1, 129, False, 0),       # keys that end in the third block of 64 of some waves and the second of others
    (8, 32, 32, 200, 1, 193, False, 0),
    (8, 32, 32, 256, 1, 256, False, 0),
    (3, 32, 32, 777, 1, 777, True, 0),       # every number of blocks on the diagonal, ragged ends of both
    (4, 16, 16, 922, 1, 922, False, 0),
    (8, 32, 32, 128, 1, 512, True, 384),     # queries behind the keys
    (16, 16, 8, 300, 1, 520, True, 219),     # two query heads to a walk, a diagonal that no block begins on
    (16, 32, 16, 150, 1, 200, False, 0),
    (13, 20, 10, 520, 1, 600, True, 80),
    (8, 32, 8, 257, 2, 449, True, 641),      # chunks that end inside key tiles
])
def test_key_tiles_of_256(device, B, Hq, Hkv, Sq, W, Sc, causal, q_offset):
    """Gradients against the fp32 reference of a batch and kv head at a time, with the bound of bf16 operands; then the forms that a
    chunk's gradients leave in: added to fp32 sums, their rounded total, not at all."""
    from picotron_amd import ops
    assert dkdv_plan(B, Hq, Sq, W * Sc, causal, q_offset, Hkv=Hkv, chunks=W)[0] == 256
    q, k, v, do = inputs(device, B, Hq, Hkv, Sq, W * Sc, 128)
    scale, group = 1 / math.sqrt(128), Hq // Hkv
    ks, vs = ([c.contiguous() for c in t.chunk(W, dim=2)] for t in (k, v))
    out, lse, _ = ops.attn_fwd_chunks(q, ks, vs, scale, causal, q_offset)

    def run(make, **more):
        dks, dvs = [make() for _ in range(W)], [make() for _ in range(W)]
        ops.attn_bwd_chunks(do, q, ks, vs, lse, scale, causal, q_offset, dks=dks, dvs=dvs, out=out, **more)
        return dks, dvs

    dks, dvs = run(lambda: torch.full_like(ks[0], float("nan"), dtype=torch.float32))
    for b in range(0, B, 5):
        for h in range(0, Hkv, 7):
            part = slice(h * group, (h + 1) * group)
            want = reference(q[b:b + 1, part], k[b:b + 1, h:h + 1], v[b:b + 1, h:h + 1], scale, q_offset, causal, do[b:b + 1, part])
            for got, w in ((torch.cat(dks, 2), want[3]), (torch.cat(dvs, 2), want[4])):
                assert rel_l2(got[b:b + 1, h:h + 1], w) <= 1e-2, (b, h)
                for r in range(0, W * Sc, 64):
                    assert rel_l2(got[b:b + 1, h:h + 1, r:r + 64], w[:, :, r:r + 64]) <= 2e-2 or w[:, :, r:r + 64].norm() < 0.05 * w.norm(), (b, h, r)
    base = torch.randn(ks[0].shape, generator=torch.Generator(device="cuda").manual_seed(1), device=device)
    added = run(base.clone, dkv_accumulate=[True] * W)
    for got, one in zip(added[0] + added[1], dks + dvs):
        assert torch.equal(got, base + one)
    totals = [torch.empty_like(t) for t in ks], [torch.empty_like(t) for t in ks]
    kept = run(base.clone, dkv_accumulate=[True] * W, dk_finals=totals[0], dv_finals=totals[1])
    for total, got, read in zip(totals[0] + totals[1], added[0] + added[1], kept[0] + kept[1]):
        assert torch.equal(total, got.to(torch.bfloat16)) and torch.equal(read, base)
    rounded = run(lambda: torch.empty_like(ks[0]))
    for got, one in zip(rounded[0] + rounded[1], dks + dvs):
        assert torch.equal(got, one.to(torch.bfloat16))
    if W > 1:
        some = [None, torch.empty_like(dks[1])], [None, torch.empty_like(dks[1])]
        ops.attn_bwd_chunks(do, q, ks, vs, lse, scale, causal, q_offset, dks=some[0], dvs=some[1], out=out)
        assert torch.equal(some[0][1], dks[1]) and torch.equal(some[1][1], dvs[1])


# ... whose last tiles have 9, 76 and 200 rows: ends in a wave's first, second and fourth block of 16, the rows n and n + 64 that leave together
@pytest.mark.parametrize("B,Hq,Hkv,S,waves", [(3, 32, 32, 777, 4), (5, 16, 16, 1100, 4), (6, 16, 16, 968, 4), (8, 32, 16, 712, 8)])
def test_gradients_leave_unrotated_and_added_in_key_tiles_of_256(device, B, Hq, Hkv, S, waves):
    assert dkdv_plan(B, Hq, S, S, True, 0, Hkv=Hkv) == (256, 1, 0)
    test_gradients_leave_unrotated_and_added_at_head_dim_128(device, B, Hq, Hkv, S, waves)


def test_chunks_in_key_tiles_of_256_leave_unrotated(device):
    """Chunks that end inside key tiles: the rotation's backward on the fp32 results (eight roundings of products of two elements of a pair, and
    the sum's), and the rounded totals are those sums rounded."""
    from picotron_amd import ops
    B, Hq, Hkv, Sq, W, Sc, offset, k_first = 8, 32, 8, 257, 2, 449, 641, 7
    assert dkdv_plan(B, Hq, Sq, W * Sc, True, offset, Hkv=Hkv, chunks=W) == (256, 1, 0)
    q, k, v, do = inputs(device, B, Hq, Hkv, Sq, W * Sc, 128)
    scale = 1 / math.sqrt(128)
    ks, vs = ([c.contiguous() for c in t.chunk(W, dim=2)] for t in (k, v))
    cos, sin = (t.to(device) for t in OL.get_cos_sin(W * Sc + k_first, 128, 10000.0, torch.float32))
    out, lse, _ = ops.attn_fwd_chunks(q, ks, vs, scale, True, offset)

    def run(make, **more):
        dks, dvs = [make() for _ in range(W)], [make() for _ in range(W)]
        ops.attn_bwd_chunks(do, q, ks, vs, lse, scale, True, offset, dks=dks, dvs=dvs, out=out, **more)
        return dks, dvs

    plain = run(lambda: torch.empty(ks[0].shape, device=device))
    base = torch.randn(ks[0].shape, generator=torch.Generator(device="cuda").manual_seed(1), device=device)
    turning = dict(rope=(cos, sin), q_pos_offset=offset, k_pos_offset=k_first, dkv_accumulate=[True] * W)
    added = run(base.clone, **turning)
    for c in range(W):
        at = slice(k_first + c * Sc, k_first + (c + 1) * Sc)
        lo, hi = plain[0][c][..., :64], plain[0][c][..., 64:]
        turned = torch.cat((lo * cos[at, :64] + hi * sin[at, :64], hi * cos[at, :64] - lo * sin[at, :64]), -1)
        size = (lo.abs() + hi.abs()).repeat(1, 1, 1, 2) + base.abs()
        assert ((added[0][c] - (base + turned)).abs() <= 9 * 2 ** -24 * size).all(), c
        assert torch.equal(added[1][c], base + plain[1][c]), c
    totals = [torch.empty_like(t) for t in ks], [torch.empty_like(t) for t in ks]
    run(base.clone, dk_finals=totals[0], dv_finals=totals[1], **turning)
    for total, got in zip(totals[0] + totals[1], added[0] + added[1]):
        assert torch.equal(total, got.to(torch.bfloat16))


def test_key_tiles_of_256_that_no_query_sees(device):
    """Nine of them, and the last blocks of the one before: zeros where the gradients are written, what was there where they are added; the others against
    the fp32 reference."""
    from picotron_amd import ops
    B, H, Sq, Sk, q_offset = 8, 8, 1201, 3782, 100
    assert dkdv_plan(B, H, Sq, Sk, True, q_offset) == (256, 1, 0)
    q, k, v, do = inputs(device, B, H, H, Sq, Sk, 128)
    scale, seen = 1 / math.sqrt(128), q_offset + Sq
    out, lse = ops.attn_fwd(q, k, v, scale, True, q_offset)
    dk, dv = (torch.full(k.shape, float("nan"), device=device) for _ in range(2))
    dq, _, _ = ops.attn_bwd(do, q, k, v, lse, None, scale, True, q_offset, None, dk, dv, out=out)
    assert (dk[:, :, seen:] == 0).all() and (dv[:, :, seen:] == 0).all()
    for b, h in ((0, 0), (B // 2, H - 1), (B - 1, 3)):
        want = reference(*(t[b:b + 1, h:h + 1] for t in (q, k, v)), scale, q_offset, True, do[b:b + 1, h:h + 1])
        for got, w in ((dq, want[2]), (dk, want[3]), (dv, want[4])):
            assert rel_l2(got[b:b + 1, h:h + 1], w) <= 1e-2, (b, h)
    base = torch.randn(k.shape, generator=torch.Generator(device="cuda").manual_seed(1), device=device)
    added = base.clone(), base.clone()
    ops.attn_bwd(do, q, k, v, lse, None, scale, True, q_offset, None, *added, out=out, dkv_accumulate=True)
    assert torch.equal(added[0], base + dk) and torch.equal(added[1], base + dv)


def test_rows_without_keys_in_key_tiles_of_256(device):
    """Rows whose lse is -inf add nothing, as rows without a gradient do: bit for bit."""
    from picotron_amd import ops
    B, H, S = 3, 32, 777
    assert dkdv_plan(B, H, S, S, True, 0) == (256, 1, 0)
    q, k, v, do = inputs(device, B, H, H, S, S, 128)
    scale = 1 / math.sqrt(128)
    out, lse = ops.attn_fwd(q, k, v, scale, True, 0)
    rows = torch.zeros(S, dtype=torch.bool, device=device)
    rows[[0, 31, 776]] = True
    rows[100:175] = True
    got = ops.attn_bwd(do, q, k, v, lse.masked_fill(rows, -math.inf), None, scale, True, 0, out=out)
    want = ops.attn_bwd(do.masked_fill(rows[:, None], 0.0), q, k, v, lse, None, scale, True, 0, out=out)
    for x, y in zip(got, want):
        assert torch.equal(x, y)


def test_a_batch_and_its_halves_at_head_dim_128(device):
    """The whole batch and its halves go to other kernels of dQ and of dK/dV, whose sums of 128 products have other orders: they differ by under 2^-17 of
    themselves, so that at most one value of P and dS in 2^9 is rounded to bf16 the other way, by at most 2^-7 of it: 2^-11.5 in rel. L2."""
    from picotron_amd import ops
    B, H, S = 8, 32, 1100
    assert plan("dq", B, H, S, S, True, 0)[0] == 8 and plan("dq", B // 2, H, S, S, True, 0)[0] == 4
    assert dkdv_plan(B, H, S, S, True, 0) == (128, 2, 0) and dkdv_plan(B // 2, H, S, S, True, 0) == (256, 1, 0)
    q, k, v, do = inputs(device, B, H, H, S, S, 128)
    scale = 1 / math.sqrt(128)
    out, lse = ops.attn_fwd(q, k, v, scale, True, 0)
    whole = ops.attn_bwd(do, q, k, v, lse, None, scale, True, 0, out=out)
    for half in (slice(0, B // 2), slice(B // 2, B)):
        part = ops.attn_bwd(do[half], q[half], k[half], v[half], lse[half], None, scale, True, 0, out=out[half])
        for x, y in zip(whole, part):
            assert rel_l2(y, x[half]) <= 2 ** -11.5


# dQ of eight waves at head_dim 128 in pieces: 264 and 288 workgroups, over a round of one per CU, beside over 8192 keys
@pytest.mark.parametrize("B,Hq,Hkv,Sq,W,Sc,q_offset", [(11, 12, 1, 274, 2, 4199, 8124), (9, 16, 1, 262, 1, 8413, 8151)])
def test_dq_of_eight_waves_in_pieces_at_head_dim_128(device, B, Hq, Hkv, Sq, W, Sc, q_offset):
    """Against the fp32 reference of a batch at a time, with the bound of bf16 operands; un-rotated and added, equal to the two on that result: eight
    roundings of products of two elements of a pair, and the sum's."""
    from picotron_amd import _lib, ops
    q, k, v, do = inputs(device, B, Hq, Hkv, Sq, W * Sc, 128)
    scale = 1 / math.sqrt(128)
    ks, vs = ([c.contiguous() for c in t.chunk(W, dim=2)] for t in (k, v))
    how = (ctypes.c_int32 * 3)()
    _lib.check(_lib.lib().pico_attn_dq_plan(ctypes.byref(ops._chunk_desc(q, ks, vs, q, scale, True, q_offset)), W, how))
    assert how[0] == 8 and how[2] > 0
    out, lse, _ = ops.attn_fwd_chunks(q, ks, vs, scale, True, q_offset)
    dq = torch.full(q.shape, float("nan"), device=device)
    ops.attn_bwd_chunks(do, q, ks, vs, lse, scale, True, q_offset, dq=dq, dks=[None] * W, dvs=[None] * W, out=out)
    for b in (0, B // 2, B - 1):
        want = reference(*(t[b:b + 1] for t in (q, k, v)), scale, q_offset, True, do[b:b + 1])[2]
        for r in range(0, Sq, 32):
            assert rel_l2(dq[b:b + 1, :, r:r + 32], want[:, :, r:r + 32]) <= 1e-2, (b, r)
    cos, sin = (t.to(device) for t in OL.get_cos_sin(W * Sc + 5, 128, 10000.0, torch.float32))
    base = torch.randn(q.shape, generator=torch.Generator(device="cuda").manual_seed(3), device=device)
    got = base.clone()
    ops.attn_bwd_chunks(do, q, ks, vs, lse, scale, True, q_offset, dq=got, dks=[None] * W, dvs=[None] * W, out=out, rope=(cos, sin), q_pos_offset=5, dq_accumulate=True)
    c, s, lo, hi = cos[5:5 + Sq, :64], sin[5:5 + Sq, :64], dq[..., :64], dq[..., 64:]
    size = (lo.abs() + hi.abs()).repeat(1, 1, 1, 2) + base.abs()
    assert ((got - (base + torch.cat((lo * c + hi * s, hi * c - lo * s), -1))).abs() <= 9 * 2 ** -24 * size).all()
