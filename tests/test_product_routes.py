"""Which projections' products may leave torch, decided from the operands' metadata alone.  The operands are tensors over
addresses that nothing follows, made through DLPack with a device that need not exist, so this runs without a GPU; in a
process of its own, which is told that the device runtime is up."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

OPERANDS = '''
import ctypes
import torch
torch.cuda._lazy_init = lambda: None
i64 = ctypes.c_int64


class DLTensor(ctypes.Structure):
    _fields_ = [("data", ctypes.c_void_p), ("device_type", ctypes.c_int32), ("device_id", ctypes.c_int32), ("ndim", ctypes.c_int32),
                ("code", ctypes.c_uint8), ("bits", ctypes.c_uint8), ("lanes", ctypes.c_uint16), ("shape", ctypes.POINTER(i64)),
                ("strides", ctypes.POINTER(i64)), ("offset", ctypes.c_uint64), ("context", ctypes.c_void_p), ("deleter", ctypes.c_void_p)]


capsule = ctypes.pythonapi.PyCapsule_New
capsule.restype, capsule.argtypes = ctypes.py_object, [ctypes.c_void_p, ctypes.c_char_p, ctypes.c_void_p]
kept = []


def operand(rows, cols, pitch=None, device=0, address=1 << 20):
    """A bf16 [rows, cols] matrix with `pitch` elements between rows."""
    ROCM, BFLOAT = 10, 4
    shape, strides = (i64 * 2)(rows, cols), (i64 * 2)(pitch or cols, 1)
    t = DLTensor(address, ROCM, device, 2, BFLOAT, 16, 1, shape, strides, 0, None, None)
    kept.append((t, shape, strides))
    return torch.utils.dlpack.from_dlpack(capsule(ctypes.addressof(t), b"dltensor", None))


def message(call, *args):
    try:
        call(*args)
    except RuntimeError as e:
        return str(e)
    return "no error"


from picotron_amd import _lib
host = _lib.host()
'''


def run(body):
    from picotron_amd import _lib
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("library not built here")
    res = subprocess.run([sys.executable, "-c", OPERANDS + body], cwd=ROOT, capture_output=True, text=True, timeout=300)
    assert res.returncode == 0, res.stdout + res.stderr


def test_operands_on_two_devices_are_refused():
    """As nn.Linear refuses them, in the forward and in both gradients, whichever route their sizes would have taken."""
    run('''
for rows, wide in ((512, 576), (4096, 2048)):
    x, w = operand(rows, 576), operand(wide, 576, device=1)
    dy = operand(rows, wide)
    for what in (message(host.linear, x, w), message(host.fused_linear, x, w, [w]), message(host.product, x, w, "NT"),
                 message(host.product, dy, w, "NN"), message(host.product, operand(rows, wide, device=1), x, "TN")):
        assert "same device" in what, what
''')


def test_the_predicate_is_what_the_kernel_refuses():
    """pico_product_takes against pico_product itself: with NULL operands an accepted shape ends at the pointers (-1)."""
    from picotron_amd import _lib
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("library not built here")
    lib, seen = _lib.lib(), set()
    for M, N, K in ((1, 8, 8), (512, 576, 576), (512, 576, 580), (516, 576, 576), (512, 580, 576), (2331, 1024, 2331)):
        for a_slow in (0, 1):
            for b_slow in (0, 1):
                for pad_a in (0, 4, 8, -8, 1 << 23, 1 << 31):
                    for pad_b in (0, 4, 8, 1 << 23):
                        lda, ldb = (M if a_slow else K) + pad_a, (N if b_slow else K) + pad_b
                        takes = lib.pico_product_takes(M, N, K, lda, ldb, a_slow, b_slow)
                        rc = lib.pico_product(None, None, None, M, N, K, lda, ldb, a_slow, b_slow, 64, 1, None)
                        assert rc == (-1 if takes else -3), (M, N, K, lda, ldb, a_slow, b_slow)
                        seen.add(takes)
    assert seen == {0, 1}


def test_row_pitches_the_kernels_refuse_go_to_the_library():
    """The sizes route to the package's kernels; the pitch (no multiple of 8, or rows too far apart) sends them past, to the library
    or, where only the operand that stays as it is does not fit, to the library with the other one transposed."""
    run('''
for kind, M, N, K, want in (("NT", 512, 576, 576, "own 64 in 2 groups"), ("NN", 512, 1024, 1024, "mid 32x64"), ("TN", 2048, 2048, 4096, "own 128 in 2 groups"),
                            ("TN", 49152, 2048, 4096, "large 256x256"), ("TN", 2048, 49152, 4096, "large 256x256")):
    (ra, ca), (rb, cb) = ((K, M) if kind == "TN" else (M, K)), ((N, K) if kind == "NT" else (K, N))
    for pad_a, pad_b in ((0, 0), (8, 0), (0, 24), (4, 0), (0, 4), (1, 1), (4, 24), (0, 1 << 24), (1 << 24, 0)):
        got = host.product_route(operand(ra, ca, ca + pad_a), operand(rb, cb, cb + pad_b), kind)
        fits = pad_a % 8 == 0 and pad_b % 8 == 0 and max(pad_a, pad_b) < 1 << 24
        turns = max(M, N) == 49152 and (pad_a if M < N else pad_b) % 8 == 0
        assert got == (want if fits else "turned" if turns else "library"), (kind, M, N, K, pad_a, pad_b, got)
    assert host.product_route(operand(ra, ca, address=(1 << 20) + 2), operand(rb, cb), kind) == "torch"
''')


def test_long_contractions_are_cut_where_pieces_are_faster():
    """Operands whose pitch leaves them to the library.  Sizes at which a cut was up to 1.44 times as slow as the whole product, or as
    another number of pieces, us: whole, in the number it was cut into, in the one expected now."""
    run('''
for kind, M, N, K, want in (("NT", 512, 2048, 8192, "library"),         # 27.0, 28.7 in 2
                            ("NT", 256, 4096, 10880, "library"),        # 1.23 times in 2
                            ("NT", 128, 2048, 8192, "library in 8"),    # 17.2, 22.1 in 2, 14.9
                            ("NT", 256, 3072, 12288, "library in 4"),   # 37.2, 53.7 in 2, 30.3
                            ("NN", 4096, 2048, 16384, "library in 2"),  # 1.11 times whole
                            ("NN", 5465, 2048, 16384, "library"),       # 286, 440 in 4
                            ("NN", 6144, 3072, 16384, "library in 2"),  # 900, 684 in 4, 558
                            ("NN", 3200, 2048, 32000, "library in 4"),  # 395, 522 in 2, 376
                            ("NN", 4608, 768, 49152, "library in 8"),   # 432, 540 in 4, 346
                            ("NN", 512, 576, 49152, "library in 16"), ("NN", 2048, 4096, 21760, "library in 2"), ("NT", 640, 2048, 8192, "library in 2")):
    (ra, ca), (rb, cb) = (M, K), ((N, K) if kind == "NT" else (K, N))
    got = host.product_route(operand(ra, ca), operand(rb, cb, cb + 4), kind)
    assert got == want, (kind, M, N, K, got)
''')


def test_weight_gradients_are_transposed_where_that_is_faster():
    """Operands of which the wider one's pitch leaves them to the library.  Us whole and with the narrower operand transposed; in the
    wrong one of the two it lost up to 58 %."""
    run('''
for K, M, N, want in ((4096, 10880, 2048, "library"),      # 172, 273
                      (1152, 10880, 2048, "library"),      # 67, 80
                      (1280, 12288, 1536, "library"),      # 64, 73
                      (1262, 12288, 4096, "library"),      # 1.06 times
                      (4096, 6144, 2048, "library"),       # level
                      (4096, 8192, 2048, "turned"), (4096, 2048, 8192, "turned"),   # 124, 112
                      (1024, 10880, 2048, "turned"),       # 1.43 times whole
                      (3266, 9216, 1152, "turned"),        # 1.23 times whole
                      (2944, 8192, 1024, "library"),       # 1.03 times
                      (4096, 49152, 2048, "turned"),       # 732, 616
                      (4096, 2048, 16384, "turned"),       # 227, 202
                      (5504, 12288, 1536, "turned"), (4096, 49152, 576, "turned")):
    got = host.product_route(operand(K, M, M + 4 * (M > N)), operand(K, N, N + 4 * (N > M)), "TN")
    assert got == want, (K, M, N, got)
''')


def test_the_large_predicate_is_what_the_kernel_refuses():
    """pico_product_large_takes against pico_product_large itself: with NULL operands an accepted shape ends at the pointers."""
    from picotron_amd import _lib
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("library not built here")
    lib, seen = _lib.lib(), set()
    for M, N, K in ((1, 8, 64), (1, 8, 72), (512, 576, 576), (512, 576, 580), (516, 576, 576), (512, 580, 576), (2331, 1024, 2331)):
        for a_slow, b_slow in ((0, 0), (0, 1), (1, 0), (1, 1)):
            for pad_a in (0, 4, 8, -8, 1 << 23, 1 << 31):
                for pad_b in (0, 4, 8, 1 << 23):
                    for parts in (0, 1, 4, 5, 65):
                        lda, ldb = (M if a_slow else K) + pad_a, (N if b_slow else K) + pad_b
                        takes = lib.pico_product_large_takes(M, N, K, lda, ldb, a_slow, b_slow, parts)
                        rc = lib.pico_product_large(None, None, None, M, N, K, lda, ldb, a_slow, b_slow, 256, 256, parts, None)
                        assert rc == (-1 if takes else -3), (M, N, K, lda, ldb, a_slow, b_slow, parts)
                        seen.add(takes)
    assert seen == {0, 1}
    assert lib.pico_product_large(1 << 20, 1 << 20, 1 << 20, 512, 576, 576, 576, 576, 0, 0, 128, 128, 1, None) == -3


def test_the_predicate_of_the_products_of_one_round_is_what_the_kernels_refuse():
    """pico_product_mid_takes against pico_product_mid and pico_product_pair themselves: with NULL operands an accepted shape ends at the pointers."""
    from picotron_amd import _lib
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("library not built here")
    lib, seen = _lib.lib(), set()
    sizes = ((1, 8, 8), (1, 8, 72), (512, 576, 576), (512, 576, 580), (516, 576, 576), (512, 580, 576), (2331, 1024, 2331), (0, 8, 8))
    pads = (0, 4, 8, -8, 1 << 23, 1 << 31)
    for M, N, K in sizes:
        for a_slow, b_slow in ((0, 0), (0, 1), (1, 0), (1, 1)):
            for pad_a in pads:
                for pad_b in pads:
                    lda, ldb = (M if a_slow else K) + pad_a, (N if b_slow else K) + pad_b
                    takes = lib.pico_product_mid_takes(M, N, K, lda, ldb, a_slow, b_slow)
                    rc = lib.pico_product_mid(None, None, None, M, N, K, lda, ldb, a_slow, b_slow, 64, 64, 1, None)
                    assert rc == (-1 if takes else -3), (M, N, K, lda, ldb, a_slow, b_slow)
                    seen.add(takes)
    for rows, out, inner in sizes:
        for pads_here in [(a, b, c) for a in pads for b in pads for c in pads]:
            ld_dy, ld_w, ld_x = (n + pad for n, pad in zip((out, inner, inner), pads_here))
            takes = lib.pico_product_mid_takes(rows, inner, out, ld_dy, ld_w, 0, 1) and lib.pico_product_mid_takes(out, inner, rows, ld_dy, ld_x, 1, 1)
            rc = lib.pico_product_pair(None, None, None, None, None, rows, out, inner, ld_dy, ld_w, ld_x, 64, 64, 64, 64, None)
            assert rc == (-1 if takes else -3), (rows, out, inner, pads_here)
            seen.add(2 + takes)
    assert seen == {0, 1, 2, 3}
    p = 1 << 20    # (refused before anything is launched: tiles that there are none of, more pieces than steps)
    for tile_m, tile_n, parts in ((96, 128, 1), (64, 64, 2), (64, 96, 10), (64, 96, 0)):
        assert lib.pico_product_mid(p, p, p, 512, 576, 576, 576, 576, 0, 0, tile_m, tile_n, parts, None) == -3
    for dx, dw in (((32, 32), (64, 64)), ((64, 64), (128, 128))):
        assert lib.pico_product_pair(p, p, p, p, p, 512, 576, 576, 576, 576, 576, *dx, *dw, None) == -3


def test_the_route_of_a_product():
    """Each route where it is taken and, beside it, where it is not: us without and with it."""
    run('''
for kind, M, N, K, want in (("TN", 4096, 4096, 4096, "large 256x256"),       # 137, 103
                            ("TN", 6144, 2048, 4096, "large 192x256"),       # 101, 91
                            ("TN", 16384, 2048, 4096, "large 256x256"),      # 216, 199
                            ("TN", 49152, 576, 512, "large 192x256"),        # 45, 40
                            ("TN", 32000, 256, 512, "mid 128x256"),          # own 17.2, 16.5
                            ("TN", 49152, 128, 7358, "turned"),              # 161, large 179
                            ("TN", 2048, 2048, 4096, "own 128 in 2 groups"), # 42, mid 39 .. 57 (operands from the caches, from memory), large 51
                            ("NN", 2242, 10880, 4096, "large 256x256"),      # 248, 178
                            ("NN", 608, 576, 49152, "mid 128x192 in 17"),    # 84, large 55
                            ("NN", 4548, 1024, 1024, "mid 128x192"),         # 17, large 20
                            ("NN", 2886, 3072, 49152, "library in 4"),       # 785, large 846
                            ("NN", 4096, 2048, 49152, "large 256x256 in 2"), # 663, 635
                            ("NN", 5108, 2816, 21504, "large 256x256"),      # 751, 472
                            ("NN", 4608, 3840, 16384, "library in 2"),       # 475, large 605
                            ("NT", 3832, 49152, 512, "large 256x256"),       # 315, 218
                            ("NT", 5856, 6144, 768, "large 192x256"),        # 79, 52
                            ("NT", 4096, 16384, 2048, "library"),            # 194, large 203
                            ("NT", 512, 49152, 576, "large 256x256"),        # 41, 34, in 128 x 256 46
                            ("NT", 512, 576, 576, "own 64 in 2 groups"),     # mid level
                            ("NN", 512, 576, 3072, "mid 32x64"),             # own 12.9, 8.7
                            ("NN", 2331, 576, 3072, "mid 96x64"),            # 27.7, 15.8
                            ("TN", 3072, 576, 2331, "mid 64x128"),
                            ("NT", 2331, 576, 1536, "mid 64x96"),            # 12.0, 9.5
                            ("NT", 256, 4096, 10880, "large 128x256 in 8"),  # 53.3, 42.9
                            ("NT", 128, 2048, 8192, "library in 8")):
    (ra, ca), (rb, cb) = ((K, M) if kind == "TN" else (M, K)), ((N, K) if kind == "NT" else (K, N))
    got = host.product_route(operand(ra, ca), operand(rb, cb), kind)
    assert got == want, (kind, M, N, K, got)
    if not want.startswith(("library", "turned")):    # pitches that the kernels refuse, and pitches that they take
        for a, b in ((operand(ra, ca, ca + 4), operand(rb, cb)), (operand(ra, ca), operand(rb, cb, cb + (1 << 24)))):
            assert host.product_route(a, b, kind).startswith(("library", "turned"))
        assert host.product_route(operand(ra, ca, ca + 8), operand(rb, cb, cb + 24), kind) == want
''')


def test_both_gradients_of_a_small_layer_go_together():
    """(rows, columns out, columns in): the tiles of dx and dw in one launch, or apart; us apart and together."""
    run('''
for rows, out, inner, want in ((512, 576, 576, "32x64 64x64"),     # 8.8, 5.2
                               (512, 3072, 576, "64x64 64x64"),    # 16.2, 13.1
                               (2331, 960, 576, "64x96 64x64"),    # 17.9, 14.0
                               (1024, 1024, 1024, "64x128 64x128"), # 15.1, 10.4
                               (1309, 1688, 1688, "apart"),        # 30.8, 37.3
                               (4096, 2048, 2048, "apart"), (512, 49152, 576, "apart"), (512, 580, 576, "apart")):
    got = host.gradient_route(operand(rows, out), operand(out, inner), operand(rows, inner))
    assert got == want, (rows, out, inner, got)
    if want != "apart":
        for a, b, c in ((operand(rows, out, out + 4), operand(out, inner), operand(rows, inner)),
                        (operand(rows, out), operand(out, inner), operand(rows, inner, inner + 4)),
                        (operand(rows, out), operand(out, inner), operand(rows, inner, device=1))):
            assert host.gradient_route(a, b, c) == "apart"
''')


def test_products_stay_where_the_other_kernels_lose():
    """Sizes of every kind that an own kernel, or another one, took and lost at: us where they go, us where they had gone."""
    run('''
for kind, M, N, K, want in (("NN", 1536, 2048, 49152, "library in 4"),       # 262, large 314
                            ("NN", 3584, 512, 32768, "library in 8"),        # 131, large 178, mid 145
                            ("NN", 1974, 1536, 12288, "library in 4"),       # 81, large 78, mid in pieces 90
                            ("NN", 1317, 4096, 49152, "large 192x256 in 2"), # 535, library in pieces 686
                            ("NN", 1025, 336, 32000, "mid 192x128 in 14"),  # 54, library in pieces 104
                            ("NN", 538, 768, 32000, "mid 192x128 in 14"),   # 55, library in pieces 104
                            ("NN", 6144, 1520, 344, "large 192x256"),        # 24, library 35
                            ("TN", 232, 184, 4819, "mid 64x96 in 21"),       # 14, mid in tiles of 64 x 32 36
                            ("TN", 32000, 192, 1987, "mid 128x192"),         # 49, library with an operand transposed 64
                            ("NT", 4096, 4096, 4096, "library"),             # 93, large 103
                            ("NT", 4096, 49152, 2048, "library"),            # 575, large 624
                            ("NN", 3274, 920, 2384, "own 128 in 2 groups"),  # 25.3, mid 28.5
                            ("NN", 64, 1784, 5376, "mid 64x96 in 6"),        # 11, mid 32x64 18
                            ("TN", 49152, 576, 6080, "turned"),              # 333, large 387
                            ("TN", 50304, 384, 243, "own 128 in 1 group"),   # 19.4, large 23.6
                            ("TN", 3072, 1024, 3584, "own 128 in 2 groups"), # 31.9, mid in pieces 35.8
                            ("TN", 2048, 2048, 5624, "large 256x256 in 4"),  # 60, own 59, mid 61
                            ("TN", 9792, 3264, 451, "large 256x256"),        # 38.8, own 49.7, mid 50.4
                            ("NT", 128, 832, 3328, "library"),               # 6.9, mid 9.0
                            ("NT", 6912, 73448, 192, "library"),             # 419, large 508
                            ("NT", 256, 2112, 2112, "own 64 in 2 groups"),   # 9.0, mid 9.4
                            ("NT", 64, 2688, 8064, "mid 64x96 in 9")):       # 0.57 of the library's time
    (ra, ca), (rb, cb) = ((K, M) if kind == "TN" else (M, K)), ((N, K) if kind == "NT" else (K, N))
    got = host.product_route(operand(ra, ca), operand(rb, cb), kind)
    assert got == want, (kind, M, N, K, got)
''')


def test_routes_that_are_kept_are_those_of_their_sizes():
    """More sizes than a thread keeps, with pitches that send some past the kernels, in one order and in the other, from two threads."""
    run('''
import threading
asked = [(kind, 64 + 40 * i, 64 + 8 * (i * 37 % 300), 64 + 8 * (i * 53 % 500), 4 * (i % 3)) for i in range(400) for kind in ("NT", "NN", "TN")]


def route(kind, M, N, K, pad):
    (ra, ca), (rb, cb) = ((K, M) if kind == "TN" else (M, K)), ((N, K) if kind == "NT" else (K, N))
    return host.product_route(operand(ra, ca, ca + pad), operand(rb, cb), kind), host.gradient_route(operand(M, K), operand(K, N), operand(M, N))


def ask(into, order):
    for q in order:
        into.append((q, route(*q), route(*q)))


answers = [[], []]
threads = [threading.Thread(target=ask, args=a) for a in zip(answers, (asked, asked[::-1]))]
for t in threads: t.start()
for t in threads: t.join()
first, second = ({q: r for q, r, again in a if r == again} for a in answers)
assert len(first) == len(set(asked)) and first == second
assert len(set(first.values())) > 20
''')
