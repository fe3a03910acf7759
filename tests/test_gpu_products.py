"""The projections' matrix products: the rule that cuts long contractions into pieces, and the sum of the pieces, against a
fp32 product on the same bf16 operands."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,M,N,K", [
    ("NN", 8, 64, 5120), ("NN", 129, 576, 49152), ("NN", 512, 576, 49152), ("NN", 300, 1024, 5376), ("NN", 2100, 2048, 16384),
    ("NT", 31, 576, 8192), ("NT", 200, 2048, 16384), ("TN", 576, 960, 4096), ("TN", 64, 8, 8192), ("NN", 7, 9, 8192), ("TN", 72, 40, 333)])
def test_products_in_pieces(device, kind, M, N, K):
    from picotron_amd import _lib
    g = torch.Generator(device="cuda").manual_seed(M + K)
    a, b = (torch.randn(*s, generator=g, device=device).to(torch.bfloat16)
            for s in (((K, M) if kind == "TN" else (M, K)), ((N, K) if kind == "NT" else (K, N))))
    want = (a.float().t() if kind == "TN" else a.float()) @ (b.float().t() if kind == "NT" else b.float())
    for parts in (0, 1, 2, 4, 16):           # 0: the rule's own choice
        if parts > 1 and (K % (32 * parts) or M * N % 8):
            continue
        got = _lib.host().product(a, b, kind, parts)
        assert got.shape == (M, N) and got.dtype == torch.bfloat16
        assert ((got.float() - want).norm() / want.norm()).item() <= 3e-3, parts


@pytest.mark.parametrize("K,M,N", [(1, 8, 16), (127, 72, 64), (130, 64, 520), (1000, 1000, 248), (1025, 16384, 1032), (1111, 1024, 32000)])
def test_weight_gradients_with_transposed_operands(device, K, M, N):
    from picotron_amd import _lib
    g = torch.Generator(device="cuda").manual_seed(K)
    a, b = (torch.randn(K, n, generator=g, device=device).to(torch.bfloat16) for n in (M, N))
    want = a.float().t() @ b.float()
    for turn in (-1, 0, 1, 2, 3):            # -1: the rule's own choice
        got = _lib.host().product(a, b, "TN", 0, turn)
        assert ((got.float() - want).norm() / want.norm()).item() <= 3e-3, turn
    # columns of a wider matrix; the padding behind a row of the result is zero
    wide = torch.randn(K, M + 24, generator=g, device=device).to(torch.bfloat16)
    pitch = (K + 7) // 8 * 8
    y = torch.full((M, pitch), 3.0, dtype=torch.bfloat16, device=device)
    rc = _lib.lib().pico_transpose(wide[:, 8:].data_ptr(), y.data_ptr(), K, M, M + 24, pitch, torch.cuda.current_stream().cuda_stream)
    assert rc == 0 and torch.equal(y[:, :K], wide[:, 8:8 + M].t()) and not y[:, K:].any()


def test_linear_layer_gradients_match_torch(device):
    from picotron_amd.model import Linear
    g = torch.Generator(device="cuda").manual_seed(3)
    layer = Linear(5376, 1024, bias=False, device=device, dtype=torch.bfloat16)
    x = torch.randn(3, 107, 5376, generator=g, device=device).to(torch.bfloat16).requires_grad_()
    dy = torch.randn(3, 107, 1024, generator=g, device=device).to(torch.bfloat16)
    got = torch.autograd.grad(layer(x), (x, layer.weight), dy)
    xf, wf = x.detach().float().requires_grad_(), layer.weight.detach().float().requires_grad_()
    want = torch.autograd.grad(torch.nn.functional.linear(xf, wf), (xf, wf), dy.float())
    for a, b in zip(got, want):
        assert a.shape == b.shape and ((a.float() - b).norm() / b.norm()).item() <= 3e-3


def test_linear_layer_where_torch_has_to_see_it(device):
    """Second derivatives, forward-mode tangents and a frozen weight: as torch's own linear has them."""
    from picotron_amd.model import Linear
    F, rel = torch.nn.functional.linear, lambda a, b: ((a.float() - b).norm() / b.norm()).item()
    g = torch.Generator(device="cuda").manual_seed(5)
    layer = Linear(64, 48, bias=False, device=device, dtype=torch.bfloat16)
    x, t = (torch.randn(24, 64, generator=g, device=device).to(torch.bfloat16) for _ in range(2))
    xg, xf, wf = x.clone().requires_grad_(), x.float().requires_grad_(), layer.weight.detach().float().requires_grad_()

    def second(y, inp, w):
        (dx,) = torch.autograd.grad(y.float().square().sum(), inp, create_graph=True)
        return torch.autograd.grad(dx.float().square().sum(), (inp, w))
    for a, b in zip(second(layer(xg), xg, layer.weight), second(F(xf, wf), xf, wf)):
        assert rel(a, b) <= 1.5e-2                # three chained products, each rounded to bf16 (2^-9 each way)

    with torch.autograd.forward_ad.dual_level():
        dual = layer(torch.autograd.forward_ad.make_dual(x, t))
        tangent = torch.autograd.forward_ad.unpack_dual(dual).tangent
    assert rel(tangent, F(t.float(), wf.detach())) <= 3e-3

    layer.weight.requires_grad_(False)
    kept = []
    with torch.autograd.graph.saved_tensors_hooks(lambda s: kept.append(s) or s, lambda s: s):
        y = layer(xg)
    assert [s.shape for s in kept] == [layer.weight.shape]
    assert rel(torch.autograd.grad(y, xg, y.detach())[0], y.float() @ wf.detach()) <= 3e-3


def test_norm_passes_a_frozen_stream_through(device):
    from picotron_amd.model import TritonRMSNorm
    norm = TritonRMSNorm(64).to(device, torch.bfloat16)
    x = torch.randn(8, 64, device=device).to(torch.bfloat16)
    y, h = norm(x, prenorm=True)
    assert h is x and not h.requires_grad and y.requires_grad


@pytest.mark.parametrize("kind,M,N,K", [
    ("NT", 1, 8, 8), ("NT", 63, 72, 64), ("NT", 65, 64, 200), ("NT", 512, 576, 576), ("NT", 300, 520, 1536), ("NT", 130, 136, 1000),
    ("NN", 1, 8, 8), ("NN", 63, 72, 64), ("NN", 65, 64, 200), ("NN", 512, 576, 960), ("NN", 300, 520, 3072),
    ("TN", 8, 8, 1), ("TN", 72, 64, 63), ("TN", 64, 72, 197), ("TN", 576, 960, 512), ("TN", 520, 136, 2331)])
def test_small_products(device, kind, M, N, K):
    """The package's own kernel: edges of its tiles of 64 and 128 and its steps of 64, contractions shorter than a group's share, wider row pitches."""
    from picotron_amd import _lib
    g = torch.Generator(device="cuda").manual_seed(M * N + K)
    shapes = ((K, M) if kind == "TN" else (M, K)), ((N, K) if kind == "NT" else (K, N))
    for pad in (0, 24):
        a, b = (torch.randn(r, c + pad, generator=g, device=device).to(torch.bfloat16)[:, :c] for r, c in shapes)
        want = (a.float().t() if kind == "TN" else a.float()) @ (b.float().t() if kind == "NT" else b.float())
        for tile, groups in ((64, 1), (64, 2), (64, 4), (128, 1), (128, 2)):
            got = _lib.host().product(a, b, kind, groups=groups, tile=tile)
            assert got.shape == (M, N) and got.dtype == torch.bfloat16
            assert ((got.float() - want).norm() / want.norm()).item() <= 3e-3, (pad, tile, groups)
            assert torch.equal(got, _lib.host().product(a, b, kind, groups=groups, tile=tile))
    exact = _lib.host().product(a.round(), b.round(), kind, groups=4)     # small integers: sums are exact in fp32
    want = (a.round().float().t() if kind == "TN" else a.round().float()) @ (b.round().float().t() if kind == "NT" else b.round().float())
    assert torch.equal(exact, want.to(torch.bfloat16))


@pytest.mark.parametrize("pad", [1, 4, 8])
@pytest.mark.parametrize("rows,cin,cout", [(512, 576, 576), (300, 520, 1536), (1024, 1024, 32000)])
def test_linear_on_columns_of_a_wider_buffer(device, rows, cin, cout, pad):
    """Rows that lie `pad` elements further apart than they are long, where the dense sizes go to the package's kernels; with
    a pitch that is no multiple of 8 the product that reads it goes to the library."""
    from picotron_amd.model import Linear
    g = torch.Generator(device="cuda").manual_seed(rows + pad)
    layer = Linear(cin, cout, bias=False, device=device, dtype=torch.bfloat16)
    x = torch.randn(rows, cin + pad, generator=g, device=device).to(torch.bfloat16)[:, :cin].requires_grad_()
    dy = torch.randn(rows, cout + pad, generator=g, device=device).to(torch.bfloat16)[:, :cout]
    y = layer(x)
    got = (y, *torch.autograd.grad(y, (x, layer.weight), dy))
    xf, wf = x.detach().float().requires_grad_(), layer.weight.detach().float().requires_grad_()
    yf = torch.nn.functional.linear(xf, wf)
    for a, b in zip(got, (yf, *torch.autograd.grad(yf, (xf, wf), dy.float()))):
        assert a.shape == b.shape and ((a.float() - b).norm() / b.norm()).item() <= 3e-3


@pytest.mark.parametrize("kind,M,N,K", [
    ("NT", 1, 8, 72), ("NT", 257, 264, 128), ("NT", 255, 200, 136), ("NT", 700, 520, 1000), ("NT", 2100, 4360, 328),
    ("NN", 1, 8, 72), ("NN", 257, 264, 128), ("NN", 255, 200, 136), ("NN", 700, 520, 1000), ("NN", 2100, 4360, 328),
    ("TN", 8, 8, 65), ("TN", 264, 256, 129), ("TN", 248, 200, 133), ("TN", 704, 520, 1001), ("TN", 4360, 2104, 331)])
def test_large_products(device, kind, M, N, K):
    """The kernel for products that fill the GPU: edges of its tiles and steps, more tiles than workgroups, pieces of unequal
    length, wider row pitches."""
    from picotron_amd import _lib
    g = torch.Generator(device="cuda").manual_seed(M * N + K)
    shapes = ((K, M) if kind == "TN" else (M, K)), ((N, K) if kind == "NT" else (K, N))
    for pad in (0, 24):
        a, b = (torch.randn(r, c + pad, generator=g, device=device).to(torch.bfloat16)[:, :c] for r, c in shapes)
        ai, bi = a.round(), b.round()            # small integers: sums are exact in fp32
        want, exact = ((x.float().t() if kind == "TN" else x.float()) @ (y.float().t() if kind == "NT" else y.float()) for x, y in ((a, b), (ai, bi)))
        for tile, tile_n in ((256, 256), (256, 192), (192, 256), (256, 128), (128, 256)):
            for parts in (1, 2, 5):
                if (K + 63) // 64 < 2 * parts:
                    continue
                got = _lib.host().product(a, b, kind, parts, tile=tile, tile_n=tile_n)
                assert got.shape == (M, N) and got.dtype == torch.bfloat16
                assert ((got.float() - want).norm() / want.norm()).item() <= 3e-3, (pad, tile, tile_n, parts)
                assert torch.equal(got, _lib.host().product(a, b, kind, parts, tile=tile, tile_n=tile_n))
                assert torch.equal(_lib.host().product(ai, bi, kind, parts, tile=tile, tile_n=tile_n), exact.to(torch.bfloat16))


@pytest.mark.parametrize("rows,out,inner", [(1, 8, 8), (64, 64, 64), (65, 72, 136), (63, 1000, 200), (512, 960, 576), (333, 3072, 576), (2100, 520, 328)])
def test_both_gradients_in_one_launch(device, rows, out, inner):
    """Edges of the tiles, every pair of tiles, operands that are columns of wider matrices, against fp32 products (rounded once:
    2^-9); the rule takes small layers and leaves large ones apart."""
    from picotron_amd import _lib
    host = _lib.host()
    g = torch.Generator(device="cuda").manual_seed(rows + out)
    wide = torch.randn(rows, out + 24, generator=g, device=device).to(torch.bfloat16)
    w, x = (torch.randn(n, inner, generator=g, device=device).to(torch.bfloat16) for n in (out, rows))
    tiles = [(32, 64), (64, 64), (64, 96), (64, 128)]
    for dy in (wide[:, 8:8 + out], wide[:, 16:16 + out].contiguous()):
        want = (dy.float() @ w.float(), dy.float().t() @ x.float())
        assert host.gradients(dy, w, x)[2] > 0
        for choice in [[]] + [[*a, *b] for a in tiles for b in tiles]:
            got = host.gradients(dy, w, x, choice)
            for a, b in zip(got, want):
                assert a.shape == b.shape and a.is_contiguous() and ((a.float() - b).norm() / b.norm()).item() <= 3e-3, choice
            again = host.gradients(dy, w, x, choice)
            assert torch.equal(got[0], again[0]) and torch.equal(got[1], again[1]), choice
    big = torch.zeros(4096, 2048, dtype=torch.bfloat16, device=device)
    assert host.gradients(big, big[:2048], big)[2] == 0


MID_TILES = [(32, 32), (32, 64), (64, 32), (64, 64), (64, 96), (96, 64), (96, 96), (64, 128), (128, 64), (128, 96), (128, 128), (128, 192), (192, 128),
             (128, 256)]


@pytest.mark.parametrize("kind,M,N,K", [(kind, *size) for size in [(8, 8, 8), (64, 96, 64), (72, 136, 200), (200, 328, 72), (264, 272, 584), (520, 40, 1032)]
                                        for kind in ("NT", "NN", "TN")] +
                         [("NT", 1, 8, 8), ("NN", 1, 8, 8), ("NT", 33, 72, 136), ("NN", 33, 72, 136), ("TN", 72, 40, 1), ("TN", 72, 40, 333)])
def test_products_of_one_round(device, kind, M, N, K):
    """Every tile, at sizes around its edges, one row, contractions of fewer steps than groups and of a ragged last step, operands that are
    columns of wider matrices, against a fp32 product (rounded once: 2^-9) and, with small integers, whose sums are exact in fp32, bit for bit."""
    from picotron_amd import _lib
    host = _lib.host()
    g = torch.Generator(device="cuda").manual_seed(M + K)
    sizes = ((K, M) if kind == "TN" else (M, K)), ((N, K) if kind == "NT" else (K, N))
    a, b = (torch.randn(r, c + 16, generator=g, device=device).to(torch.bfloat16)[:, 8:8 + c] for r, c in sizes)
    ai, bi = a.round(), b.round()
    want, exact = ((x.float().t() if kind == "TN" else x.float()) @ (y.float().t() if kind == "NT" else y.float()) for x, y in ((a, b), (ai, bi)))
    for tiles in MID_TILES:
        got, tile_m, tile_n = host.mid_product(a, b, kind, *tiles)
        assert (tile_m, tile_n) == tiles and ((got.float() - want).norm() / want.norm()).item() <= 3e-3, tiles
        assert torch.equal(got, host.mid_product(a, b, kind, *tiles)[0]), tiles
        assert torch.equal(host.mid_product(ai, bi, kind, *tiles)[0], exact.to(torch.bfloat16)), tiles
    with pytest.raises(RuntimeError, match="no tiles"):
        host.mid_product(a, b, kind, 96, 128)


@pytest.mark.parametrize("M,N,K", [(72, 136, 1000), (304, 200, 4096), (64, 96, 256), (136, 264, 8200)])
@pytest.mark.parametrize("kind", ["NT", "NN", "TN"])
def test_products_in_pieces_of_one_round(device, kind, M, N, K):
    """Every tile that takes pieces, as many as the steps allow at most, a ragged last step, and the rule's own choice."""
    from picotron_amd import _lib
    host = _lib.host()
    g = torch.Generator(device="cuda").manual_seed(K)
    sizes = ((K, M) if kind == "TN" else (M, K)), ((N, K) if kind == "NT" else (K, N))
    a, b = (torch.randn(r, c + 16, generator=g, device=device).to(torch.bfloat16)[:, 8:8 + c] for r, c in sizes)
    ai, bi = a.round(), b.round()    # small integers: sums are exact in fp32
    want, exact = ((x.float().t() if kind == "TN" else x.float()) @ (y.float().t() if kind == "NT" else y.float()) for x, y in ((a, b), (ai, bi)))
    steps = (K + 63) // 64
    for tiles in [(64, 96), (64, 128), (96, 96), (128, 128), (128, 192), (192, 128), (128, 256)]:
        for parts in {2, 3, min(steps, 15), min(steps, 64)}:
            got = host.mid_product(a, b, kind, *tiles, parts)[0]
            assert ((got.float() - want).norm() / want.norm()).item() <= 3e-3, (tiles, parts)
            assert torch.equal(host.mid_product(ai, bi, kind, *tiles, parts)[0], exact.to(torch.bfloat16)), (tiles, parts)
    assert ((host.product(a, b, kind).float() - want).norm() / want.norm()).item() <= 3e-3
    for bad in ((64, 64, 2), (64, 96, 65), (64, 96, steps + 1)):
        with pytest.raises(RuntimeError):
            host.mid_product(a, b, kind, *bad)


@pytest.mark.parametrize("kind,M,N,K", [
    ("NN", 64, 1784, 5376), ("NN", 577, 192, 24576), ("NN", 300, 512, 32768), ("NN", 1320, 2240, 3360), ("NN", 3274, 920, 2384), ("NN", 2048, 2048, 16384),
    ("NT", 128, 832, 3328), ("NT", 64, 2688, 8064), ("NT", 129, 640, 4096), ("NT", 700, 24584, 192), ("NT", 700, 24584, 320), ("NT", 256, 2112, 2112),
    ("TN", 24576, 384, 243), ("TN", 24584, 576, 3001), ("TN", 3072, 1024, 3584), ("TN", 2048, 2048, 1111), ("TN", 48, 9000, 3950)])
def test_products_by_the_rule(device, kind, M, N, K):
    """On both sides of the lines between the kernels, as dense operands and as columns of wider ones whose pitch the package's kernels
    take or refuse, against a fp32 product (rounded once: 2^-9); the package's kernels give the same on every call."""
    from picotron_amd import _lib
    host = _lib.host()
    g = torch.Generator(device="cuda").manual_seed(M + K)
    sizes = ((K, M) if kind == "TN" else (M, K)), ((N, K) if kind == "NT" else (K, N))
    for pad in (0, 16, 4):
        a, b = (torch.randn(r, c + pad, generator=g, device=device).to(torch.bfloat16)[:, :c] for r, c in sizes)
        want = (a.float().t() if kind == "TN" else a.float()) @ (b.float().t() if kind == "NT" else b.float())
        got, route = host.product(a, b, kind), host.product_route(a, b, kind)
        assert got.shape == (M, N) and ((got.float() - want).norm() / want.norm()).item() <= 3e-3, (pad, route)
        if not route.startswith(("library", "turned")):
            assert pad != 4 and torch.equal(got, host.product(a, b, kind)), (pad, route)
