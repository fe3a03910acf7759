"""The one-pass cross-entropy (forward and gradient from one read of the logits) at the edges of its workgroup sizes: the
smallest row, one entry before and after each switch of the kernel, rows that are no multiple of a vector, the longest row
and one that no longer fits (two passes), against torch in fp64."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def rel(a, b):
    return ((a.double() - b.double()).norm() / b.double().norm().clamp_min(1e-30)).item()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("pieces,extra", [(0, 3), (64 * 4, 0), (64 * 4, 1), (128 * 4, 3), (256 * 4, 0), (256 * 4, 1), (256 * 8, 1), (512 * 8, 1),
                                          (1024 * 6, 0), (1024 * 8, 1), (1024 * 16, 0), (1024 * 16 + 1, 0)])
def test_one_pass_rows_at_the_edges(device, dtype, pieces, extra):
    from picotron_amd.functional import cross_entropy
    vec = 8 if dtype == torch.bfloat16 else 4
    vocab, rows = pieces * vec + extra, 5
    g = torch.Generator(device="cuda").manual_seed(pieces + extra)
    buf = torch.zeros(rows, (vocab + vec - 1) // vec * vec, dtype=dtype, device=device)
    x = buf[:, :vocab].copy_(torch.randn(rows, vocab, generator=g, device=device) * 4).requires_grad_()
    t = torch.randint(0, vocab, (rows,), generator=g, device=device)
    t[0], t[1], t[2] = vocab - 1, 0, -100
    xd = x.detach().double().requires_grad_()
    want = torch.nn.functional.cross_entropy(xd, t)
    (gw,) = torch.autograd.grad(want, xd)
    tol = 4e-3 if dtype == torch.bfloat16 else 1e-5
    with torch.no_grad():
        assert abs(cross_entropy(x, t).item() - want.item()) <= 2e-5 * abs(want.item())
    loss = cross_entropy(x, t)
    assert abs(loss.item() - want.item()) <= 2e-5 * abs(want.item())
    # upstream gradients of 1 (the forward's own gradient) and of something else, the node used more than once
    for k, up in enumerate((1.0, 1.0, 0.37)):
        (got,) = torch.autograd.grad(loss, x, torch.full_like(loss, up), retain_graph=True)
        assert rel(got, gw * up) <= tol, (k, up)
        assert got[2].abs().max().item() == 0.0
    (got,) = torch.autograd.grad(cross_entropy(x, t), x, torch.full_like(loss, -3.0))
    assert rel(got, gw * -3.0) <= tol


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("vocab", [1003, 32000, 49152, 8 * 1024 * 17])   # (the last: two passes)
def test_a_factor_of_the_loss(device, dtype, vocab):
    """`scale` is part of the loss and of its gradient: as the division behind the loss, with an upstream gradient of 1 (the
    forward's own gradient, the same buffer) and of something else, without a gradient, and with nothing to average."""
    from picotron_amd.functional import cross_entropy
    g = torch.Generator(device="cuda").manual_seed(vocab)
    x = torch.zeros(6, (vocab + 7) // 8 * 8, dtype=dtype, device=device)[:, :vocab]
    x.copy_(torch.randn(6, vocab, generator=g, device=device) * 3).requires_grad_()
    t = torch.randint(0, vocab, (6,), generator=g, device=device)
    t[2] = -100
    xd = x.detach().double().requires_grad_()
    want = torch.nn.functional.cross_entropy(xd, t)
    (gw,) = torch.autograd.grad(want, xd)
    tol = 4e-3 if dtype == torch.bfloat16 else 1e-5                     # one rounding to the logits' type
    for scale in (1.0, 0.25, 1 / 3, 128.0):
        loss = cross_entropy(x, t, scale=scale)
        assert abs(loss.item() - scale * want.item()) <= 2e-5 * abs(scale * want.item())
        for up in (1.0, 0.37):
            (got,) = torch.autograd.grad(loss, x, torch.full_like(loss, up), retain_graph=True)
            assert rel(got, gw * scale * up) <= tol, (scale, up)
        with torch.no_grad():
            assert abs(cross_entropy(x, t, scale=scale).item() - loss.item()) <= 2e-5 * abs(loss.item())
    (one,), (div,) = (torch.autograd.grad(l, x) for l in (cross_entropy(x, t, scale=0.25), cross_entropy(x, t) / 4))
    assert rel(one, div.double()) <= tol
    assert cross_entropy(x, torch.full_like(t, -100), scale=0.5).item() == 0.0


@pytest.mark.parametrize("rows,vocab", [(1, 800), (64, 800), (65, 800), (255, 8192), (257, 8192), (1024, 40000), (1025, 40000)])
def test_rows_that_count(device, rows, vocab):
    """Around the number of rows up to which every workgroup counts for itself (one per thread of it); ignored rows, a class that is
    ignored, no row that counts."""
    from picotron_amd.functional import cross_entropy
    g = torch.Generator(device="cuda").manual_seed(rows)
    x = (torch.randn(rows, vocab, generator=g, device=device) * 2).to(torch.bfloat16).requires_grad_()
    t = torch.randint(0, vocab, (rows,), generator=g, device=device)
    t[::3] = 7
    for targets, ignored in ((t, 7), (t, -100), (torch.full_like(t, -100), -100)):
        loss = cross_entropy(x, targets, ignored)
        (got,) = torch.autograd.grad(loss, x)
        live = targets != ignored
        if not live.any():
            assert loss.item() == 0.0 and not got.any()
            continue
        xd = x.detach()[live].float().requires_grad_()
        want = torch.nn.functional.cross_entropy(xd, targets[live])
        (gw,) = torch.autograd.grad(want, xd)
        assert abs(loss.item() - want.item()) <= 2e-5 * abs(want.item())
        assert rel(got[live], gw) <= 4e-3 and not got[~live].any()     # (rounded once: 2^-9)
