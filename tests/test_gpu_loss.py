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
