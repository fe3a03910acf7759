"""The embedding's gradient against a sum in double precision: few and many tokens, repeated ids, runs of one id over many
workgroups, a padding id, both id and weight types."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens,vocab,hidden,ids_of", [
    (1, 10, 8, "random"), (7, 3, 64, "random"), (8, 1, 16, "one"), (63, 50, 576, "random"), (65, 65, 576, "few"), (129, 1000, 2056, "random"),
    (1000, 49152, 576, "zipf"), (4096, 49152, 2048, "random"), (4100, 32000, 1024, "few"), (2500, 100, 4096, "one"), (8192, 32000, 512, "zipf"),
    (32768, 1024, 64, "random"), (32769, 512, 64, "random")])
@pytest.mark.parametrize("dtype,id_dtype", [(torch.bfloat16, torch.int64), (torch.float32, torch.int32)])
def test_embedding_gradient(device, tokens, vocab, hidden, ids_of, dtype, id_dtype):
    from picotron_amd.model import Embedding
    g = torch.Generator().manual_seed(tokens)
    if ids_of == "one":
        ids = torch.full((tokens,), vocab - 1)
    elif ids_of == "few":
        ids = torch.randint(0, 3, (tokens,), generator=g) * (vocab // 3)
    elif ids_of == "zipf":
        ids = (vocab ** torch.rand(tokens, generator=g, dtype=torch.float64)).long().clamp_max(vocab) - 1
    else:
        ids = torch.randint(0, vocab, (tokens,), generator=g)
    ids = ids.to(device, id_dtype)
    dy = torch.randn(tokens, hidden, generator=g).to(device, dtype)
    for padding_idx in (None, int(ids[0])):
        layer = Embedding(vocab, hidden, padding_idx).to(device, dtype)
        out = layer(ids.view(1, -1))
        assert torch.equal(out[0], layer.weight[ids.long()])
        got, again = (torch.autograd.grad(out, layer.weight, dy[None], retain_graph=True)[0] for _ in range(2))
        want = torch.zeros(vocab, hidden, dtype=torch.float64, device=device).index_add_(0, ids.long(), dy.double())
        if padding_idx is not None:
            want[padding_idx] = 0
        assert torch.equal(got, again)
        assert (got.double() - want).abs().max().item() <= (4e-3 if dtype == torch.bfloat16 else 1e-6) * max(want.abs().max().item(), 1e-30)
        hit = torch.zeros(vocab, dtype=torch.bool, device=device)
        hit[ids.long()] = True
        assert not got[~hit].any()



@pytest.mark.parametrize("id_dtype,beyond", [(torch.int32, (2**31 - 1, -1, -2**31, 100)),
                                             (torch.int64, (2**31 - 1, 2**32 + 5, 2**63 - 1, -1, -2**63, 100, -2**32 + 7))])
@pytest.mark.parametrize("tokens", [130, 1000])
def test_ids_outside_the_vocabulary_add_nothing(device, id_dtype, beyond, tokens):
    """Through the C ABI, as torch's own lookup refuses such ids in the forward: the largest, ones that narrow to an id of the
    vocabulary, negative ones, many of each among many groups of tokens."""
    from picotron_amd import _lib
    lib, vocab, hidden = _lib.lib(), 100, 72
    g = torch.Generator().manual_seed(tokens)
    ids = torch.randint(0, vocab, (tokens,), generator=g)
    out = torch.rand(tokens, generator=g) < 0.5
    ids[out] = torch.tensor(beyond)[torch.randint(0, len(beyond), (int(out.sum()),), generator=g)]
    dy = torch.randn(tokens, hidden, generator=g).to(device, torch.bfloat16)
    want = torch.zeros(vocab, hidden, dtype=torch.float64, device=device).index_add_(0, ids[~out].to(device), dy[~out.to(device)].double())
    dev_ids = ids.to(device, id_dtype)
    dw = torch.empty(vocab, hidden, dtype=torch.bfloat16, device=device)
    ws = torch.empty(lib.pico_embedding_bwd_workspace_bytes(tokens, hidden), dtype=torch.uint8, device=device)
    _lib.check(lib.pico_embedding_bwd(dev_ids.data_ptr(), dev_ids.element_size(), dy.data_ptr(), dw.data_ptr(), ws.data_ptr(), tokens, vocab,
                                      hidden, -1, _lib.PICO_BF16, torch.cuda.current_stream().cuda_stream))
    assert (dw.double() - want).abs().max().item() <= 4e-3 * want.abs().max().item()


def test_norm_at_the_head_of_a_residual_stream(device):
    from picotron_amd.model import TritonRMSNorm
    g = torch.Generator(device="cuda").manual_seed(1)
    norm = TritonRMSNorm(576, device=device, dtype=torch.bfloat16)
    x = torch.randn(3, 50, 576, generator=g, device=device).to(torch.bfloat16).requires_grad_()
    dy, dh = (torch.randn(3, 50, 576, generator=g, device=device).to(torch.bfloat16) for _ in range(2))
    y, h = norm(x, prenorm=True)
    assert torch.equal(h, x) and torch.equal(y, norm(x))
    got = torch.autograd.grad((y, h), (x, norm.weight), (dy, dh), retain_graph=True)
    plain = torch.autograd.grad(norm(x), (x, norm.weight), dy)
    assert torch.equal(got[1], plain[1]) and (got[0].float() - (plain[0].float() + dh.float())).abs().max().item() <= 4e-2
    only_h = torch.autograd.grad(norm(x, prenorm=True)[1], x, dh)[0]
    assert torch.equal(only_h, dh)
