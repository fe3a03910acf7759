"""The hot paths on a stream of the caller's and from two threads at once: forward and backward of each give what they give on
the default stream from one thread.  On the caller's stream the inputs are written late, behind work that keeps it busy, so a
launch on any other stream would read the zeros they were before; scratch memory comes from torch's allocator and is reused
between the passes."""
import threading

import pytest
import torch

pytestmark = pytest.mark.gpu


def normal(g, *shape, dtype=torch.bfloat16, scale=1.0):
    return (torch.randn(*shape, generator=g, device="cuda") * scale).to(dtype)


def linear_case(rows, cin, cout):
    def make(g):
        return normal(g, rows, cin), normal(g, cout, cin, scale=cin ** -0.5), normal(g, rows, cout)

    def run(x, w, dy):
        from picotron_amd import _lib
        x, w = x.requires_grad_(), w.requires_grad_()
        y = _lib.host().linear(x, w)
        return (y.detach(), *torch.autograd.grad(y, (x, w), dy))
    return make, run


def attention_case(B, Hq, Hkv, S, D):
    def make(g):
        return normal(g, B, Hq, S, D), normal(g, B, Hkv, S, D), normal(g, B, Hkv, S, D), normal(g, B, S, Hq, D)

    def run(q, k, v, dout):
        from picotron_amd.model import flash_attention
        q, k, v = (t.requires_grad_() for t in (q, k, v))
        out = flash_attention(q, k, v)
        return (out.detach(), *torch.autograd.grad(out, (q, k, v), dout))
    return make, run


def loss_case(rows, vocab):
    def make(g):
        return normal(g, rows, vocab, scale=3.0), torch.randint(0, vocab, (rows,), generator=g, device="cuda")

    def run(x, t):
        from picotron_amd.functional import cross_entropy
        x = x.requires_grad_()
        loss = cross_entropy(x, t, scale=0.5)
        return (loss.detach(), *torch.autograd.grad(loss, x, retain_graph=True), *torch.autograd.grad(loss, x, torch.full_like(loss, 0.3)))
    return make, run


def embedding_case(tokens, vocab, hidden):
    def make(g):
        return torch.randint(0, vocab, (tokens,), generator=g, device="cuda"), normal(g, vocab, hidden), normal(g, tokens, hidden)

    def run(ids, w, dy):
        from picotron_amd import _lib
        y = _lib.host().embedding(ids, w.requires_grad_(), -1)
        return (y.detach(), *torch.autograd.grad(y, w, dy))
    return make, run


def norm_case(rows, hidden):
    def make(g):
        return normal(g, rows, hidden), normal(g, rows, hidden), normal(g, hidden), normal(g, rows, hidden), normal(g, rows, hidden)

    def run(x, res, w, dy, dh):
        from picotron_amd.functional import RMSNormResidualFunc
        x, res, w = (t.requires_grad_() for t in (x, res, w))
        y, h = RMSNormResidualFunc.apply(x, res, w, 1e-5)
        return (y.detach(), h.detach(), *torch.autograd.grad((y, h), (x, res, w), (dy, dh)))
    return make, run


CASES = {
    "own_products": linear_case(512, 576, 960),
    "cut_input_gradient_and_turned_weight_gradient": linear_case(1024, 2048, 32000),
    "attention_whole": attention_case(2, 9, 3, 256, 64),
    "attention_in_pieces": attention_case(1, 12, 4, 3000, 128),
    "loss_one_pass": loss_case(300, 32000),
    "embedding": embedding_case(1500, 4000, 576),
    "norm": norm_case(700, 2048),
}


def same(got, want, what):
    for a, b in zip(got, want):
        # library products may add in another order; everything else has the same bits
        assert torch.equal(a, b) or ((a.float() - b.float()).norm() / b.float().norm()).item() <= 2e-3, what


def inputs(make, seed):
    return make(torch.Generator(device="cuda").manual_seed(seed))


@pytest.mark.parametrize("name", CASES)
def test_on_a_stream_of_the_callers(device, name):
    make, run = CASES[name]
    ready = [inputs(make, seed) for seed in range(3)]
    want = [run(*(t.clone() for t in r)) for r in ready]
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    got = []
    with torch.cuda.stream(side):
        for r in ready:
            late = [torch.zeros_like(t) for t in r]
            torch.cuda._sleep(3_000_000)            # about a millisecond: the inputs are still zeros when the calls are made
            for a, b in zip(late, r):
                a.copy_(b)
            got.append(run(*late))
    side.synchronize()
    for g, w in zip(got, want):
        same(g, w, name)


@pytest.mark.parametrize("name", CASES)
def test_from_two_threads(device, name):
    make, run = CASES[name]
    ready = [inputs(make, seed) for seed in range(2)]
    want = [run(*(t.clone() for t in r)) for r in ready]
    torch.cuda.synchronize()
    start, failed, got = threading.Barrier(2), [], [[], []]

    def work(i):
        try:
            with torch.cuda.stream(torch.cuda.Stream()) as _:
                mine = [[t.clone() for t in ready[i]] for _ in range(6)]
                start.wait(timeout=60)
                for m in mine:
                    got[i].append(run(*m))
                torch.cuda.current_stream().synchronize()
        except Exception as e:      # noqa: BLE001 (reported by the test's own thread)
            failed.append(repr(e))
            start.abort()
    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(timeout=100)
    assert not failed and not any(t.is_alive() for t in threads), failed
    for i in range(2):
        assert len(got[i]) == 6
        for g in got[i]:
            same(g, want[i], (name, i))
