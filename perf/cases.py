"""The work a user of this package has it do, as cases that can be timed and compared.

Every case goes through the public entry points: the model and its training step (``model.Llama``,
``functional.cross_entropy``, ``optim.FusedAdamW``), ``model.flash_attention``, ``context_parallel.ring_attention`` over
virtual ranks, ``model.TritonRMSNorm`` / ``LlamaRMSNorm``, ``functional.cross_entropy`` on logits and ``FusedAdamW.step``.
Sizes are those of the repository's configurations (SmolLM-135M, SmolLM-1.7B and Llama-2-7B shapes, the long-context
ring) and of its sweeps; ``draw`` spreads over the ranges between them, odd lengths and widths included.
"""
from __future__ import annotations

import math
import os

import torch

import picotron_amd.process_group_manager as pgm
from picotron_amd.context_parallel import context_parallel
from picotron_amd.functional import cross_entropy
from picotron_amd.model import Llama, LlamaRMSNorm, TritonRMSNorm, flash_attention, get_cos_sin
from picotron_amd.optim import FusedAdamW
from picotron_amd.utils import ModelShape

BF16, F32 = torch.bfloat16, torch.float32

# (hidden, query heads, kv heads, intermediate, vocab) of the shapes the repository's configurations name
SMOLLM_135M = (576, 9, 3, 1536, 49152)
SMOLLM_1P7B = (2048, 32, 32, 8192, 49152)
LLAMA2_7B = (4096, 32, 32, 11008, 32000)


def _model_case(path, shape, layers, batch, seq):
    return dict(path=path, hidden=shape[0], heads=shape[1], kv_heads=shape[2], inter=shape[3], vocab=shape[4], layers=layers,
                batch=batch, seq=seq)


def listed():
    return [
        # one optimizer step of the two-layer 135M shape: the plumbing run, where launches and host work are everything
        dict(name="step_135m", **_model_case("step", SMOLLM_135M, 2, 2, 256)),
        # one optimizer step of the 1.7B shape at its real batch, two of its 24 layers
        dict(name="step_1p7b", **_model_case("step", SMOLLM_1P7B, 2, 4, 1024)),
        # validation: forward and loss without gradients, at a length that is a multiple of nothing
        dict(name="eval_135m_ragged", **_model_case("eval", SMOLLM_135M, 4, 3, 777)),
        # attention of one layer, forward and backward: the smallest shape, the two training shapes, a ragged GQA batch
        dict(name="attn_135m", path="attention", batch=2, heads=9, kv_heads=3, seq=256, head_dim=64, causal=True),
        dict(name="attn_1p7b", path="attention", batch=4, heads=32, kv_heads=32, seq=1024, head_dim=64, causal=True),
        dict(name="attn_7b", path="attention", batch=1, heads=32, kv_heads=32, seq=4096, head_dim=128, causal=True),
        dict(name="attn_gqa_ragged", path="attention", batch=2, heads=32, kv_heads=8, seq=1531, head_dim=128, causal=True),
        # ring attention of all virtual ranks, forward and backward: the short ring and the 32k long-context one
        dict(name="ring_cp4", path="ring", cp=4, batch=4, heads=32, kv_heads=32, chunk=256, head_dim=64, rope=False),
        dict(name="ring_cp8_32k", path="ring", cp=8, batch=1, heads=32, kv_heads=8, chunk=4096, head_dim=128, rope=True),
        # RMSNorm with the residual add, as every layer of the 1.7B step calls it, forward and backward
        dict(name="norm_1p7b", path="norm", rows=4096, hidden=2048, dtype="bf16", residual=True, cast=False),
        # cross-entropy over the vocabulary, forward and backward
        dict(name="loss_1p7b", path="loss", rows=4096, vocab=49152, dtype="bf16", ignored=0.0),
        # the optimizer alone over two layers of the 7B shape: bf16 parameters, fp32 moments
        dict(name="adamw_7b", path="adamw", hidden=4096, inter=11008, vocab=32000, layers=2, kv_width=4096, master=False,
             state="fp32"),
    ]


# ------------------------------------------------------------------------------------------------------- drawing
def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_attention(rng):
    while True:
        head_dim = rng.choice((64, 128))
        kv = rng.choice((1, 2, 3, 4, 8, 16, 32))
        heads = kv * rng.choice((1, 1, 3, 4))
        c = dict(path="attention", batch=rng.choice((1, 2, 3, 4, 8)), heads=heads, kv_heads=kv, seq=_log(rng, 96, 8192),
                 head_dim=head_dim, causal=rng.random() < 0.85)
        if heads <= 40 and work(c)["flops"] < 5e12:
            return c


def _draw_ring(rng):
    while True:
        kv = rng.choice((2, 3, 8, 32))
        heads = kv * rng.choice((1, 3, 4))
        # a sequence is cut into equal chunks: mostly round lengths, now and then an odd one
        chunk = _log(rng, 64, 4096)
        chunk = max(128, chunk // 128 * 128) if rng.random() < 0.7 else chunk
        c = dict(path="ring", cp=rng.choice((2, 4, 8)), batch=rng.choice((1, 2, 4)), heads=heads, kv_heads=kv, chunk=chunk,
                 head_dim=rng.choice((64, 128)), rope=rng.random() < 0.5)
        if heads <= 32 and work(c)["flops"] < 6e12:
            return c


def _draw_model(rng, path):
    while True:
        head_dim = rng.choice((64, 64, 128))
        kv = rng.choice((2, 3, 4, 8, 16, 32))
        heads = kv * rng.choice((1, 3, 4))
        hidden = heads * head_dim
        c = dict(path=path, hidden=hidden, heads=heads, kv_heads=kv, inter=int(hidden * rng.choice((8 / 3, 4))) // 64 * 64,
                 vocab=rng.choice((32000, 49152)), layers=rng.choice((1, 2, 3)), batch=rng.choice((1, 2, 3, 4)),
                 seq=_log(rng, 128, 4096))
        if hidden <= 4096 and c["batch"] * c["seq"] <= 8192 and work(c)["flops"] < 1.5e13:
            return c


def draw(rng):
    path = rng.choice(("step", "eval", "attention", "attention", "ring", "norm", "loss", "adamw"))
    if path in ("step", "eval"):
        return _draw_model(rng, path)
    if path == "attention":
        return _draw_attention(rng)
    if path == "ring":
        return _draw_ring(rng)
    if path == "norm":
        return dict(path="norm", rows=_log(rng, 256, 16384), hidden=8 * _log(rng, 64, 1024), dtype=rng.choice(("bf16", "bf16", "fp32")),
                    residual=rng.random() < 0.6, cast=rng.random() < 0.5)
    if path == "loss":
        return dict(path="loss", rows=_log(rng, 256, 8192), vocab=8 * _log(rng, 1000, 16384), dtype=rng.choice(("bf16", "bf16", "fp32")),
                    ignored=rng.choice((0.0, 0.1)))
    master = rng.random() < 0.4
    hidden = 64 * _log(rng, 9, 64)
    return dict(path="adamw", hidden=hidden, inter=int(hidden * 8 / 3) // 8 * 8, vocab=_log(rng, 8000, 49152), layers=rng.choice((1, 2, 3)),
                kv_width=hidden // rng.choice((1, 3, 4)) // 8 * 8, master=master, state="fp32" if master else rng.choice(("fp32", "bf16")))


# ------------------------------------------------------------------------------------------------------- the states
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(g, *shape, dtype=BF16, scale=1.0):
    return (torch.randn(*shape, generator=g, device="cuda", dtype=F32) * scale).to(dtype)


def _heads(g, batch, heads, seq, dim, scale=1.0):
    """[B,H,S,D] over [B,S,H,D] memory, as a projection's output reaches attention."""
    return _normal(g, batch, seq, heads, dim, scale=scale).transpose(1, 2)


def _one_gpu(cp=1):
    os.environ["CONTEXT_PARALLEL"] = "1" if cp > 1 else "0"
    return pgm.setup_process_group_manager(1, cp, 1, 1)


def _prepare_model(c, seed):
    _one_gpu()
    torch.manual_seed(seed)
    shape = ModelShape(c["hidden"], c["heads"], c["kv_heads"], c["inter"], c["vocab"], c["layers"], c["seq"])
    with torch.device("cuda"):
        model = Llama(shape).to(BF16)
    g = _gen(seed)
    tokens = torch.randint(0, c["vocab"], (c["batch"], c["seq"] + 1), generator=g, device="cuda")
    state = dict(path=c["path"], model=model, ids=tokens[:, :-1].contiguous(), targets=tokens[:, 1:].reshape(-1).contiguous())
    if c["path"] == "step":
        state["opt"] = FusedAdamW(model.parameters(), lr=3e-4, master_weights=False, state_dtype=F32)
    return state


def _prepare_attention(c, seed):
    _one_gpu()
    g = _gen(seed)
    B, S, D = c["batch"], c["seq"], c["head_dim"]
    q = _heads(g, B, c["heads"], S, D).requires_grad_()
    k, v = (_heads(g, B, c["kv_heads"], S, D).requires_grad_() for _ in range(2))
    dout = _normal(g, B, S, c["heads"], D)          # what the output projection's backward hands back
    return dict(path="attention", q=q, k=k, v=v, dout=dout, causal=c["causal"])


def _prepare_ring(c, seed):
    mgr = _one_gpu(c["cp"])
    g = _gen(seed)
    B, S, D = c["batch"], c["chunk"], c["head_dim"]
    ranks = []
    for _ in range(c["cp"]):
        q = _heads(g, B, c["heads"], S, D).requires_grad_()
        k, v = (_heads(g, B, c["kv_heads"], S, D).requires_grad_() for _ in range(2))
        ranks.append((q, k, v))
    douts = [_heads(g, B, c["heads"], S, D) for _ in range(c["cp"])]
    rope = get_cos_sin(c["cp"] * S, D, base=10000.0) if c["rope"] else None
    return dict(path="ring", mgr=mgr, ranks=ranks, douts=douts, scale=1.0 / math.sqrt(D), rope=rope)


def _prepare_norm(c, seed):
    g = _gen(seed)
    dtype = BF16 if c["dtype"] == "bf16" else F32
    rows, hidden = c["rows"], c["hidden"]
    # LlamaRMSNorm (cast before the scale) has no residual argument
    norm = LlamaRMSNorm(hidden) if c["cast"] and not c["residual"] else TritonRMSNorm(hidden)
    norm = norm.to("cuda", dtype)
    with torch.no_grad():
        norm.weight.copy_(1 + 0.1 * _normal(g, hidden, dtype=F32))
    x, res = (_normal(g, rows, hidden, dtype=dtype).requires_grad_() for _ in range(2))
    dy, dh = (_normal(g, rows, hidden, dtype=dtype) for _ in range(2))
    return dict(path="norm", norm=norm, x=x, residual=res if c["residual"] else None, dy=dy, dh=dh)


def _prepare_loss(c, seed):
    g = _gen(seed)
    dtype = BF16 if c["dtype"] == "bf16" else F32
    logits = _normal(g, c["rows"], c["vocab"], dtype=dtype, scale=2.0).requires_grad_()
    targets = torch.randint(0, c["vocab"], (c["rows"],), generator=g, device="cuda")
    if c["ignored"]:
        targets[torch.rand(c["rows"], generator=g, device="cuda") < c["ignored"]] = -100
    return dict(path="loss", logits=logits, targets=targets)


def _adamw_shapes(c):
    h, i, kv = c["hidden"], c["inter"], c["kv_width"]
    shapes = [(c["vocab"], h)]
    for _ in range(c["layers"]):
        shapes += [(h,), (h, h), (kv, h), (kv, h), (h, h), (h,), (i, h), (i, h), (h, i)]
    return shapes + [(h,), (c["vocab"], h)]


def _prepare_adamw(c, seed):
    g = _gen(seed)
    params = []
    for shape in _adamw_shapes(c):
        p = torch.nn.Parameter(_normal(g, *shape, scale=0.02))
        p.grad = _normal(g, *shape, scale=1e-3)
        params.append(p)
    if c["master"]:
        opt = FusedAdamW(params, lr=3e-4, master_weights=True)
    else:
        opt = FusedAdamW(params, lr=3e-4, master_weights=False, state_dtype=F32 if c["state"] == "fp32" else None)
    return dict(path="adamw", params=params, opt=opt)


def prepare(case, seed):
    make = dict(step=_prepare_model, eval=_prepare_model, attention=_prepare_attention, ring=_prepare_ring, norm=_prepare_norm,
                loss=_prepare_loss, adamw=_prepare_adamw)
    return make[case["path"]](case, seed)


# ------------------------------------------------------------------------------------------------------- one pass
def _run_step(s):
    model, opt = s["model"], s["opt"]
    opt.zero_grad()
    logits = model(input_ids=s["ids"])
    loss = cross_entropy(logits.view(-1, logits.size(-1)), s["targets"])
    loss.backward()
    opt.step()
    return dict(loss=loss.detach(), grads=[p.grad for p in opt.params], params=[p.detach() for p in opt.params],
                exp_avg=opt.exp_avg, exp_avg_sq=opt.exp_avg_sq)


def _run_eval(s):
    with torch.no_grad():
        logits = s["model"](input_ids=s["ids"])
        return logits, cross_entropy(logits.view(-1, logits.size(-1)), s["targets"])


def _run_attention(s):
    q, k, v = s["q"], s["k"], s["v"]
    out = flash_attention(q, k, v, causal=s["causal"])
    return (out.detach(),) + torch.autograd.grad(out, (q, k, v), s["dout"])


def _run_ring(s):
    mgr = s["mgr"]
    pgm.process_group_manager = mgr
    mgr.cp_ring.reset()
    outs = []
    for rank, (q, k, v) in enumerate(s["ranks"]):
        mgr.set_cp_rank(rank)
        outs.append(context_parallel.ring_attention(q, k, v, s["scale"], True, rope=s["rope"]))
    leaves = [t for qkv in s["ranks"] for t in qkv]
    return [o.detach() for o in outs] + list(torch.autograd.grad(outs, leaves, s["douts"]))


def _run_norm(s):
    norm, x, res = s["norm"], s["x"], s["residual"]
    if res is None:
        y = norm(x)
        return (y.detach(),) + torch.autograd.grad(y, (x, norm.weight), s["dy"])
    y, h = norm(x, residual=res, prenorm=True)
    return (y.detach(), h.detach()) + torch.autograd.grad((y, h), (x, res, norm.weight), (s["dy"], s["dh"]))


def _run_loss(s):
    loss = cross_entropy(s["logits"], s["targets"])
    return (loss.detach(),) + torch.autograd.grad(loss, (s["logits"],))


def _run_adamw(s):
    s["opt"].step()
    return [p.detach() for p in s["params"]] + [s["opt"].exp_avg, s["opt"].exp_avg_sq]


def run(state):
    go = dict(step=_run_step, eval=_run_eval, attention=_run_attention, ring=_run_ring, norm=_run_norm, loss=_run_loss,
              adamw=_run_adamw)
    return go[state["path"]](state)


# ------------------------------------------------------------------------------------------------------- what it takes
def _attention_work(batch, heads, kv_heads, seq, dim, causal):
    pairs = seq * seq / (2 if causal else 1)
    # q, dout, out, dq and k, v, dk, dv in bf16; 4 forward and 10 backward operations per (query, key, column)
    return dict(bytes=2.0 * batch * seq * dim * (4 * heads + 4 * kv_heads), flops=14.0 * batch * heads * pairs * dim)


def _model_work(c):
    h, tokens = c["hidden"], c["batch"] * c["seq"]
    dim = h // c["heads"]
    per_layer = h * (2 * h + 2 * c["kv_heads"] * dim) + 3 * h * c["inter"]
    matmul = c["layers"] * per_layer + c["vocab"] * h
    params = matmul + c["vocab"] * h + (2 * c["layers"] + 1) * h
    attention = 2.0 * c["batch"] * c["seq"] ** 2 * h * c["layers"]       # forward, causal
    if c["path"] == "eval":
        # the weights, the embedding rows of the tokens, the logits
        return dict(bytes=2.0 * (matmul + tokens * (h + c["vocab"])), flops=2.0 * matmul * tokens + attention)
    # parameter and both fp32 moments read and written, gradient written
    return dict(bytes=22.0 * params, flops=6.0 * matmul * tokens + 3.5 * attention)


def work(case):
    c = case
    if c["path"] in ("step", "eval"):
        return _model_work(c)
    if c["path"] == "attention":
        return _attention_work(c["batch"], c["heads"], c["kv_heads"], c["seq"], c["head_dim"], c["causal"])
    if c["path"] == "ring":
        return _attention_work(c["batch"], c["heads"], c["kv_heads"], c["cp"] * c["chunk"], c["head_dim"], True)
    if c["path"] == "norm":
        n = c["rows"] * c["hidden"]
        size = 2 if c["dtype"] == "bf16" else 4
        # x, dy, y, dx; with the residual also the residual, its own gradient and the sum
        return dict(bytes=float(n * size * (7 if c["residual"] else 4)), flops=12.0 * n)
    if c["path"] == "loss":
        n = c["rows"] * c["vocab"]
        return dict(bytes=float(n * (2 if c["dtype"] == "bf16" else 4) * 2), flops=8.0 * n)
    n = sum(math.prod(s) for s in _adamw_shapes(c))
    per = 28 if c["master"] else 22 if c["state"] == "fp32" else 14
    return dict(bytes=float(n * per), flops=14.0 * n)


def tolerance(case):
    if case["path"] == "step":
        # gradients of a bf16 model: every activation on the way is rounded to 8 bits
        return {"rel": 1.5e-2, "max": 0.5}
    if case["path"] in ("norm", "loss") and case["dtype"] == "fp32":
        return {"rel": 1e-5, "max": 1e-3}
    if case["path"] in ("norm", "loss", "adamw"):
        return {"rel": 5e-3, "max": 3e-2}     # one bf16 rounding of each result
    return {"rel": 1e-2, "max": 0.2}
