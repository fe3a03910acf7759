"""Tensor-level wrappers over the C ABI: they validate, allocate outputs with torch and pass raw
device pointers + the current HIP stream.  No arithmetic happens here and nothing falls back to
torch ops: a CPU tensor or a missing library is an error.  The wrappers of the hot ops are native
(``csrc/host.cpp``, reached through ``_lib.host()``); the functions below give them their keyword
arguments and defaults.
"""
from __future__ import annotations

import ctypes
from typing import Optional, Tuple

import torch

from . import _lib
from ._lib import PICO_BF16, PICO_F32, AttnDesc, KvChunks, check

_DT = {torch.bfloat16: PICO_BF16, torch.float32: PICO_F32}


def _dt(t: torch.Tensor, what: str) -> int:
    if t.dtype not in _DT:
        raise RuntimeError(f"{what}: dtype {t.dtype} not supported by the HIP kernels (bf16 / fp32 only)")
    return _DT[t.dtype]


def _dev(*tensors: Optional[torch.Tensor]) -> None:
    for t in tensors:
        if t is not None and not t.is_cuda:
            raise RuntimeError("picotron_amd kernels run on the GPU only: got a CPU tensor (there is no CPU fallback)")


def _ptr(t: Optional[torch.Tensor]):
    return ctypes.c_void_p(t.data_ptr()) if t is not None else None


def _stream():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


# ------------------------------------------------------------------------------- RMSNorm
def rmsnorm_fwd(x: torch.Tensor, weight: torch.Tensor, eps: float, cast_then_scale: bool,
                residual: Optional[torch.Tensor] = None, want_residual_out: bool = False,
                want_rstd: bool = True):
    """Returns (y, rstd or None, residual_out or None); x is [..., hidden]."""
    return _lib.host().rmsnorm_fwd(x, weight, eps, bool(cast_then_scale), residual, want_residual_out, want_rstd)


def rmsnorm_bwd(dy: torch.Tensor, x: torch.Tensor, weight: torch.Tensor, rstd: torch.Tensor,
                dresidual: Optional[torch.Tensor] = None, dw_dtype=torch.float32):
    """Returns (dx in x.dtype, dweight [hidden] in dw_dtype).  `dresidual` (x's shape and dtype), when given, is added
    to dx inside the kernel: the gradient that reached the residual stream directly."""
    return _lib.host().rmsnorm_bwd(dy, x, weight, rstd, dresidual, dw_dtype)


# ------------------------------------------------------------------------------- RoPE
def rope(x: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor, pos_offset: int = 0, inverse: bool = False,
         out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Rotates x [B,H,S,D] (any b/h/s strides, unit D stride) with table rows pos_offset + s."""
    return _lib.host().rope(x, cos, sin, int(pos_offset), bool(inverse), out)


def _dense(t: torch.Tensor) -> bool:
    """True if t's strides are a permutation of a contiguous layout (no gaps, no overlap)."""
    dims = sorted(range(t.dim()), key=lambda i: t.stride(i), reverse=True)
    expect = 1
    for i in reversed(dims):
        if t.size(i) != 1 and t.stride(i) != expect:
            return False
        expect *= t.size(i)
    return True


# ------------------------------------------------------------------------------- SwiGLU
def swiglu_fwd(gate: torch.Tensor, up: torch.Tensor) -> torch.Tensor:
    return _lib.host().swiglu_fwd(gate, up)


def swiglu_bwd(dy: torch.Tensor, gate: torch.Tensor, up: torch.Tensor, out=None):
    """(dgate, dup); `out` = (dgate, dup) buffers to write into (e.g. the two halves of one fused gradient)."""
    return _lib.host().swiglu_bwd(dy, gate, up, *(out if out is not None else (None, None)))


# ------------------------------------------------------------------------------- lse merge
def lse_merge_(out: torch.Tensor, lse: torch.Tensor, block_out: torch.Tensor, block_lse: torch.Tensor) -> None:
    """In place: (out fp32 [..., D], lse fp32 [...]) <- merge with (block_out, block_lse)."""
    _dev(out, lse, block_out, block_lse)
    if out.dtype != torch.float32 or lse.dtype != torch.float32 or block_lse.dtype != torch.float32:
        raise RuntimeError("lse_merge_: out, lse and block_lse must be fp32")
    if not (out.is_contiguous() and lse.is_contiguous()):
        raise RuntimeError("lse_merge_: out and lse must be contiguous (they are updated in place)")
    D = out.size(-1)
    rows = out.numel() // D
    bo, bl = block_out.contiguous(), block_lse.contiguous()
    check(_lib.lib().pico_lse_merge(_ptr(out), _ptr(lse), _ptr(bo), _ptr(bl), rows, D, _dt(bo, "lse_merge_"), _stream()))


# ------------------------------------------------------------------------------- attention
def _desc(q, k, v, o, sm_scale, causal, q_offset) -> AttnDesc:
    B, Hq, Sq, D = q.shape
    Hkv, Sk = k.size(1), k.size(2)
    d = AttnDesc()
    d.B, d.Hq, d.Hkv, d.Sq, d.Sk, d.D = B, Hq, Hkv, Sq, Sk, D
    d.causal, d.q_offset, d.sm_scale = int(bool(causal)), int(q_offset), float(sm_scale)
    for name, t in (("q_stride", q), ("k_stride", k), ("v_stride", v), ("o_stride", o)):
        arr = getattr(d, name)
        arr[0], arr[1], arr[2] = t.stride(0), t.stride(1), t.stride(2)
    return d


def _attn_in(t: torch.Tensor, what: str) -> torch.Tensor:
    if t.dtype != torch.bfloat16:
        raise RuntimeError(f"attention: {what} must be bf16 (got {t.dtype}); the MFMA kernels are bf16 only")
    if t.dim() != 4:
        raise RuntimeError(f"attention: {what} must be [B, H, S, D]")
    if t.stride(-1) != 1 or any(s % 8 for s in t.stride()[:3]):
        t = t.contiguous()
    return t


def empty_bshd(B: int, H: int, S: int, D: int, dtype, device) -> torch.Tensor:
    """A [B,H,S,D]-shaped view of a fresh [B,S,H,D] buffer: `.transpose(1,2).reshape(B,S,H*D)` on it is free."""
    return torch.empty(B, S, H, D, dtype=dtype, device=device).transpose(1, 2)


def attn_fwd(q, k, v, sm_scale: float, causal: bool, q_offset: int = 0, out: Optional[torch.Tensor] = None,
             lse: Optional[torch.Tensor] = None, merge: bool = False, out_dtype=torch.bfloat16,
             bshd_out: bool = False) -> Tuple[torch.Tensor, torch.Tensor]:
    """softmax(q k^T * scale + mask) v for q [B,Hq,Sq,D], k/v [B,Hkv,Sk,D]; returns (out, lse fp32 [B,Hq,Sq]).

    merge=True continues the online softmax from the running fp32 (out, lse) passed in and updates them in place.
    """
    out, lse, _ = _lib.host().attn_fwd(q, [k], [v], sm_scale, bool(causal), int(q_offset), out, lse, bool(merge), out_dtype, bshd_out,
                                       None, 0, False, None)
    return out, lse


def attn_fwd_rope(q, k_rot, v, cos, sin, sm_scale: float, causal: bool, q_offset: int = 0, q_pos_offset: int = 0,
                  want_q_rot: bool = True, out_dtype=torch.bfloat16, bshd_out: bool = True, out=None, lse=None,
                  merge: bool = False, q_rot=None):
    """RoPE on q inside the attention forward (k_rot must be rotated already): returns (out, lse, q_rot or None); q_rot is
    the rotated q, laid out like q, for attn_bwd_rope.  merge=True continues from the running fp32 (out, lse) given, as
    attn_fwd does: one step of a ring whose queries sit at positions q_pos_offset .."""
    return _lib.host().attn_fwd(q, [k_rot], [v], sm_scale, bool(causal), int(q_offset), out, lse, bool(merge), out_dtype, bshd_out,
                                (cos, sin), int(q_pos_offset), want_q_rot, q_rot)


def attn_bwd_rope(dout, q_rot, k_rot, v, out, lse, cos, sin, sm_scale: float, causal: bool, dq, dk, dv, q_offset: int = 0,
                  q_pos_offset: int = 0, k_pos_offset: int = 0, dq_accumulate: bool = False, dkv_accumulate: bool = False):
    """Backward of "rotate q and k, attend": writes (or, with the accumulate flags, adds to the fp32) dq / dk -- gradients
    of the UN-rotated q and k: RoPE's backward runs in the kernels' epilogues -- and dv in the given buffers (any strides
    with a unit D stride)."""
    if out.dtype != torch.bfloat16:
        raise RuntimeError("attn_bwd_rope: out must be the bf16 forward output")
    _lib.host().attn_bwd(dout, q_rot, [k_rot], [v], lse, sm_scale, bool(causal), int(q_offset), dq, [dk], [dv], bool(dq_accumulate),
                         [bool(dkv_accumulate)], out, None, (cos, sin), int(q_pos_offset), int(k_pos_offset), [], [])
    return dq, dk, dv


# ---- all ring steps of one rank in one launch: K / V as a list of equally shaped chunk tensors
FINAL_TOTAL_DTYPES = (torch.bfloat16,)   # dtypes attn_bwd_chunks can write a chunk's rounded totals in (dk_finals / dv_finals)


def chunks_fit_one_launch(ks, vs) -> bool:
    """True if the chunk tensors can go to the chunk-list entry points as they are: at most 16 bf16 chunks of one shape
    and one stride triple (k's may differ from v's), unit D stride, strides that are multiples of 8, and -- with several
    chunks -- a chunk length over 64 (multiples of 128 leave no partly filled key tile at the end of a chunk)."""
    return _lib.host().chunks_fit(ks, vs)


def _kv_chunks(ks, vs, dks=None, dvs=None, accumulate=None, dk_finals=None, dv_finals=None) -> KvChunks:
    c = KvChunks()
    c.count, c.chunk_len = len(ks), ks[0].size(2)
    mask = 0
    for i, (k, v) in enumerate(zip(ks, vs)):
        c.k[i], c.v[i] = k.data_ptr(), v.data_ptr()
        if dks is not None and dks[i] is not None:
            c.dk[i], c.dv[i] = dks[i].data_ptr(), dvs[i].data_ptr()
            if accumulate is not None and accumulate[i]:
                mask |= 1 << i
        if dk_finals is not None and dk_finals[i] is not None:
            c.dk_final[i], c.dv_final[i] = dk_finals[i].data_ptr(), dv_finals[i].data_ptr()
            c.final_stride[0], c.final_stride[1], c.final_stride[2] = dk_finals[i].stride()[:3]
    c.accumulate_mask = mask
    return c


def _chunk_desc(q, ks, vs, o, sm_scale, causal, q_offset) -> AttnDesc:
    d = _desc(q, ks[0], vs[0], o, sm_scale, causal, q_offset)
    d.Sk = len(ks) * ks[0].size(2)
    return d


def attn_fwd_chunks(q, ks, vs, sm_scale: float, causal: bool, q_offset: int = 0, out=None, lse=None, merge: bool = False,
                    out_dtype=torch.bfloat16, bshd_out: bool = False, rope=None, q_pos_offset: int = 0,
                    want_q_rot: bool = False, checked: bool = False):
    """attn_fwd over K / V given as lists of chunk tensors (see chunks_fit_one_launch) that follow each other along the
    key axis: key j sits at position j of the concatenation, which is never materialised.  rope = (cos, sin): q is
    rotated inside the kernel (the chunks' k must be rotated already).  Returns (out, lse, q_rot or None)."""
    return _lib.host().attn_fwd(q, ks, vs, sm_scale, bool(causal), int(q_offset), out, lse, bool(merge), out_dtype, bshd_out, rope,
                                int(q_pos_offset), want_q_rot, None)


def attn_bwd_chunks(dout, q, ks, vs, lse, sm_scale: float, causal: bool, q_offset: int = 0, dq=None, dks=None, dvs=None,
                    dq_accumulate: bool = False, dkv_accumulate=None, out=None, delta=None, rope=None,
                    q_pos_offset: int = 0, k_pos_offset: int = 0, dk_finals=None, dv_finals=None, checked: bool = False):
    """attn_bwd over a chunk list.  dks / dvs: per chunk a gradient buffer (all of one dtype and stride triple) or None
    (not wanted); dkv_accumulate: per chunk, add to the fp32 buffer instead of writing it.  dq None: not wanted.  With
    `out` (forward output) delta is computed inside the call, otherwise `delta` must be given.  rope = (cos, sin): q and
    the chunks' k are rotated tensors, dq / dk leave un-rotated.  dk_finals / dv_finals: per chunk a bf16 buffer (all of
    one stride triple) or None; where given, this call holds the last block the chunk's gradient waits for, and the
    total -- the fp32 sums in dks / dvs (if the chunk's dkv_accumulate flag is set) plus this block -- is written there,
    rounded once; the fp32 buffers are only read.  Returns delta."""
    return _lib.host().attn_bwd(dout, q, ks, vs, lse, sm_scale, bool(causal), int(q_offset), dq, dks or [], dvs or [], bool(dq_accumulate),
                                dkv_accumulate or [], out, delta, rope, int(q_pos_offset), int(k_pos_offset), dk_finals or [],
                                dv_finals or [])


def attn_bwd_preprocess(dout: torch.Tensor, out: torch.Tensor, dq_acc: Optional[torch.Tensor] = None,
                        delta: Optional[torch.Tensor] = None) -> torch.Tensor:
    """delta = sum(dout * out, -1) as fp32 [B,H,S]; zeroes dq_acc (fp32 contiguous [B,H,S,D]) if given."""
    _dev(dout, out, dq_acc)
    dout = _attn_in(dout, "dout")
    if out.stride() != dout.stride():
        out = _like_strided(out, dout)
    B, H, S, D = dout.shape
    if delta is None:
        delta = torch.empty(B, H, S, dtype=torch.float32, device=dout.device)
    elif not (delta.is_contiguous() and delta.dtype == torch.float32 and delta.numel() == B * H * S):
        raise RuntimeError("attn_bwd_preprocess: delta must be contiguous fp32 [B,H,S]")
    d = _desc(dout, dout, dout, dout, 1.0, False, 0)
    if dq_acc is not None and not (dq_acc.is_contiguous() and dq_acc.dtype == torch.float32):
        raise RuntimeError("attn_bwd_preprocess: dq_acc must be contiguous fp32")
    check(_lib.lib().pico_attn_bwd_preprocess(ctypes.byref(d), _ptr(dout), _ptr(out), _dt(out, "attn out"), _ptr(delta),
                                              _ptr(dq_acc), _stream()))
    return delta


def _like_strided(t: torch.Tensor, ref: torch.Tensor) -> torch.Tensor:
    """Copy of t laid out with ref's strides (so one stride triple describes both)."""
    r = torch.empty_strided(ref.shape, ref.stride(), dtype=t.dtype, device=t.device)
    r.copy_(t)
    return r


def attn_bwd(dout, q, k, v, lse, delta, sm_scale: float, causal: bool, q_offset: int = 0,
             dq: Optional[torch.Tensor] = None, dk: Optional[torch.Tensor] = None, dv: Optional[torch.Tensor] = None,
             dq_accumulate: bool = False, dkv_accumulate: bool = False, dq_dtype=torch.float32,
             dkv_dtype=torch.float32, dq_like: Optional[torch.Tensor] = None, want_dq: bool = True,
             want_dkv: bool = True, side_stream: Optional["torch.cuda.Stream"] = None,
             out: Optional[torch.Tensor] = None, dkv_like: Optional[torch.Tensor] = None):
    """Gradients of one attention block; returns (dq [B,Hq,Sq,D], dk, dv [B,Hkv,Sk,D]).

    Buffers that are passed in are written in place (fp32 ones can be accumulated into: the running dq of a
    rank and the travelling dk / dv of the ring); missing ones are allocated in the requested dtype, dq with
    the strides of `dq_like` if given, dk / dv with the strides of `dkv_like` (so that a gradient for a [B,H,S,D] view
    of [B,S,H,D] memory needs no layout copy on its way back).  want_dq / want_dkv = False skips that gradient.
    With `out` (the forward output) `delta` may be None or a buffer to fill: the row sums delta = sum_d dout * out are
    then computed inside the call (by the dQ kernel itself when out is bf16 and dq is wanted), as in the reference's
    ring_attention_backward, instead of by a separate attn_bwd_preprocess.
    With `side_stream` the dQ kernel is enqueued there and the dK/dV kernel on the current stream (the two are
    independent); the current stream waits for both.  Measured on MI355X it is a wash at the benchmark shape
    (+3 % on one box, -4 % on another: the fork / join costs what the overlapped tails save), so nothing in
    this package turns it on by default.
    """
    _dev(q, k)
    B, Hq, Sq, D = q.shape
    Hkv, Sk = k.size(1), k.size(2)
    if out is not None and side_stream is not None:
        raise RuntimeError("attn_bwd: out= (delta computed by the dQ kernel) orders the two kernels; no side_stream")
    if dq is None and want_dq:
        if dq_accumulate:
            raise RuntimeError("attn_bwd: dq_accumulate=True needs an existing dq")
        if dq_like is not None and _dense(dq_like) and dq_like.stride(-1) == 1 and dq_like.shape == q.shape:
            dq = torch.empty_strided(q.shape, dq_like.stride(), dtype=dq_dtype, device=q.device)
        else:
            dq = torch.empty(B, Hq, Sq, D, dtype=dq_dtype, device=q.device)
    if (dk is None or dv is None) and want_dkv:
        if dkv_accumulate:
            raise RuntimeError("attn_bwd: dkv_accumulate=True needs existing dk / dv")
        if dkv_like is not None and _dense(dkv_like) and dkv_like.stride(-1) == 1 and dkv_like.shape == k.shape:
            dk = torch.empty_strided(k.shape, dkv_like.stride(), dtype=dkv_dtype, device=q.device)
            dv = torch.empty_strided(k.shape, dkv_like.stride(), dtype=dkv_dtype, device=q.device)
        else:
            dk = torch.empty(B, Hkv, Sk, D, dtype=dkv_dtype, device=q.device)
            dv = torch.empty(B, Hkv, Sk, D, dtype=dkv_dtype, device=q.device)
    if not want_dq:
        dq = None
    if not want_dkv:
        dk = dv = None

    def launch(dq_, dk_, dv_):
        _lib.host().attn_bwd(dout, q, [k], [v], lse, sm_scale, bool(causal), int(q_offset), dq_, [dk_], [dv_], bool(dq_accumulate),
                             [bool(dkv_accumulate)], out, delta, None, 0, 0, [], [])

    if side_stream is not None and dq is not None and dk is not None:
        cur = torch.cuda.current_stream()
        side_stream.wait_stream(cur)
        with torch.cuda.stream(side_stream):
            launch(dq, None, None)
        launch(None, dk, dv)
        cur.wait_stream(side_stream)
    else:
        launch(dq, dk, dv)
    return dq, dk, dv


def convert_f32(src: torch.Tensor, dtype, like: Optional[torch.Tensor] = None, bshd: bool = False,
                strides=None) -> torch.Tensor:
    """fp32 contiguous [B,H,S,D] -> dtype; laid out like `like` (same strides) or with the given `strides` (of a
    dense layout with a unit D stride), as a view over [B,S,H,D] memory (bshd=True), or contiguous."""
    _dev(src, like)
    if src.dtype != torch.float32 or not src.is_contiguous() or src.dim() != 4:
        raise RuntimeError("convert_f32: src must be a contiguous fp32 [B,H,S,D] tensor")
    B, H, S, D = src.shape
    if bshd:
        dst = empty_bshd(B, H, S, D, dtype, src.device)
    elif strides is not None:
        dst = torch.empty_strided(src.shape, tuple(strides), dtype=dtype, device=src.device)
        if dst.stride(-1) != 1 or not _dense(dst):
            raise RuntimeError("convert_f32: strides must describe a dense layout with a unit D stride")
    elif like is not None and _dense(like) and like.stride(-1) == 1:
        dst = torch.empty_strided(src.shape, like.stride(), dtype=dtype, device=src.device)
    else:
        dst = torch.empty(src.shape, dtype=dtype, device=src.device)
    check(_lib.lib().pico_convert_f32(_ptr(src), _ptr(dst), B, H, S, D, dst.stride(0), dst.stride(1), dst.stride(2),
                                      _DT[dtype], _stream()))
    return dst


def adamw_(param_lp: Optional[torch.Tensor], master: torch.Tensor, grad: torch.Tensor, exp_avg: torch.Tensor,
           exp_avg_sq: torch.Tensor, step: int, lr: float, beta1: float = 0.9, beta2: float = 0.999, eps: float = 1e-8,
           weight_decay: float = 0.01, grad_scale: float = 1.0) -> None:
    """In-place AdamW step on fp32 (master, exp_avg, exp_avg_sq) from a bf16 / fp32 gradient; rewrites the bf16
    parameter `param_lp` (if given) from the new master weight.  `step` counts from 1."""
    _dev(param_lp, master, grad, exp_avg, exp_avg_sq)
    n = master.numel()
    for t, what in ((master, "master"), (exp_avg, "exp_avg"), (exp_avg_sq, "exp_avg_sq")):
        if t.dtype != torch.float32 or not t.is_contiguous() or t.numel() != n:
            raise RuntimeError(f"adamw_: {what} must be a contiguous fp32 tensor of {n} elements")
    if not grad.is_contiguous() or grad.numel() != n:
        grad = grad.contiguous()
        if grad.numel() != n:
            raise RuntimeError("adamw_: grad has the wrong number of elements")
    if param_lp is not None and (param_lp.dtype != torch.bfloat16 or not param_lp.is_contiguous() or param_lp.numel() != n):
        raise RuntimeError("adamw_: param_lp must be a contiguous bf16 tensor of the same size")
    check(_lib.lib().pico_adamw(_ptr(param_lp), _ptr(master), _ptr(grad), _dt(grad, "grad"), _ptr(exp_avg), _ptr(exp_avg_sq),
                                n, float(lr), float(beta1), float(beta2), float(eps), float(weight_decay), int(step),
                                float(grad_scale), _stream()))


def adamw_lp_(param: torch.Tensor, grad: torch.Tensor, exp_avg: torch.Tensor, exp_avg_sq: torch.Tensor, step: int,
              lr: float, beta1: float = 0.9, beta2: float = 0.999, eps: float = 1e-8, weight_decay: float = 0.01,
              grad_scale: float = 1.0) -> None:
    """In-place AdamW step on a bf16 parameter (no master copy) with fp32 moments, or with bf16 moments (the state
    torch.optim.AdamW holds for a bf16 model); fp32 arithmetic, one rounding per stored value.  `step` counts from 1."""
    _dev(param, grad, exp_avg, exp_avg_sq)
    n = param.numel()
    if param.dtype != torch.bfloat16 or not param.is_contiguous():
        raise RuntimeError("adamw_lp_: param must be a contiguous bf16 tensor")
    sdt = exp_avg.dtype
    for t, what in ((exp_avg, "exp_avg"), (exp_avg_sq, "exp_avg_sq")):
        if t.dtype != sdt or sdt not in _DT or not t.is_contiguous() or t.numel() != n:
            raise RuntimeError(f"adamw_lp_: {what} must be a contiguous bf16 or fp32 tensor of {n} elements")
    if grad.numel() != n:
        raise RuntimeError("adamw_lp_: grad has the wrong number of elements")
    grad = grad.contiguous()
    check(_lib.lib().pico_adamw_lp(_ptr(param), _ptr(grad), _dt(grad, "grad"), _ptr(exp_avg), _ptr(exp_avg_sq), n,
                                   _dt(param, "param"), _DT[sdt], float(lr), float(beta1), float(beta2), float(eps),
                                   float(weight_decay), int(step), float(grad_scale), _stream()))


class AdamWMultiPlan:
    """The AdamW step for a fixed list of tensors in as few launches as they fit (48 tensors each).  Weights, moments
    and sizes are checked and their pointer tables built once; a step only fills in the gradients' addresses, so its
    host cost is a fraction of a millisecond for a few hundred tensors.  All weights share one dtype and both moments
    of all tensors another: fp32 weights with fp32 moments (master weights; `param_lps` optionally lists the bf16
    parameters to rewrite, None entries allowed), or bf16 weights (the parameters themselves; `param_lps` must be None)
    with fp32 or bf16 moments.  The plan keeps the tensors alive."""

    def __init__(self, weights, exp_avgs, exp_avg_sqs, param_lps=None):
        self.count = len(weights)
        self._plan = _lib.host().AdamWPlan(weights, exp_avgs, exp_avg_sqs, param_lps)

    def step(self, grads, step: int, lr: float, beta1: float = 0.9, beta2: float = 0.999, eps: float = 1e-8,
             weight_decay: float = 0.01, grad_scale: float = 1.0) -> None:
        self._plan.step(grads, step, lr, beta1, beta2, eps, weight_decay, grad_scale)

    def step_params(self, params, step: int, lr: float, beta1: float = 0.9, beta2: float = 0.999, eps: float = 1e-8,
                    weight_decay: float = 0.01, grad_scale: float = 1.0) -> bool:
        """The step with the .grad of `params`, the parameters this plan was built for.  False, with nothing done, if a
        gradient is missing, their dtypes differ or a parameter has been moved since."""
        return self._plan.step_params(params, step, lr, beta1, beta2, eps, weight_decay, grad_scale)


def adamw_multi_(weights, grads, exp_avgs, exp_avg_sqs, step: int, lr: float, beta1: float = 0.9, beta2: float = 0.999,
                 eps: float = 1e-8, weight_decay: float = 0.01, grad_scale: float = 1.0, param_lps=None) -> None:
    """One AdamW step for a list of tensors (see AdamWMultiPlan, which a training loop should build once)."""
    if len(weights) == 0 and len(grads) == 0:
        return
    AdamWMultiPlan(weights, exp_avgs, exp_avg_sqs, param_lps).step(grads, step, lr, beta1, beta2, eps, weight_decay, grad_scale)


def cross_entropy_fwd(logits: torch.Tensor, targets: torch.Tensor, ignore_index: int = -100):
    """Per-row loss and logsumexp, both fp32 [rows]."""
    return _lib.host().cross_entropy_fwd(logits, targets, ignore_index)


def cross_entropy_bwd(logits: torch.Tensor, targets: torch.Tensor, lse: torch.Tensor, scale: torch.Tensor,
                      ignore_index: int = -100, inplace: bool = False) -> torch.Tensor:
    """dlogits = (softmax(logits) - onehot(targets)) * scale, scale a one-element fp32 tensor on the device."""
    return _lib.host().cross_entropy_bwd(logits, targets, lse, scale, ignore_index, inplace)
