"""Differentiable ops of the model code on the HIP forward and backward kernels.  The autograd nodes are native
(``csrc/host.cpp``); the classes here keep the ``<Name>.apply(...)`` call shape of ``torch.autograd.Function``."""
from __future__ import annotations

import os

import torch

from . import _lib, ops


class RMSNormFunc:
    """``apply(x, weight, eps, cast_then_scale)``: y = rmsnorm(x) * w.  cast_then_scale selects LlamaRMSNorm's rounding
    order (``model.py:81-86``)."""

    @staticmethod
    def apply(x, weight, eps, cast_then_scale):
        return _lib.host().rms_norm(x, weight, eps, cast_then_scale)


class RMSNormResidualFunc:
    """``apply(x, residual, weight, eps)``: h = x + residual; returns (rmsnorm(h) * w, h) -- the prenorm form of
    flash-attn's layer_norm_fn.  The backward adds h's own gradient inside the kernel."""

    @staticmethod
    def apply(x, residual, weight, eps):
        return _lib.host().rms_norm_residual(x, residual, weight, eps)


class RMSNormHeadFunc:
    """``apply(x, weight, eps)``: returns (rmsnorm(x) * w, x): RMSNormResidualFunc where there is nothing to add yet.  The
    gradients of both outputs meet inside the backward kernel."""

    @staticmethod
    def apply(x, weight, eps):
        return _lib.host().rms_norm_head(x, weight, eps)


class RotaryFunc:
    """``apply(x, cos, sin, pos_offset)``: non-interleaved RoPE on [B,H,S,D]; the backward is the rotation by -theta."""

    @staticmethod
    def apply(x, cos, sin, pos_offset):
        return _lib.host().rotary(x, cos, sin, pos_offset)


class SwiGLUFunc:
    """``apply(gate, up)``: silu(gate) * up (``model.py:186``)."""

    @staticmethod
    def apply(gate, up):
        return _lib.host().swiglu(gate, up)


class FlashAttnFunc:
    """``apply(q, k, v, sm_scale, causal)``: single-chunk causal / dense attention on [B,H,S,D] views; K/V may carry fewer
    (GQA) heads.  Gradients come back in the dtype and memory layout of their inputs."""

    @staticmethod
    def apply(q, k, v, sm_scale, causal):
        return _lib.host().flash_attention(q, k, v, sm_scale, causal, True)


class CrossEntropyFunc:
    """``apply(logits, targets, ignore_index, scale)``: `scale` times the mean cross-entropy of [rows, vocab] logits against
    int64 targets (``train.py:46-49``), fp32 loss.  The gradient leaves in the dtype of the logits; the upstream gradient and the
    1 / count factor reach the kernels through device scalars, so nothing synchronises with the host.  Where a gradient
    will be wanted the forward already writes the gradient for an upstream gradient of 1 (one pass over the logits instead
    of two), so that buffer, as large as the logits, lives from the forward to the backward.  Another upstream gradient makes
    the backward recompute it from the logits, two passes more: a factor that is known beforehand -- the reference divides
    the loss by the accumulation steps (``train.py:29-55``) -- goes into `scale`, where it costs nothing.  A loss that will
    not be differentiated is best computed under ``torch.no_grad()``: nothing is written then."""

    @staticmethod
    def apply(logits, targets, ignore_index=-100, scale=1.0):
        if os.getenv("PICO_CHECK_TARGETS", "0") == "1":
            # F.cross_entropy asserts on the device for a target outside [0, vocab) (train.py:46-49); the kernels skip such
            # a row instead (they may not index with it), which would hide a tokenizer / vocabulary mismatch.  This
            # opt-in check costs a host synchronisation.
            bad = (targets != ignore_index) & ((targets < 0) | (targets >= logits.size(-1)))
            if bool(bad.any()):
                raise RuntimeError(f"cross_entropy: {int(bad.sum())} targets lie outside [0, {logits.size(-1)}) and are not "
                                   f"ignore_index={ignore_index}")
        return _lib.host().cross_entropy(logits, targets, ignore_index, scale)


def cross_entropy(logits, targets, ignore_index: int = -100, scale: float = 1.0):
    """Drop-in for ``F.cross_entropy(logits, targets, reduction='mean')`` on 2-D logits, times `scale`.  With gradient
    accumulation ``cross_entropy(logits, targets, scale=1 / steps).backward()`` is the fast form of
    ``(cross_entropy(logits, targets) / steps).backward()``: [4096, 49152] in bf16 150 us against 293."""
    return CrossEntropyFunc.apply(logits, targets, ignore_index, scale)


# ---------------------------------------------------------------------------------------------------------------
# Fused projections.  The reference's q_proj / k_proj / v_proj (and gate_proj / up_proj) read the same activation;
# their weights are kept as separate Parameters but laid out back to back in one buffer, so one GEMM produces all
# outputs, one GEMM all weight gradients and one GEMM the (already summed) input gradient.  The pieces below hand
# strided views of those fused buffers to the kernels, which take row pitches / element strides as they are, and
# write the pieces of the fused gradient in place: no concatenation, split or layout copy on either pass.

class FusedLinearFunc:
    """``apply(x, w_fused, *parts)``: y = x @ w_fused^T where w_fused is the buffer that the Parameters `parts` (rows of
    it, in order) alias."""

    @staticmethod
    def apply(x, w_fused, *parts):
        return _lib.host().fused_linear(x, w_fused, parts)


def _fused_rope() -> bool:
    """RoPE inside the attention kernels (default); PICO_FUSED_ROPE=0 keeps it a launch of its own over q and k."""
    return os.getenv("PICO_FUSED_ROPE", "1") != "0"


class QKVAttentionFunc:
    """``apply(qkv, cos, sin, n_heads, n_kv_heads, head_dim, causal)``: RoPE on the q and k parts of a fused [B,S,(Hq+2Hkv)*D] projection, then causal / dense attention (one chunk);
    returns [B,S,Hq*D].

    Default: q is rotated inside the attention forward (every query once, in the prologue of the workgroup that owns
    it; the kernel leaves the rotated q behind for the backward), only k -- which many workgroups read -- is rotated by a
    launch of its own, and the backward un-rotates dq and dk in the epilogues of its kernels: one small RoPE launch per
    layer in the forward, none in the backward.  The backward writes dq, dk, dv straight into the matching columns of
    one [B,S,(Hq+2Hkv)*D] buffer.  With PICO_FUSED_ROPE=0 q and k are rotated by one launch (they lie side by side in
    the projection) and dq / dk are un-rotated in place by another."""

    @staticmethod
    def apply(qkv, cos, sin, n_heads, n_kv_heads, head_dim, causal):
        return _lib.host().qkv_attention(qkv, cos, sin, n_heads, n_kv_heads, head_dim, causal, _fused_rope())


class SwiGLUFusedFunc:
    """``apply(gate_up)``: silu(gate) * up where gate and up are the two halves of one [..., 2I] projection output; the
    backward writes dgate and dup into the halves of one [..., 2I] buffer."""

    @staticmethod
    def apply(gate_up):
        return _lib.host().swiglu_fused(gate_up)
