// The host path of the hot ops: tensor checks, output allocation, the C-ABI calls of libpicotron_amd.so and the autograd
// nodes of the model's ops, as one Python extension (picotron_amd/_host.so).
//
// At the small end of the range a call is host work: the kernels of a [2,9,256,64] attention forward + backward take
// 40 us of GPU time, and with torch.autograd.Function classes and ctypes in Python a pass took 180 us, whatever the
// kernels did.  Here a call is one C++ function: no ctypes conversions, no Python frames in the backward (the autograd
// thread never takes the GIL), views replaced by pointer + strides.  Nothing is kept from one call
// for the next but the GEMM library's plans, by shape, and which kernel a product of given sizes goes to.
#include <torch/extension.h>
#include <ATen/Context.h>
#include <ATen/autocast_mode.h>
#include <c10/hip/HIPStream.h>
#include <hipblaslt/hipblaslt.h>

#include <array>
#include <cstdlib>
#include <mutex>
#include <optional>
#include <unordered_map>
#include <vector>

#include "../../include/picotron_amd.h"
#include "product_route.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::Variable;
using torch::autograd::variable_list;
using OptTensor = std::optional<Tensor>;

// ------------------------------------------------------------------------------------------------ small helpers
void check(int rc) { TORCH_CHECK(rc == PICO_OK, "picotron_amd error ", rc, ": ", pico_last_error()); }

void on_gpu(const Tensor& t) {
  TORCH_CHECK(t.is_cuda(), "picotron_amd kernels run on the GPU only: got a CPU tensor (there is no CPU fallback)");
}
void on_gpu(const OptTensor& t) {
  if (t) on_gpu(*t);
}

int dtype_code(const Tensor& t, const char* what) {
  if (t.scalar_type() == at::kBFloat16) return PICO_BF16;
  TORCH_CHECK(t.scalar_type() == at::kFloat, what, ": dtype ", t.scalar_type(), " not supported by the HIP kernels (bf16 / fp32 only)");
  return PICO_F32;
}

void* stream_now() { return c10::hip::getCurrentHIPStream().stream(); }
void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
void* ptr(const OptTensor& t) { return t ? ptr(*t) : nullptr; }
float* fptr(const Tensor& t) { return static_cast<float*>(ptr(t)); }
float* fptr(const OptTensor& t) { return static_cast<float*>(ptr(t)); }

using Stride3 = std::array<int64_t, 3>;
Stride3 strides3(const Tensor& t) { return {t.stride(0), t.stride(1), t.stride(2)}; }
void put(int64_t (&dst)[3], const Stride3& s) {
  for (int i = 0; i < 3; ++i) dst[i] = s[i];
}
// strides of a [B,H,S,D] view of [B,S,H,D] memory: `.transpose(1,2).reshape(B,S,H*D)` on it is free
Stride3 bshd(int64_t H, int64_t S, int64_t D) { return {S * H * D, D, H * D}; }

Tensor empty_bhsd(int64_t B, int64_t H, int64_t S, int64_t D, bool bshd_memory, const at::TensorOptions& o) {
  if (!bshd_memory) return at::empty({B, H, S, D}, o);
  return at::empty_strided({B, H, S, D}, {S * H * D, D, H * D, 1}, o);
}
// fresh tensor laid out like `t` where that layout is dense with a unit last stride, contiguous otherwise
Tensor empty_like_layout(const Tensor& t, const at::TensorOptions& o) {
  if (t.stride(-1) == 1 && t.is_non_overlapping_and_dense()) return at::empty_strided(t.sizes(), t.strides(), o);
  return at::empty(t.sizes(), o);
}

// ------------------------------------------------------------------------------------------------ RMSNorm
struct NormOut {
  Tensor y, rstd, sum;
};

NormOut rmsnorm_forward(const Tensor& x, const Tensor& weight, double eps, bool cast_then_scale, const OptTensor& residual,
                        bool want_sum, bool want_rstd) {
  on_gpu(x);
  on_gpu(weight);
  on_gpu(residual);
  const int64_t hidden = x.size(-1);
  const Tensor xc = x.contiguous();
  const Tensor w = (weight.scalar_type() == x.scalar_type() ? weight : weight.to(x.scalar_type())).contiguous();
  const int64_t rows = hidden ? xc.numel() / hidden : 0;
  Tensor res;
  if (residual) {
    res = residual->contiguous();
    TORCH_CHECK(res.scalar_type() == x.scalar_type() && res.sizes() == x.sizes(), "rmsnorm_fwd: residual must match x in dtype and shape");
  }
  NormOut o;
  o.y = at::empty(xc.sizes(), xc.options());
  if (want_rstd) o.rstd = at::empty({rows}, xc.options().dtype(at::kFloat));
  if (res.defined() && want_sum) o.sum = at::empty(xc.sizes(), xc.options());
  check(pico_rmsnorm_fwd(ptr(xc), ptr(w), ptr(o.y), fptr(o.rstd), ptr(res), ptr(o.sum), rows, hidden, static_cast<float>(eps),
                         cast_then_scale, dtype_code(x, "rmsnorm_fwd"), stream_now()));
  return o;
}

std::pair<Tensor, Tensor> rmsnorm_backward(const Tensor& dy, const Tensor& x, const Tensor& weight, const Tensor& rstd,
                                           const OptTensor& dresidual, at::ScalarType dw_dtype) {
  on_gpu(dy);
  on_gpu(x);
  on_gpu(weight);
  on_gpu(rstd);
  on_gpu(dresidual);
  const int64_t hidden = x.size(-1);
  const auto dt = x.scalar_type();
  const Tensor xc = x.contiguous(), dyc = dy.contiguous().to(dt), w = weight.contiguous().to(dt);
  Tensor dres;
  if (dresidual && dresidual->defined()) {
    TORCH_CHECK(dresidual->sizes() == x.sizes(), "rmsnorm_bwd: dresidual must have x's shape");
    dres = dresidual->contiguous().to(dt);
  }
  const int64_t rows = hidden ? xc.numel() / hidden : 0;
  Tensor dx = at::empty(xc.sizes(), xc.options());
  Tensor dw = at::empty({hidden}, xc.options().dtype(dw_dtype));
  const int64_t bytes = pico_rmsnorm_bwd_workspace_bytes(rows, hidden);
  const Tensor ws = at::empty({std::max<int64_t>(bytes, 16)}, xc.options().dtype(at::kByte));
  check(pico_rmsnorm_bwd(ptr(dyc), ptr(xc), ptr(w), fptr(rstd), ptr(dres), ptr(dx), ptr(dw), dtype_code(dw, "rmsnorm_bwd dweight"),
                         ptr(ws), bytes, rows, hidden, dtype_code(x, "rmsnorm_bwd"), stream_now()));
  return {dx, dw};
}

// y = rmsnorm(x) * w.  cast_then_scale selects LlamaRMSNorm's rounding order (model.py:81-86).
struct RMSNorm : torch::autograd::Function<RMSNorm> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& weight, double eps, bool cast_then_scale) {
    NormOut o = rmsnorm_forward(x, weight, eps, cast_then_scale, std::nullopt, false, true);
    ctx->save_for_backward({x, weight, o.rstd});
    return o.y;
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& g) {
    const auto s = ctx->get_saved_variables();
    auto [dx, dw] = rmsnorm_backward(g[0], s[0], s[1], s[2], std::nullopt, s[1].scalar_type());
    return {dx, dw, Tensor(), Tensor()};
  }
};

// h = x + residual; returns (rmsnorm(h) * w, h): the prenorm form of flash-attn's layer_norm_fn.
struct RMSNormResidual : torch::autograd::Function<RMSNormResidual> {
  static variable_list forward(AutogradContext* ctx, const Tensor& x, const Tensor& residual, const Tensor& weight, double eps) {
    NormOut o = rmsnorm_forward(x, weight, eps, false, residual, true, true);
    ctx->save_for_backward({o.sum, weight, o.rstd});
    ctx->set_materialize_grads(false);   // the last norm's h has no consumer: no zero tensor is made for it
    return {o.y, o.sum};
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& g) {
    const Tensor &dy = g[0], &dh = g[1];
    if (!dy.defined()) return {dh, dh, Tensor(), Tensor()};   // only the residual stream carried a gradient
    const auto s = ctx->get_saved_variables();
    // dh, the gradient that reached h without passing the norm, is added inside the kernel
    auto [dx, dw] = rmsnorm_backward(dy, s[0], s[1], s[2], dh.defined() ? OptTensor(dh) : std::nullopt, s[1].scalar_type());
    return {dx, dx, dw, Tensor()};
  }
};

// (rmsnorm(x) * w, x): the same at the head of a residual stream, where there is nothing to add yet; the gradients of both
// uses of x meet in the kernel instead of in an addition of their own (10 us at [4096, 2048]).
struct RMSNormHead : torch::autograd::Function<RMSNormHead> {
  static variable_list forward(AutogradContext* ctx, const Tensor& x, const Tensor& weight, double eps) {
    NormOut o = rmsnorm_forward(x, weight, eps, false, std::nullopt, false, true);
    ctx->save_for_backward({x, weight, o.rstd});
    ctx->set_materialize_grads(false);
    return {o.y, x};
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& g) {
    const Tensor &dy = g[0], &dh = g[1];
    if (!dy.defined()) return {dh, Tensor(), Tensor()};
    const auto s = ctx->get_saved_variables();
    auto [dx, dw] = rmsnorm_backward(dy, s[0], s[1], s[2], dh.defined() ? OptTensor(dh) : std::nullopt, s[1].scalar_type());
    return {dx, dw, Tensor()};
  }
};

bool records(std::initializer_list<const Tensor*> inputs) {
  if (!at::GradMode::is_enabled()) return false;
  for (const Tensor* t : inputs)
    if (t->requires_grad()) return true;
  return false;
}

// (without a gradient to record -- evaluation -- no node is built and rstd is not written)
Tensor rms_norm(const Tensor& x, const Tensor& weight, double eps, bool cast_then_scale) {
  if (!records({&x, &weight})) return rmsnorm_forward(x, weight, eps, cast_then_scale, std::nullopt, false, false).y;
  return RMSNorm::apply(x, weight, eps, cast_then_scale);
}

std::pair<Tensor, Tensor> rms_norm_head(const Tensor& x, const Tensor& weight, double eps) {
  if (!records({&x})) return {rms_norm(x, weight, eps, false), x};   // (x has no gradient: it passes as it is)
  auto o = RMSNormHead::apply(x, weight, eps);
  return {o[0], o[1]};
}

std::pair<Tensor, Tensor> rms_norm_residual(const Tensor& x, const Tensor& residual, const Tensor& weight, double eps) {
  if (!records({&x, &residual, &weight})) {
    NormOut o = rmsnorm_forward(x, weight, eps, false, residual, true, false);
    return {o.y, o.sum};
  }
  auto o = RMSNormResidual::apply(x, residual, weight, eps);
  return {o[0], o[1]};
}

// ------------------------------------------------------------------------------------------------ RoPE
void check_tables(const Tensor& cos, const Tensor& sin) {
  on_gpu(cos);
  on_gpu(sin);
  TORCH_CHECK(cos.scalar_type() == sin.scalar_type() && cos.dim() == 2 && cos.sizes() == sin.sizes() && cos.stride(-1) == 1 &&
                  sin.stride(-1) == 1 && cos.stride(0) == sin.stride(0),
              "rope tables: cos and sin must be [positions, columns] of one dtype and row pitch, with contiguous rows");
}
pico_rope_tables rope_tables(const Tensor& cos, const Tensor& sin) {
  check_tables(cos, sin);
  return {ptr(cos), ptr(sin), cos.stride(0), dtype_code(cos, "rope tables"), static_cast<int32_t>(cos.size(0))};
}

Tensor rope(const Tensor& x_in, const Tensor& cos, const Tensor& sin, int64_t pos_offset, bool inverse, const OptTensor& out) {
  on_gpu(x_in);
  on_gpu(cos);
  on_gpu(sin);
  on_gpu(out);
  TORCH_CHECK(x_in.dim() == 4, "rope: x must be [B, H, S, D]");
  const Tensor x = x_in.stride(-1) == 1 ? x_in : x_in.contiguous();
  TORCH_CHECK(cos.scalar_type() == sin.scalar_type() && cos.stride(-1) == 1 && sin.stride(-1) == 1 && cos.stride(0) == sin.stride(0),
              "rope: cos and sin must share dtype and row pitch, with contiguous rows");
  TORCH_CHECK(cos.size(0) >= pos_offset + x.size(2), "rope: tables have ", cos.size(0), " rows, need ", pos_offset + x.size(2));
  // the memory order of x is kept, so that a transposed view stays a free view downstream
  const Tensor y = out ? *out : empty_like_layout(x, x.options());
  check(pico_rope(ptr(x), ptr(y), ptr(cos), ptr(sin), x.size(0), x.size(1), x.size(2), x.size(3), x.stride(0), x.stride(1), x.stride(2),
                  y.stride(0), y.stride(1), y.stride(2), cos.stride(0), pos_offset, inverse, dtype_code(cos, "rope tables"),
                  dtype_code(x, "rope"), stream_now()));
  return y;
}

// Non-interleaved RoPE on [B,H,S,D]; the backward is the rotation by -theta.
struct Rotary : torch::autograd::Function<Rotary> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& cos, const Tensor& sin, int64_t pos_offset) {
    ctx->save_for_backward({cos, sin});
    ctx->saved_data["pos"] = pos_offset;
    return rope(x, cos, sin, pos_offset, false, std::nullopt);
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& g) {
    const auto s = ctx->get_saved_variables();
    return {rope(g[0], s[0], s[1], ctx->saved_data["pos"].toInt(), true, std::nullopt), Tensor(), Tensor(), Tensor()};
  }
};

Tensor rotary(const Tensor& x, const Tensor& cos, const Tensor& sin, int64_t pos_offset) {
  if (!records({&x})) return rope(x, cos, sin, pos_offset, false, std::nullopt);
  return Rotary::apply(x, cos, sin, pos_offset);
}

// ------------------------------------------------------------------------------------------------ SwiGLU
// [..., C] as rows of one pitch: the tensor itself where its leading dimensions collapse to one row pitch (a column slice
// of a contiguous buffer does), a contiguous copy otherwise.
struct Rows {
  Tensor t;
  int64_t rows, cols, pitch;
};
bool one_pitch(const Tensor& t) {
  if (t.dim() == 0 || t.stride(-1) != 1) return false;
  for (int64_t i = t.dim() - 3; i >= 0; --i)
    if (t.size(i) != 1 && t.stride(i) != t.stride(i + 1) * t.size(i + 1)) return false;
  return true;
}
Rows as_rows(const Tensor& t_in) {
  const Tensor t = one_pitch(t_in) ? t_in : t_in.contiguous();
  const int64_t cols = t.size(-1), rows = cols ? t.numel() / cols : 0;
  int64_t pitch = cols;
  for (int64_t i = t.dim() - 2; i >= 0; --i)
    if (t.size(i) != 1) { pitch = t.stride(i); break; }
  return {t, rows, cols, pitch < cols ? cols : pitch};
}

Tensor swiglu_forward(const Tensor& gate, const Tensor& up) {
  on_gpu(gate);
  on_gpu(up);
  TORCH_CHECK(gate.sizes() == up.sizes() && gate.scalar_type() == up.scalar_type(), "swiglu_fwd: gate and up must match");
  const Rows g = as_rows(gate), u = as_rows(up);
  Tensor y = at::empty(gate.sizes(), gate.options());
  check(pico_swiglu_fwd(ptr(g.t), ptr(u.t), ptr(y), g.rows, g.cols, g.pitch, u.pitch, g.cols, dtype_code(gate, "swiglu_fwd"), stream_now()));
  return y;
}

std::pair<Tensor, Tensor> swiglu_backward(const Tensor& dy, const Tensor& gate, const Tensor& up, const OptTensor& dgate_out,
                                          const OptTensor& dup_out) {
  on_gpu(dy);
  on_gpu(gate);
  on_gpu(up);
  const Rows g = as_rows(gate), u = as_rows(up), d = as_rows(dy.to(gate.scalar_type()));
  const Tensor dg = dgate_out ? *dgate_out : at::empty(gate.sizes(), gate.options());
  const Tensor du = dup_out ? *dup_out : at::empty(gate.sizes(), gate.options());
  TORCH_CHECK(dg.sizes() == gate.sizes() && du.sizes() == gate.sizes() && dg.scalar_type() == gate.scalar_type() &&
                  du.scalar_type() == gate.scalar_type(),
              "swiglu_bwd: out buffers must match gate in shape and dtype");
  TORCH_CHECK(one_pitch(dg) && one_pitch(du), "swiglu_bwd: out buffers need a unit last stride and one row pitch");
  const Rows dgr = as_rows(dg), dur = as_rows(du);
  check(pico_swiglu_bwd(ptr(d.t), ptr(g.t), ptr(u.t), ptr(dg), ptr(du), g.rows, g.cols, d.pitch, g.pitch, u.pitch, dgr.pitch, dur.pitch,
                        dtype_code(gate, "swiglu_bwd"), stream_now()));
  return {dg, du};
}

// silu(gate) * up (model.py:186)
struct SwiGLU : torch::autograd::Function<SwiGLU> {
  static Tensor forward(AutogradContext* ctx, const Tensor& gate, const Tensor& up) {
    ctx->save_for_backward({gate, up});
    return swiglu_forward(gate, up);
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& g) {
    const auto s = ctx->get_saved_variables();
    auto [dg, du] = swiglu_backward(g[0], s[0], s[1], std::nullopt, std::nullopt);
    return {dg, du};
  }
};
Tensor swiglu(const Tensor& gate, const Tensor& up) {
  if (!records({&gate, &up})) return swiglu_forward(gate, up);
  return SwiGLU::apply(gate, up);
}

// the same where gate and up are the two halves of one [..., 2I] projection output; the backward writes dgate and dup
// into the halves of one [..., 2I] buffer
Tensor swiglu_halves(const Tensor& gate_up) {
  const int64_t half = gate_up.size(-1) / 2;
  return swiglu_forward(gate_up.narrow(-1, 0, half), gate_up.narrow(-1, half, half));
}
struct SwiGLUFused : torch::autograd::Function<SwiGLUFused> {
  static Tensor forward(AutogradContext* ctx, const Tensor& gate_up) {
    ctx->save_for_backward({gate_up});
    return swiglu_halves(gate_up);
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& g) {
    const Tensor gate_up = ctx->get_saved_variables()[0];
    const int64_t half = gate_up.size(-1) / 2;
    Tensor d = at::empty(gate_up.sizes(), gate_up.options());
    swiglu_backward(g[0], gate_up.narrow(-1, 0, half), gate_up.narrow(-1, half, half), d.narrow(-1, 0, half), d.narrow(-1, half, half));
    return {d};
  }
};
Tensor swiglu_fused(const Tensor& gate_up) {
  if (!records({&gate_up})) return swiglu_halves(gate_up);
  return SwiGLUFused::apply(gate_up);
}

// ------------------------------------------------------------------------------------------------ attention
// A [B,H,S,D] operand: first element and element strides (b, h, s); the D stride is 1.
struct Operand {
  void* p;
  Stride3 s;
};

Tensor attn_in(const Tensor& t, const char* what) {
  TORCH_CHECK(t.scalar_type() == at::kBFloat16, "attention: ", what, " must be bf16 (got ", t.scalar_type(), "); the MFMA kernels are bf16 only");
  TORCH_CHECK(t.dim() == 4, "attention: ", what, " must be [B, H, S, D]");
  if (t.stride(3) != 1 || t.stride(0) % 8 || t.stride(1) % 8 || t.stride(2) % 8) return t.contiguous();
  return t;
}
Operand operand(const Tensor& t) { return {ptr(t), strides3(t)}; }

// The two launches with the scratch memory they ask for, from torch's allocator (reused in stream order).
Tensor scratch(int64_t bytes, const at::TensorOptions& o) { return bytes > 0 ? at::empty({bytes}, o.dtype(at::kByte)) : Tensor(); }
void launch_fwd(const pico_attn_desc& d, const void* q, const pico_kv_chunks& kv, void* out, float* lse, int out_dtype, bool merge,
                const pico_rope_tables* rope, int64_t q_pos, void* q_rot, const int64_t* q_rot_stride, const at::TensorOptions& o) {
  const int64_t bytes = pico_attn_fwd_workspace_bytes(&d, kv.count);
  const Tensor ws = scratch(bytes, o);
  check(pico_attn_fwd_chunks_ws(&d, q, &kv, out, lse, out_dtype, merge, rope, static_cast<int>(q_pos), q_rot, q_rot_stride, ptr(ws), bytes,
                                stream_now()));
}
void launch_bwd(const pico_attn_desc& d, const void* q, const pico_kv_chunks& kv, const void* dout, const void* out, int out_dtype,
                const float* lse, float* delta, void* dq, const int64_t* dq_stride, int dq_dtype, bool dq_accumulate,
                const int64_t* dkv_stride, int dkv_dtype, const pico_rope_tables* rope, int64_t q_pos, int64_t k_pos,
                const at::TensorOptions& o) {
  const int64_t bytes = pico_attn_bwd_workspace_bytes(&d, kv.count);
  const Tensor ws = scratch(bytes, o);
  check(pico_attn_bwd_chunks_ws(&d, q, &kv, dout, out, out_dtype, lse, delta, dq, dq_stride, dq_dtype, dq_accumulate, dkv_stride, dkv_dtype,
                                rope, static_cast<int>(q_pos), static_cast<int>(k_pos), ptr(ws), bytes, stream_now()));
}

struct AttnShape {
  int64_t B, Hq, Hkv, Sq, Sk, D;
};
pico_attn_desc attn_desc(const AttnShape& n, const Stride3& q, const Stride3& k, const Stride3& v, const Stride3& o, double sm_scale,
                         bool causal, int64_t q_offset) {
  pico_attn_desc d;
  d.B = static_cast<int32_t>(n.B);
  d.Hq = static_cast<int32_t>(n.Hq);
  d.Hkv = static_cast<int32_t>(n.Hkv);
  d.Sq = static_cast<int32_t>(n.Sq);
  d.Sk = static_cast<int32_t>(n.Sk);
  d.D = static_cast<int32_t>(n.D);
  d.causal = causal;
  d.q_offset = static_cast<int32_t>(q_offset);
  d.sm_scale = static_cast<float>(sm_scale);
  d.reserved = 0;
  put(d.q_stride, q);
  put(d.k_stride, k);
  put(d.v_stride, v);
  put(d.o_stride, o);
  return d;
}

// The chunk tensors can go to the chunk-list entry points as they are: at most PICO_MAX_KV_CHUNKS bf16 chunks of one shape
// and one stride triple (k's may differ from v's), unit D stride, strides that are multiples of 8, and -- with several
// chunks -- a length over 64 (every chunk ends with a partly filled key tile unless its length is a multiple of 128).
bool chunks_fit(const std::vector<Tensor>& ks, const std::vector<Tensor>& vs) {
  if (ks.empty() || ks.size() != vs.size() || ks.size() > PICO_MAX_KV_CHUNKS) return false;
  const Tensor &k0 = ks[0], &v0 = vs[0];
  if (k0.dim() != 4 || v0.dim() != 4 || (ks.size() > 1 && k0.size(2) <= 64)) return false;
  for (const Tensor* t : {&k0, &v0})
    if (t->stride(3) != 1 || t->stride(0) % 8 || t->stride(1) % 8 || t->stride(2) % 8) return false;
  auto fits = [&](const Tensor& t, const Tensor& first) {
    return t.scalar_type() == at::kBFloat16 && t.sizes() == k0.sizes() && t.strides() == first.strides() && t.is_cuda() &&
           reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
  };
  for (size_t i = 0; i < ks.size(); ++i)
    if (!fits(ks[i], k0) || !fits(vs[i], v0)) return false;
  return true;
}

void check_kv(const Tensor& q, const Tensor& k, const Tensor& v) {
  TORCH_CHECK(k.sizes() == v.sizes() && k.size(0) == q.size(0) && k.size(3) == q.size(3), "attention: shape mismatch q", q.sizes(), " k",
              k.sizes(), " v", v.sizes());
}

using Rope = std::optional<std::pair<Tensor, Tensor>>;

// softmax(q k^T * scale + mask) v over one K / V tensor or a list of chunks; returns (out, lse, rotated q or None).
std::tuple<Tensor, Tensor, OptTensor> attn_fwd(const Tensor& q_in, std::vector<Tensor> ks, std::vector<Tensor> vs, double sm_scale,
                                               bool causal, int64_t q_offset, const OptTensor& out_in, const OptTensor& lse_in, bool merge,
                                               at::ScalarType out_dtype, bool bshd_out, const Rope& rope, int64_t q_pos_offset,
                                               bool want_q_rot, const OptTensor& q_rot_in) {
  const at::NoGradGuard no_grad;
  on_gpu(q_in);
  on_gpu(out_in);
  on_gpu(lse_in);
  on_gpu(q_rot_in);
  for (const auto* list : {&ks, &vs})
    for (const Tensor& t : *list) on_gpu(t);
  const Tensor q = attn_in(q_in, "q");
  if (ks.size() == 1 && vs.size() == 1) {
    ks[0] = attn_in(ks[0], "k");
    vs[0] = attn_in(vs[0], "v");
    check_kv(q, ks[0], vs[0]);
  }
  TORCH_CHECK(chunks_fit(ks, vs), "attn_fwd: the K / V chunks do not fit one launch (see chunks_fit_one_launch)");
  check_kv(q, ks[0], vs[0]);
  const int64_t B = q.size(0), Hq = q.size(1), Sq = q.size(2), D = q.size(3);
  TORCH_CHECK(!merge || (out_in && lse_in && out_in->scalar_type() == at::kFloat), "attention: merge=True needs the running fp32 out and lse");
  const Tensor out = out_in ? *out_in : empty_bhsd(B, Hq, Sq, D, bshd_out, q.options().dtype(out_dtype));
  const Tensor lse = lse_in ? *lse_in : at::empty({B, Hq, Sq}, q.options().dtype(at::kFloat));
  TORCH_CHECK(lse.is_contiguous() && lse.scalar_type() == at::kFloat && out.stride(-1) == 1,
              "attention: lse must be contiguous fp32 and out must have a unit D stride");
  pico_kv_chunks kv = {};
  kv.count = static_cast<int32_t>(ks.size());
  kv.chunk_len = static_cast<int32_t>(ks[0].size(2));
  for (size_t i = 0; i < ks.size(); ++i) {
    kv.k[i] = ptr(ks[i]);
    kv.v[i] = ptr(vs[i]);
  }
  pico_attn_desc d = attn_desc({B, Hq, ks[0].size(1), Sq, kv.count * ks[0].size(2), D}, strides3(q), strides3(ks[0]), strides3(vs[0]),
                               strides3(out), sm_scale, causal, q_offset);
  OptTensor q_rot = q_rot_in;
  pico_rope_tables tables;
  Stride3 qrs = {};
  if (rope) {
    tables = rope_tables(rope->first, rope->second);
    if (want_q_rot && !q_rot) q_rot = empty_bhsd(B, Hq, Sq, D, true, q.options());
    if (q_rot) qrs = strides3(*q_rot);
  }
  launch_fwd(d, ptr(q), kv, ptr(out), fptr(lse), dtype_code(out, "attention out"), merge, rope ? &tables : nullptr, q_pos_offset,
             rope ? ptr(q_rot) : nullptr, rope && q_rot ? qrs.data() : nullptr, q.options());
  return {out, lse, rope ? q_rot : std::nullopt};
}

// Copy of t laid out like `ref` (so that one stride triple describes both).
Tensor in_layout_of(const Tensor& t, const Tensor& ref) {
  Tensor r = at::empty_strided(ref.sizes(), ref.strides(), t.options());
  r.copy_(t);
  return r;
}

using OptTensors = std::vector<OptTensor>;

// Backward of attn_fwd into the buffers given (dq, per chunk dk / dv and optionally the bf16 buffers of a chunk's rounded
// total); a missing buffer means that gradient is not wanted.  With `out` delta = sum_d dout * out is computed inside the
// call.  Returns delta.
Tensor attn_bwd(const Tensor& dout_in, const Tensor& q_in, std::vector<Tensor> ks, std::vector<Tensor> vs, const Tensor& lse_in,
                double sm_scale, bool causal, int64_t q_offset, const OptTensor& dq, const OptTensors& dks, const OptTensors& dvs,
                bool dq_accumulate, const std::vector<bool>& dkv_accumulate, const OptTensor& out_in, const OptTensor& delta_in,
                const Rope& rope, int64_t q_pos_offset, int64_t k_pos_offset, const OptTensors& dk_finals, const OptTensors& dv_finals) {
  const at::NoGradGuard no_grad;
  on_gpu(dout_in);
  on_gpu(q_in);
  on_gpu(lse_in);
  on_gpu(dq);
  on_gpu(out_in);
  on_gpu(delta_in);
  for (const auto* list : {&ks, &vs})
    for (const Tensor& t : *list) on_gpu(t);
  const Tensor q = attn_in(q_in, "q");
  Tensor dout = attn_in(dout_in, "dout");
  if (ks.size() == 1 && vs.size() == 1) {
    ks[0] = attn_in(ks[0], "k");
    vs[0] = attn_in(vs[0], "v");
  }
  TORCH_CHECK(chunks_fit(ks, vs), "attn_bwd: the K / V chunks do not fit one launch (see chunks_fit_one_launch)");
  check_kv(q, ks[0], vs[0]);
  TORCH_CHECK(dout.sizes() == q.sizes(), "attention: dout", dout.sizes(), " must have q's shape ", q.sizes());
  const int64_t B = q.size(0), Hq = q.size(1), Sq = q.size(2), D = q.size(3);
  Tensor out;
  if (out_in) {
    out = *out_in;
    TORCH_CHECK(out.sizes() == q.sizes(), "attention: out must have q's shape");
    if (out.strides() != dout.strides()) {
      // one stride triple serves both: dout takes out's layout where the kernels can use that, out dout's otherwise
      if (out.scalar_type() == at::kBFloat16 && out.stride(3) == 1 && out.is_non_overlapping_and_dense() && out.stride(0) % 8 == 0 &&
          out.stride(1) % 8 == 0 && out.stride(2) % 8 == 0)
        dout = in_layout_of(dout, out);
      else
        out = in_layout_of(out, dout = dout.contiguous());
    }
  }
  TORCH_CHECK(out_in || delta_in, "attention backward: delta (or out, to compute it) is required");
  const Tensor delta = !delta_in ? at::empty({B, Hq, Sq}, q.options().dtype(at::kFloat)) : out_in ? *delta_in : delta_in->contiguous();
  TORCH_CHECK(delta.is_contiguous() && delta.scalar_type() == at::kFloat && delta.numel() == B * Hq * Sq,
              "attention backward: delta must be contiguous fp32 [B,H,S]");
  TORCH_CHECK(lse_in.scalar_type() == at::kFloat && lse_in.numel() == B * Hq * Sq, "attention backward: lse must be fp32 [B,H,S]");
  const Tensor lse = lse_in.contiguous();
  TORCH_CHECK(!dq || (dq->stride(-1) == 1 && dq->sizes() == q.sizes()), "attention backward: dq needs q's shape and a unit D stride");

  pico_kv_chunks kv = {};
  const size_t n = ks.size();
  kv.count = static_cast<int32_t>(n);
  kv.chunk_len = static_cast<int32_t>(ks[0].size(2));
  const Tensor *g0 = nullptr, *f0 = nullptr;
  auto pair_ok = [&](const OptTensors& as, const OptTensors& bs, const Tensor*& first, bool bf16_only, const char* what) {
    TORCH_CHECK(as.size() == bs.size() && (as.empty() || as.size() == n), "attention backward: one ", what, " entry per chunk is needed");
    for (size_t i = 0; i < as.size(); ++i) {
      TORCH_CHECK(as[i].has_value() == bs[i].has_value(), "attention backward: ", what, " of a chunk must be given together");
      if (!as[i]) continue;
      if (!first) first = &*as[i];
      for (const Tensor* t : {&*as[i], &*bs[i]})
        TORCH_CHECK(t->is_cuda() && t->scalar_type() == first->scalar_type() && t->strides() == first->strides() && t->stride(-1) == 1 &&
                        t->sizes() == ks[0].sizes() && (!bf16_only || t->scalar_type() == at::kBFloat16),
                    "attention backward: all ", what, " buffers must share dtype", bf16_only ? " (bf16)" : "",
                    " and strides (unit D stride) and have the chunks' shape");
    }
  };
  pair_ok(dks, dvs, g0, false, "dk / dv");
  pair_ok(dk_finals, dv_finals, f0, true, "dk_final / dv_final");
  for (size_t i = 0; i < n; ++i) {
    kv.k[i] = ptr(ks[i]);
    kv.v[i] = ptr(vs[i]);
    if (!dks.empty() && dks[i]) {
      kv.dk[i] = ptr(*dks[i]);
      kv.dv[i] = ptr(*dvs[i]);
      if (i < dkv_accumulate.size() && dkv_accumulate[i]) kv.accumulate_mask |= 1u << i;
    }
    if (!dk_finals.empty() && dk_finals[i]) {
      kv.dk_final[i] = ptr(*dk_finals[i]);
      kv.dv_final[i] = ptr(*dv_finals[i]);
    }
  }
  if (f0) put(kv.final_stride, strides3(*f0));
  const Stride3 dks3 = g0 ? strides3(*g0) : Stride3{}, dqs3 = dq ? strides3(*dq) : Stride3{};
  pico_attn_desc d = attn_desc({B, Hq, ks[0].size(1), Sq, kv.count * ks[0].size(2), D}, strides3(q), strides3(ks[0]), strides3(vs[0]),
                               strides3(dout), sm_scale, causal, q_offset);
  pico_rope_tables tables;
  if (rope) tables = rope_tables(rope->first, rope->second);
  launch_bwd(d, ptr(q), kv, ptr(dout), ptr(out), out.defined() ? dtype_code(out, "out") : PICO_BF16, fptr(lse), fptr(delta), ptr(dq),
             dqs3.data(), dq ? dtype_code(*dq, "dq") : PICO_F32, dq_accumulate, g0 ? dks3.data() : nullptr,
             g0 ? dtype_code(*g0, "dk/dv") : PICO_F32, rope ? &tables : nullptr, q_pos_offset, k_pos_offset, q.options());
  return delta;
}

// Single-chunk causal / dense attention; K/V may carry fewer (GQA) heads.  q, k, v are [B,H,S,D] views; the result is
// [B,S,H,D] (flash_attn_func's layout), or the [B,H,S,D] view of the same memory.
struct FlashAttention : torch::autograd::Function<FlashAttention> {
  static Tensor forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v, double sm_scale, bool causal,
                        bool heads_first) {
    TORCH_CHECK(q.dim() == 4, "attention: q must be [B, H, S, D]");
    const int64_t B = q.size(0), H = q.size(1), S = q.size(2), D = q.size(3);
    // (the result itself must not be a view: it becomes this node's output)
    const Tensor result = heads_first ? empty_bhsd(B, H, S, D, true, q.options()) : at::empty({B, S, H, D}, q.options());
    const Tensor lse = std::get<1>(attn_fwd(q, {k}, {v}, sm_scale, causal, 0, heads_first ? result : result.transpose(1, 2), std::nullopt,
                                            false, at::kBFloat16, true, std::nullopt, 0, false, std::nullopt));
    ctx->save_for_backward({q, k, v, result, lse});
    ctx->saved_data["scale"] = sm_scale;
    ctx->saved_data["causal"] = causal;
    ctx->saved_data["heads_first"] = heads_first;
    return result;
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& g) {
    const auto s = ctx->get_saved_variables();
    const bool heads_first = ctx->saved_data["heads_first"].toBool();
    const Tensor dout = heads_first ? g[0] : g[0].transpose(1, 2), out = heads_first ? s[3] : s[3].transpose(1, 2);
    // delta = sum_d dout * out is computed inside the call; gradients leave in the dtype and memory layout of their
    // inputs: no accumulation buffer, no cast pass
    const Tensor &q = s[0], &k = s[1], &v = s[2];
    Tensor dq = empty_like_layout(q, q.options()), dk, dv;
    if (k.strides() == v.strides()) {
      dk = empty_like_layout(k, k.options());
      dv = empty_like_layout(k, k.options());
    } else {
      dk = at::empty(k.sizes(), k.options());
      dv = at::empty(k.sizes(), k.options());
    }
    attn_bwd(dout, q, {k}, {v}, s[4], ctx->saved_data["scale"].toDouble(), ctx->saved_data["causal"].toBool(), 0, dq, {dk}, {dv}, false,
             {}, out, std::nullopt, std::nullopt, 0, 0, {}, {});
    return {dq, dk, dv, Tensor(), Tensor(), Tensor()};
  }
};

Tensor flash_attention(const Tensor& q, const Tensor& k, const Tensor& v, double sm_scale, bool causal, bool heads_first) {
  on_gpu(q);
  return FlashAttention::apply(q, k, v, sm_scale, causal, heads_first);
}

// ------------------------------------------------------------------------------------------------ ring attention
// The autograd nodes of ring attention over virtual ranks (context_parallel.py) where all ring steps of a rank are one
// launch.  They share one GradBox per published chunk, which belongs to the mailbox's chunk.
// the gradient of a chunk leaves in the chunk's own layout where that is dense with a unit last stride (as k and v share it)
bool dense_layout(const Tensor& t) { return t.stride(-1) == 1 && t.is_non_overlapping_and_dense(); }

// fp32 dK / dV accumulators of one published chunk: what travels round the ring in the reference (context_parallel.py:85-106).
// Every rank's backward adds its block here; the chunk's own autograd node hands the total back once all of them have run.
// All bookkeeping of the sums is here, for the native nodes and for the Python ones (one launch per ring step) alike.
struct GradBox : torch::CustomClassHolder {
  OptTensor dk, dv;               // sums so far; the first block to reach them writes
  OptTensor final_dk, final_dv;   // totals in the chunk's dtype, written by the kernel that completes them
  int64_t readers = 0;            // ranks whose forward read the chunk and will add a block in their backward
  int64_t arrived = 0;            // ... and how many of them have done so since the sums were last handed back
  std::mutex mutex;

  // Where a rank's block goes: added to (add) or written into dk, dv; with final_dk the launch writes bf16(sums so far + block)
  // there instead and reads dk, dv only where there are any.
  struct Share {
    OptTensor dk, dv;
    bool add = false;
    OptTensor final_dk, final_dv;
  };
  // `whole`: the rank's whole block arrives in this launch (not one ring step of it), so that the block every other reader has
  // waited for may leave as the total; `rounds`: the launch can write totals in the chunk's dtype
  Share claim(const Tensor& k, const Tensor& v, bool whole, bool rounds) {
    std::lock_guard<std::mutex> lock(mutex);
    Share s{dk, dv, dk.has_value(), {}, {}};
    if (whole && ++arrived == readers && rounds && k.scalar_type() == v.scalar_type()) {
      const bool own_layout = dense_layout(k) && k.strides() == v.strides();
      auto total = [&] { return own_layout ? at::empty_strided(k.sizes(), k.strides(), k.options()) : at::empty(k.sizes(), k.options()); };
      final_dk = s.final_dk = total();
      final_dv = s.final_dv = total();
    } else if (!s.add) {
      dk = s.dk = at::empty(k.sizes(), k.options().dtype(at::kFloat));
      dv = s.dv = at::empty(k.sizes(), k.options().dtype(at::kFloat));
    }
    return s;
  }
  // What this backward pass left, the totals or else the sums; the next backward through the chunk starts afresh.
  Share take() {
    std::lock_guard<std::mutex> lock(mutex);
    Share s{dk, dv, false, final_dk, final_dv};
    if (final_dk) s.dk = s.dv = std::nullopt;
    dk = dv = final_dk = final_dv = std::nullopt;
    arrived = 0;
    return s;
  }
};
using GradBoxPtr = c10::intrusive_ptr<GradBox>;
struct GradBoxes : torch::CustomClassHolder {
  std::vector<GradBoxPtr> boxes;
  explicit GradBoxes(std::vector<GradBoxPtr> b) : boxes(std::move(b)) {}
};

Tensor convert_sum(const Tensor& src, at::ScalarType dtype, bool dense, at::IntArrayRef strides) {
  Tensor dst = dense ? at::empty_strided(src.sizes(), strides, src.options().dtype(dtype)) : at::empty(src.sizes(), src.options().dtype(dtype));
  check(pico_convert_f32(fptr(src), ptr(dst), src.size(0), src.size(1), src.size(2), src.size(3), dst.stride(0), dst.stride(1), dst.stride(2),
                         dtype_code(dst, "convert_f32"), stream_now()));
  return dst;
}

// Identity on a rank's (k, v) chunk -- with rope tables k is rotated -- that marks where the ring's dK / dV come back: the
// native form of _PublishKV.  It keeps no saved variables: the node may run in several backward calls.
struct PublishKV : torch::autograd::Function<PublishKV> {
  static variable_list forward(AutogradContext* ctx, const Tensor& k, const Tensor& v, const GradBoxPtr& box,
                               const Rope& rope_cs, int64_t pos) {
    ctx->saved_data["box"] = c10::IValue::make_capsule(box);
    ctx->saved_data["dtypes"] = std::vector<int64_t>{static_cast<int64_t>(k.scalar_type()), static_cast<int64_t>(v.scalar_type())};
    ctx->saved_data["k_strides"] = k.strides().vec();
    ctx->saved_data["v_strides"] = v.strides().vec();
    ctx->saved_data["dense"] = std::vector<int64_t>{dense_layout(k), dense_layout(v)};
    ctx->set_materialize_grads(false);
    if (rope_cs) {
      ctx->saved_data["cos"] = rope_cs->first;
      ctx->saved_data["sin"] = rope_cs->second;
      ctx->saved_data["pos"] = pos;
      return {rope(k, rope_cs->first, rope_cs->second, pos, false, std::nullopt), v.variable_data()};
    }
    return {k.variable_data(), v.variable_data()};
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& g) {
    const GradBox::Share left = static_cast<GradBox*>(ctx->saved_data["box"].toCapsule().get())->take();
    OptTensor dk = left.final_dk, dv = left.final_dv;   // (the last reader's kernel wrote the rounded totals itself)
    const auto dtypes = ctx->saved_data["dtypes"].toIntVector(), dense = ctx->saved_data["dense"].toIntVector();
    if (left.dk) {
      dk = convert_sum(*left.dk, static_cast<at::ScalarType>(dtypes[0]), dense[0], ctx->saved_data["k_strides"].toIntVector());
      dv = convert_sum(*left.dv, static_cast<at::ScalarType>(dtypes[1]), dense[1], ctx->saved_data["v_strides"].toIntVector());
    }
    if (g[0].defined()) {   // a gradient that reached the (rotated) chunk some other way
      Tensor gk = g[0];
      if (ctx->saved_data.count("cos"))
        gk = rope(gk, ctx->saved_data["cos"].toTensor(), ctx->saved_data["sin"].toTensor(), ctx->saved_data["pos"].toInt(), true, std::nullopt);
      dk = dk ? *dk + gk : gk;
    }
    if (g[1].defined()) dv = dv ? *dv + g[1] : g[1];
    return {dk.value_or(Tensor()), dv.value_or(Tensor()), Tensor(), Tensor(), Tensor()};
  }
};

std::pair<Tensor, Tensor> publish_kv(const Tensor& k, const Tensor& v, const GradBoxPtr& box, const Rope& rope_cs, int64_t pos) {
  auto r = PublishKV::apply(k, v, box, rope_cs, pos);
  return {r[0], r[1]};
}

// What the launch of a rank's forward left behind, for its backward.
struct RingPass {
  Tensor out, lse, q;   // q: the rotated copy where rope tables are given
  c10::intrusive_ptr<GradBoxes> boxes;
  Rope rope;
  double sm_scale;
  bool causal;
  int64_t q_offset, q_pos, k_pos;
};

// One rank's attention over the chunks it reads (their k, v in the order of their positions).  The forward has run already;
// this node carries its backward: one launch pair for all chunks, whose dK / dV blocks are added to the chunks' fp32 sums
// -- or, where this is the last block a chunk waits for, leave as the chunk's rounded totals.
struct RingAttention : torch::autograd::Function<RingAttention> {
  static Tensor forward(AutogradContext* ctx, const Tensor& q, at::TensorList kvs, const RingPass& p) {
    variable_list saved = {p.q.defined() ? p.q : q, p.lse, p.out};
    for (const Tensor& t : kvs) saved.push_back(t);
    if (p.rope) {
      saved.push_back(p.rope->first);
      saved.push_back(p.rope->second);
    }
    ctx->save_for_backward(saved);
    ctx->saved_data["boxes"] = c10::IValue::make_capsule(p.boxes);
    ctx->saved_data["scale"] = p.sm_scale;
    ctx->saved_data["meta"] = std::vector<int64_t>{p.causal, p.q_offset, p.q_pos, p.k_pos, static_cast<int64_t>(kvs.size() / 2), p.rope.has_value()};
    return p.out;
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& g) {
    const auto s = ctx->get_saved_variables();
    const auto meta = ctx->saved_data["meta"].toIntVector();
    const size_t n = meta[4];
    const Tensor &q = s[0], &lse = s[1], &out = s[2];
    std::vector<Tensor> ks, vs;
    for (size_t i = 0; i < n; ++i) {
      ks.push_back(s[3 + 2 * i]);
      vs.push_back(s[4 + 2 * i]);
    }
    Rope rope_cs;
    if (meta[5]) rope_cs = std::make_pair(s[3 + 2 * n], s[4 + 2 * n]);
    OptTensors dks(n), dvs(n), dk_finals(n), dv_finals(n);
    std::vector<bool> add(n, false);
    bool any_final = false;
    const auto& boxes = static_cast<GradBoxes*>(ctx->saved_data["boxes"].toCapsule().get())->boxes;
    for (size_t i = 0; i < n; ++i) {
      if (!ctx->needs_input_grad(1 + 2 * i) && !ctx->needs_input_grad(2 + 2 * i)) continue;
      const GradBox::Share s = boxes[i]->claim(ks[i], vs[i], true, true);
      dks[i] = s.dk;
      dvs[i] = s.dv;
      add[i] = s.add;
      dk_finals[i] = s.final_dk;
      dv_finals[i] = s.final_dv;
      any_final |= s.final_dk.has_value();
    }
    OptTensor dq;
    if (ctx->needs_input_grad(0)) dq = empty_like_layout(q, q.options());
    attn_bwd(g[0], q, ks, vs, lse, ctx->saved_data["scale"].toDouble(), meta[0], meta[1], dq, dks, dvs, false, add, out, std::nullopt, rope_cs,
             meta[2], meta[3], any_final ? dk_finals : OptTensors(), any_final ? dv_finals : OptTensors());
    variable_list r(2 + 2 * n);
    r[0] = dq.value_or(Tensor());
    return r;
  }
};

Tensor ring_node(const Tensor& q, const std::vector<Tensor>& ks, const std::vector<Tensor>& vs, const Tensor& out, const Tensor& lse,
                 const OptTensor& q_rot, const std::vector<GradBoxPtr>& boxes, double sm_scale, bool causal, int64_t q_offset,
                 const Rope& rope_cs, int64_t q_pos, int64_t k_pos) {
  RingPass p = {out, lse, q_rot.value_or(Tensor()), c10::make_intrusive<GradBoxes>(boxes), rope_cs, sm_scale, causal, q_offset, q_pos, k_pos};
  std::vector<Tensor> kvs;
  for (size_t i = 0; i < ks.size(); ++i) {
    kvs.push_back(ks[i]);
    kvs.push_back(vs[i]);
  }
  return RingAttention::apply(q, at::TensorList(kvs), p);
}

// ------------------------------------------------------------------------------------------------ projections
// The model's large matrix products are plain library GEMMs (hipBLASLt, the library torch calls too).  torch asks the library's
// heuristic for an algorithm on every call, which is most of the 25-30 us of host time a product costs there; here the
// answer is kept with the shape, and a product costs its launch.  At most kMaxPlans shapes are kept; all are dropped when
// one more is asked for.
class GemmPlans {
 public:
  // parts > 1: k is cut into that many equal pieces whose products, each in fp32, lie one after the other in C
  struct Shape {
    int64_t device, ta, tb, m, n, k, lda, ldb, parts;
    bool operator==(const Shape& o) const {
      return device == o.device && ta == o.ta && tb == o.tb && m == o.m && n == o.n && k == o.k && lda == o.lda && ldb == o.ldb && parts == o.parts;
    }
  };

  // column-major C[m,n] = op(A) op(B), bf16 in, bf16 (or, in parts, fp32) out, fp32 accumulation; false: the library has no
  // algorithm for it
  bool run(const Shape& s, const void* a, const void* b, void* c, const at::TensorOptions& options) {
    std::lock_guard<std::mutex> lock(mutex_);   // (several host threads may come here with one device's handle)
    auto it = plans_.find(s);
    if (it == plans_.end()) {
      if (plans_.size() >= kMaxPlans) clear();
      it = plans_.emplace(s, make(s)).first;
    }
    const Plan& p = it->second;
    if (!p.usable) return false;
    Tensor ws;   // (from torch's allocator: reused in stream order, safe with several streams)
    if (p.ws_bytes) ws = at::empty({static_cast<int64_t>(p.ws_bytes)}, options.dtype(at::kByte));
    const float one = 1.f, zero = 0.f;
    const auto rc = hipblasLtMatmul(handles_[s.device], p.desc, &one, a, p.a, b, p.b, &zero, c, p.c, c, p.c, &p.algo, ptr(ws), p.ws_bytes,
                                    c10::hip::getCurrentHIPStream().stream());
    TORCH_CHECK(rc == HIPBLAS_STATUS_SUCCESS, "hipblasLtMatmul failed with status ", static_cast<int>(rc));
    return true;
  }

 private:
  static constexpr size_t kMaxPlans = 1024;
  static constexpr uint64_t kMaxWorkspace = 76ull << 20;
  struct Plan {
    hipblasLtMatmulDesc_t desc = nullptr;
    hipblasLtMatrixLayout_t a = nullptr, b = nullptr, c = nullptr;
    hipblasLtMatmulAlgo_t algo = {};
    size_t ws_bytes = 0;
    bool usable = false;
  };
  struct Hash {
    size_t operator()(const Shape& s) const {
      uint64_t h = 1469598103934665603ull;
      for (int64_t v : {s.device, s.ta, s.tb, s.m, s.n, s.k, s.lda, s.ldb, s.parts}) h = (h ^ static_cast<uint64_t>(v)) * 1099511628211ull;
      return static_cast<size_t>(h ^ (h >> 29));
    }
  };

  static void ok(hipblasStatus_t rc, const char* what) {
    TORCH_CHECK(rc == HIPBLAS_STATUS_SUCCESS, what, " failed with status ", static_cast<int>(rc));
  }
  Plan make(const Shape& s) {
    auto& handle = handles_[s.device];
    if (!handle) ok(hipblasLtCreate(&handle), "hipblasLtCreate");
    Plan p;
    ok(hipblasLtMatmulDescCreate(&p.desc, HIPBLAS_COMPUTE_32F, HIP_R_32F), "hipblasLtMatmulDescCreate");
    const int32_t op_a = s.ta ? HIPBLAS_OP_T : HIPBLAS_OP_N, op_b = s.tb ? HIPBLAS_OP_T : HIPBLAS_OP_N;
    ok(hipblasLtMatmulDescSetAttribute(p.desc, HIPBLASLT_MATMUL_DESC_TRANSA, &op_a, sizeof op_a), "TRANSA");
    ok(hipblasLtMatmulDescSetAttribute(p.desc, HIPBLASLT_MATMUL_DESC_TRANSB, &op_b, sizeof op_b), "TRANSB");
    const int64_t k = s.k / s.parts;
    ok(hipblasLtMatrixLayoutCreate(&p.a, HIP_R_16BF, s.ta ? k : s.m, s.ta ? s.m : k, s.lda), "layout A");
    ok(hipblasLtMatrixLayoutCreate(&p.b, HIP_R_16BF, s.tb ? s.n : k, s.tb ? k : s.n, s.ldb), "layout B");
    ok(hipblasLtMatrixLayoutCreate(&p.c, s.parts > 1 ? HIP_R_32F : HIP_R_16BF, s.m, s.n, s.m), "layout C");
    if (s.parts > 1) {
      const int32_t count = static_cast<int32_t>(s.parts);
      const int64_t step_a = s.ta ? k : k * s.lda, step_b = s.tb ? k * s.ldb : k, step_c = s.m * s.n;
      for (auto [layout, step] : {std::pair(p.a, step_a), std::pair(p.b, step_b), std::pair(p.c, step_c)}) {
        ok(hipblasLtMatrixLayoutSetAttribute(layout, HIPBLASLT_MATRIX_LAYOUT_BATCH_COUNT, &count, sizeof count), "batch count");
        ok(hipblasLtMatrixLayoutSetAttribute(layout, HIPBLASLT_MATRIX_LAYOUT_STRIDED_BATCH_OFFSET, &step, sizeof step), "batch stride");
      }
    }
    hipblasLtMatmulPreference_t pref = nullptr;
    ok(hipblasLtMatmulPreferenceCreate(&pref), "hipblasLtMatmulPreferenceCreate");
    const uint64_t ws = kMaxWorkspace;
    ok(hipblasLtMatmulPreferenceSetAttribute(pref, HIPBLASLT_MATMUL_PREF_MAX_WORKSPACE_BYTES, &ws, sizeof ws), "workspace preference");
    hipblasLtMatmulHeuristicResult_t best = {};
    int found = 0;
    const auto rc = hipblasLtMatmulAlgoGetHeuristic(handle, p.desc, p.a, p.b, p.c, p.c, pref, 1, &best, &found);
    hipblasLtMatmulPreferenceDestroy(pref);
    if (rc == HIPBLAS_STATUS_SUCCESS && found > 0) {
      p.algo = best.algo;
      p.ws_bytes = best.workspaceSize;
      p.usable = true;
    }
    return p;
  }
  void clear() {
    for (auto& [shape, p] : plans_) {
      hipblasLtMatrixLayoutDestroy(p.a);
      hipblasLtMatrixLayoutDestroy(p.b);
      hipblasLtMatrixLayoutDestroy(p.c);
      hipblasLtMatmulDescDestroy(p.desc);
    }
    plans_.clear();
  }

  std::mutex mutex_;
  std::unordered_map<int64_t, hipblasLtHandle_t> handles_;   // per device, kept until the process ends
  std::unordered_map<Shape, Plan, Hash> plans_;
};

GemmPlans& gemm_plans() {
  static GemmPlans* plans = new GemmPlans;   // never destroyed: the library may be gone before static destructors run
  return *plans;
}

// The product is one for the plans above: bf16 on the GPU, rows of one pitch, 16-byte aligned, and no torch setting asks for
// another route (autocast, another BLAS backend, TunableOp; PICO_TORCH_GEMM=1 sends every product through torch).
bool torch_gemm_only() {
  static const bool v = [] {
    auto on = [](const char* name) { const char* e = std::getenv(name); return e && std::string(e) == "1"; };
    return on("PICO_TORCH_GEMM") || on("PYTORCH_TUNABLEOP_ENABLED");
  }();
  return v || at::autocast::is_autocast_enabled(at::kCUDA) ||
         (at::globalContext().blasPreferredBackend() != at::BlasBackend::Default &&
          at::globalContext().blasPreferredBackend() != at::BlasBackend::Cublaslt);
}
bool plain(const Tensor& t) {
  return t.is_cuda() && t.scalar_type() == at::kBFloat16 && t.dim() == 2 && t.stride(1) == 1 && t.stride(0) >= t.size(1) &&
         reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0 && t.numel() > 0;
}
Tensor matrix(const Tensor& t) { return t.dim() == 2 ? t : t.reshape({-1, t.size(-1)}); }

// Ordinary tensors in ordinary code: no forward-mode tangent, no wrapper (vmap, torch.func transforms, functionalization,
// __torch_dispatch__ subclasses, lazy conj / neg) and no dispatch mode or tracer that has to see the operators.  Where this is
// not so an op that torch has goes through torch.
bool ordinary(std::initializer_list<const Tensor*> inputs) {
  using K = c10::DispatchKey;
  static constexpr c10::DispatchKeySet wrapped({K::Python, K::FuncTorchBatched, K::FuncTorchGradWrapper, K::BatchedNestedTensor,
                                                K::Functionalize, K::Conjugate, K::Negative, K::ZeroTensor});
  static constexpr c10::DispatchKeySet modes({K::Python, K::PythonTLSSnapshot, K::FuncTorchDynamicLayerFrontMode, K::FuncTorchVmapMode,
                                              K::Functionalize, K::Tracer});
  if (c10::impl::tls_local_dispatch_key_set().included_.has_any(modes)) return false;
  for (const Tensor* t : inputs)
    if (t->key_set().has_any(wrapped) || t->_fw_grad(0).defined()) return false;
  return true;
}

// [K, N] -> [N, K], rows padded to 16 bytes
Tensor turned(const Tensor& t) {
  const int64_t K = t.size(0), N = t.size(1), pitch = (K + 7) / 8 * 8;
  Tensor y = at::empty({N, pitch}, t.options());
  check(pico_transpose(ptr(t), ptr(y), K, N, t.stride(0), pitch, stream_now()));
  return y;
}

ProductSizes product_sizes(const Tensor& a, const Tensor& b, Product kind) {
  const ProductSizes n = {kind == Product::TN ? a.size(1) : a.size(0), kind == Product::NT ? b.size(0) : b.size(1),
                          kind == Product::TN ? a.size(0) : a.size(1), a.stride(0), b.stride(0)};
  TORCH_CHECK((kind == Product::NT ? b.size(1) : b.size(0)) == n.K, "matrix product: shapes ", a.sizes(), " and ", b.sizes(), " do not match");
  return n;
}
Tensor torch_product(const Tensor& a, const Tensor& b, Product kind) {
  return kind == Product::NT ? at::mm(a, b.t()) : kind == Product::NN ? at::mm(a, b) : at::mm(a.t(), b);
}
// What torch would do differently, or refuse (operands on two devices), stays with torch.
bool stays_with_torch(const Tensor& a, const Tensor& b) {
  // (a backward that is itself to be differentiated, create_graph, stays with torch)
  const bool recorded = at::GradMode::is_enabled() && (a.requires_grad() || b.requires_grad());
  return recorded || !ordinary({&a, &b}) || !plain(a) || !plain(b) || a.device() != b.device() || torch_gemm_only();
}

// a product in the kernel of its route; the operands do not stay with torch
Tensor product(const Tensor& a, const Tensor& b, Product kind, const ProductSizes& n, const ProductRoute& route) {
  const c10::OptionalDeviceGuard device(a.device());
  const auto [M, N, K, lda, ldb] = n;
  const int a_slow = kind == Product::TN, b_slow = kind != Product::NT, tile_m = static_cast<int>(route.tile_m), tile_n = static_cast<int>(route.tile_n);
  const int parts = static_cast<int>(route.parts);
  TORCH_CHECK(parts >= 1 && (route.kernel != ProductRoute::Library || K % parts == 0), "matrix product: a contraction of ", K, " cannot be cut into ", parts, " equal pieces");
  Tensor c = at::empty({M, N}, a.options());
  const Tensor sums = parts > 1 ? at::empty({parts, M, N}, a.options().dtype(at::kFloat)) : Tensor();
  void* out = parts > 1 ? ptr(sums) : ptr(c);
  switch (route.kernel) {
    case ProductRoute::Own:
      check(pico_product(ptr(a), ptr(b), ptr(c), M, N, K, lda, ldb, a_slow, b_slow, tile_m, static_cast<int>(route.groups), stream_now()));
      return c;
    case ProductRoute::Mid:
      check(pico_product_mid(ptr(a), ptr(b), out, M, N, K, lda, ldb, a_slow, b_slow, tile_m, tile_n, parts, stream_now()));
      break;
    case ProductRoute::Large:
      check(pico_product_large(ptr(a), ptr(b), out, M, N, K, lda, ldb, a_slow, b_slow, tile_m, tile_n, parts, stream_now()));
      break;
    case ProductRoute::Library: {
      // row-major C = op(a) op(b) is column-major C^T = op(b)^T op(a)^T: the operands change places
      const Tensor at_ = route.turn & 1 ? turned(a) : a, bt = route.turn & 2 ? turned(b) : b;
      GemmPlans::Shape s = {a.device().index(), kind == Product::NT || (route.turn & 2), kind == Product::TN && !(route.turn & 1), N, M, K,
                            bt.stride(0), at_.stride(0), parts};
      if (gemm_plans().run(s, bt.data_ptr(), at_.data_ptr(), out, a.options())) break;
      s.parts = 1;
      if (parts > 1 && gemm_plans().run(s, bt.data_ptr(), at_.data_ptr(), c.data_ptr(), a.options())) return c;
      return torch_product(a, b, kind);
    }
  }
  if (parts > 1) check(pico_sum_parts(fptr(sums), ptr(c), parts, M * N, PICO_BF16, stream_now()));
  return c;
}
Tensor product(const Tensor& a, const Tensor& b, Product kind) {
  if (stays_with_torch(a, b)) return torch_product(a, b, kind);
  const ProductSizes n = product_sizes(a, b, kind);
  return product(a, b, kind, n, product_route(kind, n));
}

// dx = dy w and dw = dy^T x, in one launch where neither fills the GPU for long by itself: the launch of the second product and the
// idle CUs of both are what it saves.  Us apart and together:
//   [512 x 576] and [576 x 576] 8.8, 5.2; [512 x 3072] and [3072 x 576] 16.2, 13.1; [2331 x 960] and [960 x 576] 17.9, 14.0; [1024
//   x 1024] and [1024 x 1024] 15.1, 10.4.
// The tiles of both are chosen together: their times alike mid_time's, and the workgroups dealt to 256 CUs, the longer ones first; 7.7 %
// error over 8900 timed (layer, tiles), 2 % over the best tiles in the mean.  It is taken where it promises 0.94 of the two products'
// estimates: of 557 drawn layers (64 .. 5000 rows, 192 .. 2400 columns in, up to 5.3 times that out) 494, which take 0.75 of the time in
// the geometric mean, four over 1.02 and 1.15 at most; the others would take 0.95 ([1309 x 1688] and [1688 x 1688] 30.8, 37.3).
struct Gradients {
  Tensor dx, dw;
};
GradientTiles gradient_tiles(const Tensor& dy, const Tensor& w, const Tensor& x) {
  if (stays_with_torch(dy, w) || stays_with_torch(dy, x)) return {};
  const ProductSizes n = product_sizes(dy, w, Product::NN);
  const int64_t rows = n.M, in = n.N, out = n.K;
  product_sizes(dy, x, Product::TN);
  if (rows < 1 || in < 1 || out < 1 || !pico_product_mid_takes(rows, in, out, dy.stride(0), w.stride(0), 0, 1) ||
      !pico_product_mid_takes(out, in, rows, dy.stride(0), x.stride(0), 1, 1))
    return {};
  return gradient_tiles(rows, out, in);
}
Gradients gradients(const Tensor& dy, const Tensor& w, const Tensor& x, const GradientTiles& tiles) {
  if (tiles.dx.tile_m == 0) return {product(dy, w, Product::NN), product(dy, x, Product::TN)};
  const c10::OptionalDeviceGuard device(dy.device());
  const int64_t rows = dy.size(0), out = dy.size(1), in = w.size(1);
  Gradients r = {at::empty({rows, in}, dy.options()), at::empty({out, in}, dy.options())};
  check(pico_product_pair(ptr(dy), ptr(w), ptr(x), ptr(r.dx), ptr(r.dw), rows, out, in, dy.stride(0), w.stride(0), x.stride(0),
                          static_cast<int>(tiles.dx.tile_m), static_cast<int>(tiles.dx.tile_n), static_cast<int>(tiles.dw.tile_m),
                          static_cast<int>(tiles.dw.tile_n), stream_now()));
  return r;
}
Gradients gradients(const Tensor& dy, const Tensor& w, const Tensor& x) { return gradients(dy, w, x, gradient_tiles(dy, w, x)); }

Tensor linear_forward(const Tensor& x, const Tensor& w) {
  if (x.dim() < 1 || w.dim() != 2 || !x.is_cuda() || x.scalar_type() != at::kBFloat16 || torch_gemm_only() || !ordinary({&x, &w}))
    return at::linear(x, w);
  const Tensor y = product(matrix(x), w, Product::NT);
  if (x.dim() == 2) return y;
  auto sizes = x.sizes().vec();
  sizes.back() = w.size(0);
  return y.view(sizes);
}

// y = x @ w^T; each operand is kept only for the other's gradient (a frozen weight keeps no activations)
struct Linear : torch::autograd::Function<Linear> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& w) {
    ctx->save_for_backward({w.requires_grad() ? x : Tensor(), x.requires_grad() ? w : Tensor()});
    ctx->saved_data["sizes"] = x.sizes().vec();
    return linear_forward(x, w);
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& g) {
    const auto s = ctx->get_saved_variables();
    const Tensor dy = matrix(g[0]);
    variable_list r(2);
    if (ctx->needs_input_grad(0) && ctx->needs_input_grad(1)) {
      Gradients d = gradients(dy, s[1], matrix(s[0]));
      return {d.dx.view(ctx->saved_data["sizes"].toIntVector()), d.dw};
    }
    if (ctx->needs_input_grad(0)) r[0] = product(dy, s[1], Product::NN).view(ctx->saved_data["sizes"].toIntVector());
    if (ctx->needs_input_grad(1)) r[1] = product(dy, matrix(s[0]), Product::TN);
    return r;
  }
};
Tensor linear(const Tensor& x, const Tensor& w) {
  if (!x.is_cuda() || x.scalar_type() != at::kBFloat16 || w.scalar_type() != at::kBFloat16 || torch_gemm_only() || !ordinary({&x, &w}))
    return at::linear(x, w);
  return records({&x, &w}) ? Linear::apply(x, w) : linear_forward(x, w);
}

// y = x @ w^T where w is the buffer that the Parameters `parts` (rows of it, in order) alias; one GEMM for all outputs, one
// for all weight gradients, one for the summed input gradient.
struct FusedLinear : torch::autograd::Function<FusedLinear> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& w, at::TensorList parts) {
    ctx->save_for_backward({x, w});
    std::vector<int64_t> rows;
    for (const Tensor& p : parts) rows.push_back(p.size(0));
    ctx->saved_data["rows"] = rows;
    return linear_forward(x, w);
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& g) {
    const auto s = ctx->get_saved_variables();
    const Tensor &x = s[0], &w = s[1];
    const auto rows = ctx->saved_data["rows"].toIntVector();
    const Tensor dy = matrix(g[0]);
    variable_list r(2 + rows.size());
    bool any = false;
    for (size_t i = 0; i < rows.size(); ++i) any |= ctx->needs_input_grad(2 + i);
    Gradients d;
    if (any && ctx->needs_input_grad(0)) d = gradients(dy, w, matrix(x));
    else if (any) d.dw = product(dy, matrix(x), Product::TN);
    else if (ctx->needs_input_grad(0)) d.dx = product(dy, w, Product::NN);
    if (ctx->needs_input_grad(0)) r[0] = d.dx.view(x.sizes());
    if (any) {
      const Tensor& dw = d.dw;
      int64_t at_row = 0;
      for (size_t i = 0; i < rows.size(); ++i, at_row += rows[i - 1]) r[2 + i] = dw.narrow(0, at_row, rows[i]);
    }
    return r;
  }
};

Tensor fused_linear(const Tensor& x, const Tensor& w, const std::vector<Tensor>& parts) {
  if (!at::GradMode::is_enabled()) return linear_forward(x, w);
  return FusedLinear::apply(x, w, at::TensorList(parts));
}

// ------------------------------------------------------------------------------------------------ embedding
// torch's gather; the gradient is a kernel here (torch's, with a sort of its own, takes 155 us in 13 launches for 4096 tokens
// of 2048 columns and 44 us for 1024 of 576).
struct Embedding : torch::autograd::Function<Embedding> {
  static Tensor forward(AutogradContext* ctx, const Tensor& ids, const Tensor& weight, int64_t padding_idx) {
    ctx->save_for_backward({ids});
    ctx->saved_data["rows"] = weight.size(0);
    ctx->saved_data["padding_idx"] = padding_idx;
    return at::embedding(weight, ids, padding_idx);
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& g) {
    const Tensor ids = ctx->get_saved_variables()[0].contiguous(), dy = g[0].contiguous();
    const int64_t rows = ctx->saved_data["rows"].toInt(), padding_idx = ctx->saved_data["padding_idx"].toInt();
    const int64_t tokens = ids.numel(), hidden = dy.size(-1);
    // (a gradient that is itself to be differentiated stays with torch)
    if (tokens < 1 || tokens > PICO_EMBEDDING_MAX_TOKENS || hidden % 8 || hidden < 8 || hidden > (1 << 20) || at::GradMode::is_enabled() ||
        (dy.scalar_type() != at::kBFloat16 && dy.scalar_type() != at::kFloat) || reinterpret_cast<uintptr_t>(dy.data_ptr()) % 16)
      return {Tensor(), at::embedding_dense_backward(dy, ids, rows, padding_idx, false), Tensor()};
    Tensor dw = at::empty({rows, hidden}, dy.options());
    const Tensor ws = at::empty({pico_embedding_bwd_workspace_bytes(tokens, hidden)}, dy.options().dtype(at::kByte));
    check(pico_embedding_bwd(ptr(ids), static_cast<int>(ids.element_size()), ptr(dy), ptr(dw), ptr(ws), tokens, rows, hidden, padding_idx,
                             dtype_code(dy, "embedding"), stream_now()));
    return {Tensor(), dw, Tensor()};
  }
};
Tensor embedding(const Tensor& ids, const Tensor& weight, int64_t padding_idx) {
  if (!records({&weight}) || !weight.is_cuda() || (ids.scalar_type() != at::kLong && ids.scalar_type() != at::kInt) ||
      !ordinary({&ids, &weight}))
    return at::embedding(weight, ids, padding_idx);
  return Embedding::apply(ids, weight, padding_idx);
}

// RoPE on the q and k parts of a fused [B,S,(Hq+2Hkv)*D] projection, then causal / dense attention; returns [B,S,Hq*D].
// `in_kernel`: q is rotated inside the attention forward (which leaves the rotated q behind for the backward), k by a
// launch of its own, and the backward un-rotates dq and dk in the epilogues of its kernels; otherwise q and k are rotated
// by one launch (they lie side by side in the projection) and dq / dk un-rotated in place by another.  The backward writes
// dq, dk, dv into the matching columns of one buffer.
struct QKVShape {
  AttnShape n;
  int64_t width;
  Operand q, k, v;
};
QKVShape qkv_parts(const Tensor& qkv, int64_t Hq, int64_t Hkv, int64_t D) {
  const int64_t B = qkv.size(0), S = qkv.size(1), W = qkv.size(2);
  TORCH_CHECK(W == (Hq + 2 * Hkv) * D, "attention: the fused projection has ", W, " columns, expected ", (Hq + 2 * Hkv) * D);
  auto* base = static_cast<char*>(qkv.data_ptr());
  const Stride3 s = {S * W, D, W};
  return {{B, Hq, Hkv, S, S, D}, W, {base, s}, {base + 2 * Hq * D, s}, {base + 2 * (Hq + Hkv) * D, s}};
}
pico_kv_chunks one_chunk(const AttnShape& n, void* k, void* v, void* dk, void* dv) {
  pico_kv_chunks kv = {};
  kv.count = 1;
  kv.chunk_len = static_cast<int32_t>(n.Sk);
  kv.k[0] = k;
  kv.v[0] = v;
  kv.dk[0] = dk;
  kv.dv[0] = dv;
  return kv;
}

struct QKVForward {
  Tensor out, lse, qk;   // qk: the rotated q and k, side by side as [B,S,(Hq+Hkv)*D], or the rotated q in front of k's own buffer
};

// rotates `heads` heads lying side by side in rows of pitch x.s[2] (element strides) into y
void rope_heads(const Operand& x, const Operand& y, const Tensor& cos, const Tensor& sin, int64_t B, int64_t heads, int64_t S, int64_t D,
                bool inverse) {
  check_tables(cos, sin);
  TORCH_CHECK(cos.size(0) >= S, "rope: tables have ", cos.size(0), " rows, need ", S);
  check(pico_rope(x.p, y.p, ptr(cos), ptr(sin), B, heads, S, D, x.s[0], x.s[1], x.s[2], y.s[0], y.s[1], y.s[2], cos.stride(0), 0, inverse,
                  dtype_code(cos, "rope tables"), PICO_BF16, stream_now()));
}

QKVForward qkv_forward(const Tensor& qkv, const Tensor& cos, const Tensor& sin, int64_t Hq, int64_t Hkv, int64_t D, bool causal,
                       double sm_scale, bool in_kernel) {
  const QKVShape m = qkv_parts(qkv, Hq, Hkv, D);
  const int64_t B = m.n.B, S = m.n.Sq, W = (Hq + Hkv) * D;
  QKVForward r;
  r.qk = at::empty({B, S, W}, qkv.options());
  r.out = at::empty({B, S, Hq * D}, qkv.options());
  r.lse = at::empty({B, Hq, S}, qkv.options().dtype(at::kFloat));
  auto* base = static_cast<char*>(r.qk.data_ptr());
  const Operand q_rot = {base, {S * W, D, W}}, k_rot = {base + 2 * Hq * D, {S * W, D, W}};
  const Stride3 o = bshd(Hq, S, D);
  pico_kv_chunks kv = one_chunk(m.n, k_rot.p, m.v.p, nullptr, nullptr);
  if (in_kernel) {
    rope_heads(m.k, k_rot, cos, sin, B, Hkv, S, D, false);
    pico_rope_tables tables = rope_tables(cos, sin);
    pico_attn_desc d = attn_desc(m.n, m.q.s, k_rot.s, m.v.s, o, sm_scale, causal, 0);
    launch_fwd(d, m.q.p, kv, ptr(r.out), fptr(r.lse), PICO_BF16, false, &tables, 0, q_rot.p, q_rot.s.data(), qkv.options());
  } else {
    rope_heads(m.q, q_rot, cos, sin, B, Hq + Hkv, S, D, false);
    pico_attn_desc d = attn_desc(m.n, q_rot.s, k_rot.s, m.v.s, o, sm_scale, causal, 0);
    launch_fwd(d, q_rot.p, kv, ptr(r.out), fptr(r.lse), PICO_BF16, false, nullptr, 0, nullptr, nullptr, qkv.options());
  }
  return r;
}

struct QKVAttention : torch::autograd::Function<QKVAttention> {
  static Tensor forward(AutogradContext* ctx, const Tensor& qkv_in, const Tensor& cos, const Tensor& sin, int64_t Hq, int64_t Hkv,
                        int64_t D, bool causal, double sm_scale, bool in_kernel) {
    const Tensor qkv = qkv_in.contiguous();
    QKVForward r = qkv_forward(qkv, cos, sin, Hq, Hkv, D, causal, sm_scale, in_kernel);
    ctx->save_for_backward({qkv, r.qk, r.out, r.lse, cos, sin});
    ctx->saved_data["heads"] = std::vector<int64_t>{Hq, Hkv, D};
    ctx->saved_data["causal"] = causal;
    ctx->saved_data["scale"] = sm_scale;
    ctx->saved_data["in_kernel"] = in_kernel;
    return r.out;
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& g) {
    const auto s = ctx->get_saved_variables();
    const auto heads = ctx->saved_data["heads"].toIntVector();
    const int64_t Hq = heads[0], Hkv = heads[1], D = heads[2];
    const bool causal = ctx->saved_data["causal"].toBool(), in_kernel = ctx->saved_data["in_kernel"].toBool();
    const double sm_scale = ctx->saved_data["scale"].toDouble();
    const Tensor &qkv = s[0], &qk = s[1], &out = s[2], &lse = s[3], &cos = s[4], &sin = s[5];
    const QKVShape m = qkv_parts(qkv, Hq, Hkv, D);
    const int64_t B = m.n.B, S = m.n.Sq, W = (Hq + Hkv) * D;
    const Tensor dout = g[0].contiguous().to(at::kBFloat16);
    Tensor dqkv = at::empty(qkv.sizes(), qkv.options());
    const Tensor delta = at::empty({B, Hq, S}, lse.options());
    const QKVShape dm = qkv_parts(dqkv, Hq, Hkv, D);
    auto* base = static_cast<char*>(qk.data_ptr());
    const Stride3 rot = {S * W, D, W};
    pico_attn_desc d = attn_desc(m.n, rot, rot, m.v.s, bshd(Hq, S, D), sm_scale, causal, 0);
    pico_kv_chunks kv = one_chunk(m.n, base + 2 * Hq * D, m.v.p, dm.k.p, dm.v.p);
    pico_rope_tables tables;
    if (in_kernel) tables = rope_tables(cos, sin);
    launch_bwd(d, base, kv, ptr(dout), ptr(out), PICO_BF16, fptr(lse), fptr(delta), dm.q.p, dm.q.s.data(), PICO_BF16, false, dm.k.s.data(),
               PICO_BF16, in_kernel ? &tables : nullptr, 0, 0, qkv.options());
    if (!in_kernel) rope_heads(dm.q, dm.q, cos, sin, B, Hq + Hkv, S, D, true);
    return {dqkv, Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

Tensor qkv_attention(const Tensor& qkv, const Tensor& cos, const Tensor& sin, int64_t Hq, int64_t Hkv, int64_t D, bool causal,
                     bool in_kernel) {
  on_gpu(qkv);
  TORCH_CHECK(qkv.scalar_type() == at::kBFloat16, "attention: q must be bf16 (got ", qkv.scalar_type(), "); the MFMA kernels are bf16 only");
  TORCH_CHECK(qkv.dim() == 3, "attention: the fused projection must be [B, S, columns]");
  const double sm_scale = 1.0 / std::sqrt(static_cast<double>(D));
  if (!records({&qkv})) return qkv_forward(qkv.contiguous(), cos, sin, Hq, Hkv, D, causal, sm_scale, in_kernel).out;
  return QKVAttention::apply(qkv, cos, sin, Hq, Hkv, D, causal, sm_scale, in_kernel);
}

// ------------------------------------------------------------------------------------------------ cross-entropy
void check_loss(const Tensor& logits, const Tensor& targets) {
  on_gpu(logits);
  on_gpu(targets);
  TORCH_CHECK(logits.dim() == 2 && logits.stride(1) == 1, "cross_entropy: logits must be [rows, vocab] with a unit stride on vocab");
  TORCH_CHECK(targets.scalar_type() == at::kLong && targets.is_contiguous() && targets.numel() == logits.size(0),
              "cross_entropy: targets must be a contiguous int64 tensor with one entry per row");
}
int64_t pitch_of(const Tensor& logits) { return logits.size(0) ? logits.stride(0) : logits.size(1); }

std::pair<Tensor, Tensor> cross_entropy_fwd(const Tensor& logits, const Tensor& targets, int64_t ignore_index) {
  check_loss(logits, targets);
  const int64_t rows = logits.size(0), vocab = logits.size(1);
  Tensor loss = at::empty({rows}, logits.options().dtype(at::kFloat)), lse = at::empty({rows}, loss.options());
  check(pico_cross_entropy_fwd(ptr(logits), targets.data_ptr<int64_t>(), fptr(loss), fptr(lse), rows, vocab, pitch_of(logits), ignore_index,
                               dtype_code(logits, "logits"), stream_now()));
  return {loss, lse};
}

Tensor cross_entropy_bwd(const Tensor& logits, const Tensor& targets, const Tensor& lse, const Tensor& scale, int64_t ignore_index,
                         bool inplace) {
  check_loss(logits, targets);
  on_gpu(lse);
  on_gpu(scale);
  TORCH_CHECK(scale.scalar_type() == at::kFloat && scale.numel() == 1 && lse.scalar_type() == at::kFloat && lse.is_contiguous(),
              "cross_entropy_bwd: lse must be contiguous fp32 [rows], scale one fp32 element");
  // same row pitch as the logits (a view into a padded buffer keeps its 16-byte-aligned rows)
  const Tensor out = inplace ? logits : at::empty_strided(logits.sizes(), logits.strides(), logits.options());
  check(pico_cross_entropy_bwd(ptr(logits), targets.data_ptr<int64_t>(), fptr(lse), fptr(scale), ptr(out), logits.size(0), logits.size(1),
                               pitch_of(logits), pitch_of(out), ignore_index, dtype_code(logits, "logits"), stream_now()));
  return out;
}

// Mean cross-entropy of [rows, vocab] logits against int64 targets (train.py:46-49), fp32 loss.  Where a gradient will be
// wanted and the row fits (pico_cross_entropy_one_pass) the forward writes the gradient for a unit upstream gradient while
// it holds the row: forward and backward then read the logits once.  The backward hands that buffer over; the kernel it
// launches looks at the upstream gradient on the device and recomputes only if it is not 1.  `scale` is a factor of the loss
// that the caller knows beforehand (1 / accumulation steps): part of the loss and of the gradient written in the forward.
struct CrossEntropy : torch::autograd::Function<CrossEntropy> {
  static Tensor forward(AutogradContext* ctx, const Tensor& logits, const Tensor& targets, int64_t ignore_index, double scale) {
    Tensor unit;
    const auto [mean, lse, inv_count] = run(logits, targets, ignore_index, scale, &unit);
    ctx->save_for_backward({logits, targets, lse, inv_count, unit});
    ctx->saved_data["ignore"] = ignore_index;
    ctx->saved_data["spent"] = false;
    return mean;
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& g) {
    const auto s = ctx->get_saved_variables();
    const Tensor &logits = s[0], &targets = s[1], &lse = s[2], &inv_count = s[3];
    const Tensor up = g[0].to(at::kFloat).contiguous();
    // a second backward through this node (retain_graph) gets a buffer of its own
    const bool have_unit = s[4].defined() && !ctx->saved_data["spent"].toBool();
    Tensor d = have_unit ? s[4] : empty_like_rows(logits);
    ctx->saved_data["spent"] = true;
    check(pico_cross_entropy_mean_bwd(ptr(logits), targets.data_ptr<int64_t>(), fptr(lse), fptr(inv_count), fptr(up), ptr(d), have_unit,
                                      logits.size(0), logits.size(1), pitch_of(logits), pitch_of(d), ctx->saved_data["ignore"].toInt(),
                                      dtype_code(logits, "logits"), stream_now()));
    return {d, Tensor(), Tensor(), Tensor()};
  }
  // same row pitch as the logits (a view into a padded buffer keeps its 16-byte-aligned rows)
  static Tensor empty_like_rows(const Tensor& logits) { return at::empty_strided(logits.sizes(), logits.strides(), logits.options()); }
  static std::tuple<Tensor, Tensor, Tensor> run(const Tensor& logits, const Tensor& targets, int64_t ignore_index, double scale, Tensor* unit) {
    check_loss(logits, targets);
    const int64_t rows = logits.size(0), vocab = logits.size(1);
    const int dt = dtype_code(logits, "logits");
    const auto f32 = logits.options().dtype(at::kFloat);
    const Tensor loss = at::empty({rows}, f32), lse = at::empty({rows}, f32), mean = at::empty({}, f32), inv_count = at::empty({}, f32);
    if (unit && rows > 0 && pico_cross_entropy_one_pass(vocab, dt)) *unit = empty_like_rows(logits);
    check(pico_cross_entropy_scaled_mean_fwd(ptr(logits), targets.data_ptr<int64_t>(), fptr(loss), fptr(lse), fptr(mean), fptr(inv_count),
                                             unit ? ptr(*unit) : nullptr, static_cast<float>(scale), rows, vocab, pitch_of(logits),
                                             unit && unit->defined() ? pitch_of(*unit) : 0, ignore_index, dt, stream_now()));
    return {mean, lse, inv_count};
  }
};

Tensor cross_entropy(const Tensor& logits, const Tensor& targets, int64_t ignore_index, double scale) {
  if (!records({&logits})) return std::get<0>(CrossEntropy::run(logits, targets, ignore_index, scale, nullptr));
  return CrossEntropy::apply(logits, targets, ignore_index, scale);
}

// ------------------------------------------------------------------------------------------------ AdamW
// The step for a fixed list of tensors in as few launches as they fit.  Weights, moments and sizes are checked and their
// pointer tables built once; a step only fills in the gradients' addresses.
struct AdamWPlan {
  std::vector<Tensor> keep;
  std::vector<void*> w, m, v, lp;
  std::vector<int64_t> sizes;
  int weight_dt = 0, state_dt = 0;
  bool with_lp = false;

  AdamWPlan(const std::vector<Tensor>& weights, const std::vector<Tensor>& exp_avgs, const std::vector<Tensor>& exp_avg_sqs,
            const std::optional<OptTensors>& param_lps) {
    const size_t n = weights.size();
    TORCH_CHECK(n > 0 && exp_avgs.size() == n && exp_avg_sqs.size() == n && (!param_lps || param_lps->size() == n),
                "adamw_multi_: the lists must have one entry per tensor (and at least one)");
    const auto wt = weights[0].scalar_type(), st = exp_avgs[0].scalar_type();
    for (size_t i = 0; i < n; ++i) {
      const int64_t numel = weights[i].numel();
      auto use = [&](const Tensor& t, at::ScalarType dt, const char* what) {
        on_gpu(t);
        TORCH_CHECK(t.scalar_type() == dt && t.is_contiguous() && t.numel() == numel, "adamw_multi_: tensor ", i, ": ", what,
                    " must be a contiguous ", dt, " tensor of ", numel, " elements");
        keep.push_back(t);
        return ptr(t);
      };
      w.push_back(use(weights[i], wt, "weight"));
      m.push_back(use(exp_avgs[i], st, "exp_avg"));
      v.push_back(use(exp_avg_sqs[i], st, "exp_avg_sq"));
      if (param_lps) lp.push_back((*param_lps)[i] ? use(*(*param_lps)[i], at::kBFloat16, "param_lp") : nullptr);
      sizes.push_back(numel);
    }
    with_lp = param_lps.has_value();
    weight_dt = dtype_code(weights[0], "weight");
    state_dt = dtype_code(exp_avgs[0], "exp_avg");
  }

  void step(const std::vector<Tensor>& grads, int64_t step, double lr, double b1, double b2, double eps, double wd, double grad_scale) const {
    TORCH_CHECK(grads.size() == w.size(), "adamw_multi_: the lists must have one entry per tensor");
    const auto gt = grads[0].scalar_type();
    std::vector<Tensor> copies;   // contiguous copies of gradients must outlive the launch call
    std::vector<const void*> g(grads.size());
    for (size_t i = 0; i < grads.size(); ++i) {
      const Tensor& t = grads[i];
      on_gpu(t);
      TORCH_CHECK(t.scalar_type() == gt && t.numel() == sizes[i], "adamw_multi_: tensor ", i, ": grad must have dtype ", gt, " and ",
                  sizes[i], " elements");
      if (!t.is_contiguous()) copies.push_back(t.contiguous());
      g[i] = t.is_contiguous() ? ptr(t) : ptr(copies.back());
    }
    check(pico_adamw_multi(static_cast<int>(w.size()), w.data(), with_lp ? lp.data() : nullptr, g.data(), m.data(), v.data(), sizes.data(),
                           weight_dt, state_dt, dtype_code(grads[0], "grad"), static_cast<float>(lr), static_cast<float>(b1),
                           static_cast<float>(b2), static_cast<float>(eps), static_cast<float>(wd), step, static_cast<float>(grad_scale),
                           stream_now()));
  }

  // The step with every parameter's own .grad.  Returns false, with nothing done, where that is not this plan's case: a
  // gradient is missing, the gradients' dtypes differ, or a parameter was moved since the plan was built.
  bool step_params(const std::vector<Tensor>& params, int64_t step_no, double lr, double b1, double b2, double eps, double wd,
                   double grad_scale) const {
    if (params.size() != w.size()) return false;
    std::vector<Tensor> grads;
    grads.reserve(params.size());
    for (size_t i = 0; i < params.size(); ++i) {
      const Tensor& g = params[i].grad();
      if (!g.defined() || (i && g.scalar_type() != grads[0].scalar_type()) || ptr(params[i]) != (with_lp ? lp[i] : w[i])) return false;
      grads.push_back(g);
    }
    step(grads, step_no, lr, b1, b2, eps, wd, grad_scale);
    return true;
  }
};

void zero_grads(const std::vector<Tensor>& params) {
  for (const Tensor& p : params) p.mutable_grad().reset();
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  namespace py = pybind11;
  using nogil = py::call_guard<py::gil_scoped_release>;
  py::register_local_exception_translator([](std::exception_ptr p) {
    try {
      if (p) std::rethrow_exception(p);
    } catch (const c10::Error& e) {
      PyErr_SetString(PyExc_RuntimeError, e.what_without_backtrace());
    }
  });
  m.doc() = "Native host path of picotron_amd: tensor-level wrappers over the C ABI and the autograd nodes of the model's ops.";
  m.def("rmsnorm_fwd", [](const Tensor& x, const Tensor& w, double eps, bool cast, const OptTensor& res, bool want_sum, bool want_rstd) {
    NormOut o = rmsnorm_forward(x, w, eps, cast, res, want_sum, want_rstd);
    auto opt = [](const Tensor& t) { return t.defined() ? OptTensor(t) : std::nullopt; };
    return std::make_tuple(o.y, opt(o.rstd), opt(o.sum));
  }, nogil());
  m.def("rmsnorm_bwd", [](const Tensor& dy, const Tensor& x, const Tensor& w, const Tensor& rstd, const OptTensor& dres, at::ScalarType dt) {
    return rmsnorm_backward(dy, x, w, rstd, dres, dt);
  }, nogil());
  m.def("rms_norm", &rms_norm, nogil());
  m.def("rms_norm_residual", &rms_norm_residual, nogil());
  m.def("rms_norm_head", &rms_norm_head, nogil());
  m.def("rope", &rope, nogil());
  m.def("rotary", &rotary, nogil());
  m.def("swiglu_fwd", &swiglu_forward, nogil());
  m.def("swiglu_bwd", &swiglu_backward, nogil());
  m.def("swiglu", &swiglu, nogil());
  m.def("swiglu_fused", &swiglu_fused, nogil());
  m.def("chunks_fit", &chunks_fit, nogil());
  m.def("attn_fwd", &attn_fwd, nogil());
  m.def("attn_bwd", &attn_bwd, nogil());
  py::class_<GradBox, GradBoxPtr>(m, "GradBox", "fp32 dK / dV sums of one published chunk; see csrc/host.cpp")
      .def(py::init([] { return c10::make_intrusive<GradBox>(); }))
      .def_readonly("dk", &GradBox::dk)
      .def_readonly("dv", &GradBox::dv)
      .def_readwrite("readers", &GradBox::readers)
      .def_readonly("arrived", &GradBox::arrived)
      .def("claim", &GradBox::claim, py::arg("k"), py::arg("v"), py::arg("whole"), py::arg("rounds"))
      .def("take", &GradBox::take);
  py::class_<GradBox::Share>(m, "GradShare")
      .def_readonly("dk", &GradBox::Share::dk)
      .def_readonly("dv", &GradBox::Share::dv)
      .def_readonly("add", &GradBox::Share::add)
      .def_readonly("final_dk", &GradBox::Share::final_dk)
      .def_readonly("final_dv", &GradBox::Share::final_dv);
  m.def("publish_kv", &publish_kv, nogil());
  m.def("ring_node", &ring_node, nogil());
  m.def("flash_attention", &flash_attention, nogil());
  const auto product_kind = [](const std::string& kind) {
    TORCH_CHECK(kind == "NT" || kind == "NN" || kind == "TN", "product: kind must be NT, NN or TN");
    return kind == "NT" ? Product::NT : kind == "NN" ? Product::NN : Product::TN;
  };
  m.def("product_route", [=](const Tensor& a, const Tensor& b, const std::string& kind) {
    const Product k = product_kind(kind);
    return stays_with_torch(a, b) ? std::string("torch") : route_name(product_route(k, product_sizes(a, b, k)));
  }, pybind11::arg("a"), pybind11::arg("b"), pybind11::arg("kind"));
  m.def("gradient_route", [](const Tensor& dy, const Tensor& w, const Tensor& x) {
    return route_name(gradient_tiles(dy, w, x));
  }, pybind11::arg("dy"), pybind11::arg("w"), pybind11::arg("x"));
  // by the rules; tile_n > 0: in pico_product_large; groups > 0: in pico_product; anything else given: in the library, parts 0 and
  // turn -1 by the rules
  m.def("product", [=](const Tensor& a, const Tensor& b, const std::string& kind, int64_t parts, int64_t turn, int64_t groups, int64_t tile, int64_t tile_n) {
    const Product k = product_kind(kind);
    if (stays_with_torch(a, b) || (parts == 0 && turn < 0 && groups < 0 && tile_n == 0)) return product(a, b, k);
    const ProductSizes n = product_sizes(a, b, k);
    if (tile_n > 0) return product(a, b, k, n, {ProductRoute::Large, tile, tile_n, 0, std::max<int64_t>(parts, 1), 0});
    if (groups > 0) return product(a, b, k, n, {ProductRoute::Own, tile, tile, groups, 1, 0});
    return product(a, b, k, n, {ProductRoute::Library, 0, 0, 0, parts == 0 ? contraction_parts(k, n.M, n.N, n.K) : parts, turn < 0 ? turned_operand(k, n) : turn});
  }, pybind11::arg("a"), pybind11::arg("b"), pybind11::arg("kind"), pybind11::arg("parts") = 0, pybind11::arg("turn") = -1,
        pybind11::arg("groups") = -1, pybind11::arg("tile") = 64, pybind11::arg("tile_n") = 0);
  m.def("mid_product", [=](const Tensor& a, const Tensor& b, const std::string& kind, int64_t tile_m, int64_t tile_n, int64_t parts) {
    TORCH_CHECK(!stays_with_torch(a, b), "mid_product: operands that stay with torch");
    const Product k = product_kind(kind);
    return std::make_tuple(product(a, b, k, product_sizes(a, b, k), {ProductRoute::Mid, tile_m, tile_n, 0, parts, 0}), tile_m, tile_n);
  }, pybind11::arg("a"), pybind11::arg("b"), pybind11::arg("kind"), pybind11::arg("tile_m"), pybind11::arg("tile_n"), pybind11::arg("parts") = 1);
  // (dx, dw, the tiles of each or 0); tiles given: in one launch of these
  m.def("gradients", [](const Tensor& dy, const Tensor& w, const Tensor& x, std::vector<int64_t> tiles) {
    TORCH_CHECK(tiles.empty() || (tiles.size() == 4 && !stays_with_torch(dy, w) && !stays_with_torch(dy, x)),
                "gradients: four tile sides, operands that do not stay with torch");
    const GradientTiles t = tiles.empty() ? gradient_tiles(dy, w, x) : GradientTiles{{tiles[0], tiles[1], 1}, {tiles[2], tiles[3], 1}};
    Gradients d = gradients(dy, w, x, t);
    return std::make_tuple(d.dx, d.dw, t.dx.tile_m, t.dx.tile_n, t.dw.tile_m, t.dw.tile_n);
  }, pybind11::arg("dy"), pybind11::arg("w"), pybind11::arg("x"), pybind11::arg("tiles") = std::vector<int64_t>());
  m.def("linear", &linear, nogil());
  m.def("fused_linear", &fused_linear, nogil());
  m.def("embedding", &embedding, nogil());
  m.def("qkv_attention", &qkv_attention, nogil());
  m.def("cross_entropy", &cross_entropy, pybind11::arg("logits"), pybind11::arg("targets"), pybind11::arg("ignore_index"),
        pybind11::arg("scale") = 1.0, nogil());
  m.def("cross_entropy_fwd", &cross_entropy_fwd, nogil());
  m.def("cross_entropy_bwd", &cross_entropy_bwd, nogil());
  m.def("zero_grads", &zero_grads);
  py::class_<AdamWPlan>(m, "AdamWPlan")
      .def(py::init<const std::vector<Tensor>&, const std::vector<Tensor>&, const std::vector<Tensor>&, const std::optional<OptTensors>&>())
      .def("step", &AdamWPlan::step)
      .def("step_params", &AdamWPlan::step_params);
}
