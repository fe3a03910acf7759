// AdamW steps as one streaming pass per parameter tensor; nothing is read twice.
//   pico_adamw     fp32 master weights and moments for low-precision parameters: reads the gradient, the master
//                  weight and both moments, writes the three fp32 states plus the bf16 copy of the parameter that the
//                  model computes with.  28 bytes per parameter with a bf16 gradient.
//   pico_adamw_lp  the bf16 parameter is updated in place, no master copy; the moments are fp32 (22 bytes per
//                  parameter) or bf16 (what torch.optim.AdamW holds for a bf16 model; 14 bytes).  The arithmetic is
//                  fp32 and every stored value is rounded once.
#include "common.h"

#include <type_traits>

namespace pico {
namespace {

constexpr int kThreads = 256;
// elements of a thread: one access of each array where the step streams past the caches, otherwise two (one where all arrays are bf16)
template <bool kStream>
constexpr int kPerThread = kStream ? 4 : 8;

// What bounds a step is HBM, and what it reaches depends on how its streams meet there (22 bytes per parameter unless said).  Times as shares
// of a kernel that read fp32 arrays as two 16-byte halves of 32 bytes per lane, through the caches, single blocks; lists of a model's
// tensors, every kernel on the same arrays:
//   * Every access of a wave is one run of consecutive bytes, 16 per lane of the widest type; the halves touch every line twice, which streaming
//     accesses pay for (63 M parameters 250 us, streamed 265).  By itself it gives nothing past the caches: 36 lists of 0.3 to 11 GiB 1.03
//     of the time, 28 bytes 1.01, 14 bytes 1.00.
//   * Weights and moments are streamed past the caches, loads and stores, where the arrays are larger than the Infinity Cache: nothing
//     is there when the next step reads it.  Gradients are not: the last of them are still there behind a backward pass (63 M parameters,
//     the same gradients again: 214 us, with streamed gradients 240).  Smaller steps find everything in the cache: arrays of 218 MB
//     58.2 us, streamed 62.9; arrays of 285 MB 124, streamed 106.
//   * A thread of a streamed step has one access of each array, 4 elements.  With two (one of 8 where all arrays are bf16), how far apart the
//     compiler laid loads, arithmetic and stores moved the time by up to 8 % either way (28 bytes: all eight loads first 1.07 of the time that the
//     loads around the first wait took).  30 lists of 0.1 to 1.6 G parameters: 0.892 of the time with one, 0.902 with two; 28 bytes 0.910, 0.921;
//     14 bytes 0.836, 0.938.  Steps in the cache keep two: 30 lists of 0.5 to 23 M parameters took 1.001 to 1.008 of the time with one, up to 1.09.
//   * The XCDs take runs of neighbouring blocks instead of every eighth (block_of_workgroup), of 32 K elements.  It hangs on where the arrays lie,
//     and what sets this length apart is not known: 24 lists with runs of 32 blocks 0.966 of the time of two accesses and runs of 16, 64 blocks
//     0.974, single ones 0.961; 28 bytes 0.990, 1.000, 0.999; 14 bytes 0.897, 0.893, 0.911.  In the cache 60 lists with two accesses took 0.977 of
//     the time of single blocks.  Where all arrays are bf16 and in the cache there is nothing in runs.
//   Before all of it and now, on one card, us: 667 M parameters 2694 -> 2478 (5.9 TB/s), fp32 weights (28 bytes) 3502 -> 3249, bf16 moments (14
//   bytes) 1702 -> 1491 (6.3 TB/s); 64 M, the same gradients again, 263 -> 210, 342 -> 279, 174 -> 135.  (512 threads are 2 to 3 % behind.)
constexpr int64_t kCacheBytes = int64_t(256) << 20;

// N consecutive elements (8 or 16 bytes) as floats
template <bool kStream, int N, typename T>
__device__ __forceinline__ void load_piece(const T* p, float* out, int at) {
  if constexpr (sizeof(T) == 4) {
    static_assert(N == 4);
    const f32x4* from = reinterpret_cast<const f32x4*>(p);
    const f32x4 raw = kStream ? __builtin_nontemporal_load(from) : *from;
#pragma unroll
    for (int i = 0; i < 4; ++i) out[at + i] = raw[i];
  } else {
    using Raw = std::conditional_t<N == 8, u32x4, u32x2>;
    const Raw* from = reinterpret_cast<const Raw*>(p);
    const Raw raw = kStream ? __builtin_nontemporal_load(from) : *from;
#pragma unroll
    for (int i = 0; i < N / 2; ++i) {
      out[at + 2 * i] = __uint_as_float(raw[i] << 16);
      out[at + 2 * i + 1] = __uint_as_float(raw[i] & 0xffff0000u);
    }
  }
}
template <bool kStream, int N, typename T>
__device__ __forceinline__ void store_piece(T* p, const float* in, int at) {
  auto put = [&](auto raw) {
    if constexpr (kStream) {
      // (as it is: otherwise the compiler rebuilds the 16 bytes of eight bf16 values into a vector of its own and stores that without the hint)
      asm("" : "+v"(raw));
      __builtin_nontemporal_store(raw, reinterpret_cast<decltype(raw)*>(p));
    } else {
      *reinterpret_cast<decltype(raw)*>(p) = raw;
    }
  };
  if constexpr (sizeof(T) == 4) {
    static_assert(N == 4);
    f32x4 raw;
#pragma unroll
    for (int i = 0; i < 4; ++i) raw[i] = in[at + i];
    put(raw);
  } else {
    std::conditional_t<N == 8, u32x4, u32x2> raw;
#pragma unroll
    for (int i = 0; i < N / 2; ++i) raw[i] = pack_bf16x2(in[at + 2 * i], in[at + 2 * i + 1]);
    put(raw);
  }
}

// The arithmetic follows torch.optim.AdamW's (non-amsgrad) order of operations so that fp32 states match it to
// rounding: p *= 1 - lr*wd;  m = m + (g - m)*(1 - b1);  v = v*b2 + g*g*(1 - b2);
// p -= step_size * m / (sqrt(v) / sqrt(bc2) + eps),  step_size = lr / bc1.
// TW is the type of the weight that is updated, TM that of both moments; param_lp, when given, receives a bf16 copy
// of the updated weight.
struct Hyper {
  float decay, one_minus_b1, b2, one_minus_b2, step_size, inv_sqrt_bc2, eps, grad_scale;
};

// elements of one access: 16 bytes of the widest type, at most a thread's
template <bool kStream, typename TW, typename TM, typename TG>
constexpr int kPiece = !kStream && sizeof(TW) == 2 && sizeof(TM) == 2 && sizeof(TG) == 2 ? 8 : 4;

// The block of a workgroup: neighbouring workgroups run on different XCDs (they go round all eight), and each XCD takes kRun blocks in
// a row.  What does not fill a round of runs is dealt block by block.
template <bool kStream, int N>
__device__ __forceinline__ unsigned block_of_workgroup(unsigned workgroup, unsigned count) {
  constexpr unsigned kRun = kStream ? 32 : N == 8 ? 1 : 16, kXcds = 8, kRound = kXcds * kRun;
  if constexpr (kRun == 1) return workgroup;
  const unsigned round = workgroup / kRound, in = workgroup % kRound;
  return (round + 1) * kRound <= count ? round * kRound + in % kXcds * kRun + in / kXcds : workgroup;
}

template <bool kStream, typename TW, typename TM, typename TG>
__device__ __forceinline__ void adamw_block(__bf16* __restrict__ param_lp, TW* __restrict__ master,
                                            const TG* __restrict__ grad, TM* __restrict__ exp_avg,
                                            TM* __restrict__ exp_avg_sq, int64_t n, int64_t block, const Hyper& h) {
  constexpr int N = kPiece<kStream, TW, TM, TG>, kMine = kPerThread<kStream>, kPieces = kMine / N;
  const int64_t i0 = block * (kThreads * kMine) + threadIdx.x * N;
  if (i0 >= n) return;
  auto at = [&](int j) { return i0 + j * (kThreads * N); };
  float g[kMine], p[kMine], m[kMine], v[kMine];
  auto load = [&](int j) {
    load_piece<false, N>(grad + at(j), g, j * N);
    load_piece<kStream, N>(master + at(j), p, j * N);
    load_piece<kStream, N>(exp_avg + at(j), m, j * N);
    load_piece<kStream, N>(exp_avg_sq + at(j), v, j * N);
  };
  auto store = [&](int j) {
    store_piece<kStream, N>(master + at(j), p, j * N);
    store_piece<kStream, N>(exp_avg + at(j), m, j * N);
    store_piece<kStream, N>(exp_avg_sq + at(j), v, j * N);
    if (param_lp) store_piece<kStream, N>(param_lp + at(j), p, j * N);
  };
  // (the FMAs are written out: left to the compiler, which of two products it takes into one differs from block to last block)
  auto update = [&]() {
#pragma unroll
    for (int e = 0; e < kMine; ++e) {
      const float ge = g[e] * h.grad_scale;
      m[e] = __builtin_fmaf(__builtin_fmaf(g[e], h.grad_scale, -m[e]), h.one_minus_b1, m[e]);
      v[e] = __builtin_fmaf(v[e], h.b2, ge * ge * h.one_minus_b2);
      const float denom = __builtin_fmaf(__builtin_sqrtf(v[e]), h.inv_sqrt_bc2, h.eps);
      p[e] = __builtin_fmaf(p[e], h.decay, -(h.step_size * (m[e] / denom)));
    }
  };
  if ((block + 1) * (kThreads * kMine) <= n) {
#pragma unroll
    for (int j = 0; j < kPieces; ++j) load(j);
    update();
#pragma unroll
    for (int j = 0; j < kPieces; ++j) store(j);
    return;
  }
  // A tensor's last block has code of its own, in which every access is judged by itself and only the one that the tensor ends in goes
  // element by element.  Where all accesses of a thread had to be there for any to be whole (a thread's two lie 1024 elements apart), 48 tensors of 576
  // elements took 4.5 us and take 3.8, 80 drawn lists of 0.2 to 13 M parameters 0.89 of the time, 28 bytes 0.92, 14 bytes 0.95.
#pragma unroll
  for (int j = 0; j < kPieces; ++j) {
    if (at(j) + N <= n) {
      load(j);
      continue;
    }
#pragma unroll
    for (int e = j * N; e < (j + 1) * N; ++e) {
      const int64_t i = at(j) + e % N;
      const bool in = i < n;
      g[e] = in ? static_cast<float>(grad[i]) : 0.f;
      p[e] = in ? static_cast<float>(master[i]) : 0.f;
      m[e] = in ? static_cast<float>(exp_avg[i]) : 0.f;
      v[e] = in ? static_cast<float>(exp_avg_sq[i]) : 0.f;
    }
  }
  update();
#pragma unroll
  for (int j = 0; j < kPieces; ++j) {
    if (at(j) + N <= n) {
      store(j);
      continue;
    }
#pragma unroll
    for (int e = j * N; e < (j + 1) * N; ++e) {
      const int64_t i = at(j) + e % N;
      if (i >= n) continue;
      master[i] = static_cast<TW>(p[e]);
      exp_avg[i] = static_cast<TM>(m[e]);
      exp_avg_sq[i] = static_cast<TM>(v[e]);
      if (param_lp) param_lp[i] = static_cast<__bf16>(p[e]);
    }
  }
}

template <bool kStream, typename TW, typename TM, typename TG>
__global__ __launch_bounds__(kThreads) void adamw_kernel(__bf16* __restrict__ param_lp, TW* __restrict__ master,
                                                         const TG* __restrict__ grad, TM* __restrict__ exp_avg,
                                                         TM* __restrict__ exp_avg_sq, int64_t n, Hyper h) {
  adamw_block<kStream, TW, TM, TG>(param_lp, master, grad, exp_avg, exp_avg_sq, n, block_of_workgroup<kStream, kPiece<kStream, TW, TM, TG>>(blockIdx.x, gridDim.x), h);
}

// Many tensors in one launch: the pointers travel in the kernel arguments (no table in device memory to keep alive),
// and a workgroup finds its tensor by bisecting the running block count, which is uniform scalar work.
constexpr int kMaxTensors = 48;
struct TensorTable {
  void* weight[kMaxTensors];
  void* param_lp[kMaxTensors];
  const void* grad[kMaxTensors];
  void* exp_avg[kMaxTensors];
  void* exp_avg_sq[kMaxTensors];
  int64_t n[kMaxTensors];
  unsigned block_start[kMaxTensors + 1];
  int count;
};

template <bool kStream, typename TW, typename TM, typename TG>
__global__ __launch_bounds__(kThreads) void adamw_multi_kernel(TensorTable t, Hyper h) {
  const unsigned bid = block_of_workgroup<kStream, kPiece<kStream, TW, TM, TG>>(blockIdx.x, gridDim.x);
  int lo = 0, hi = t.count;   // block_start[lo] <= bid < block_start[hi]
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (bid >= t.block_start[mid]) lo = mid; else hi = mid;
  }
  adamw_block<kStream, TW, TM, TG>(static_cast<__bf16*>(t.param_lp[lo]), static_cast<TW*>(t.weight[lo]),
                          static_cast<const TG*>(t.grad[lo]), static_cast<TM*>(t.exp_avg[lo]),
                          static_cast<TM*>(t.exp_avg_sq[lo]), t.n[lo], bid - t.block_start[lo], h);
}

}  // namespace
}  // namespace pico

using namespace pico;

namespace {

int hyper_check(const char* who, int grad_dtype, int64_t step) {
  if (grad_dtype != PICO_BF16 && grad_dtype != PICO_F32)
    return fail(PICO_ERR_DTYPE, "%s: gradient dtype code %d not supported", who, grad_dtype);
  if (step < 1) return fail(PICO_ERR_SHAPE, "%s: step=%lld must be >= 1", who, static_cast<long long>(step));
  return PICO_OK;
}

Hyper make_hyper(float lr, float beta1, float beta2, float eps, float weight_decay, int64_t step, float grad_scale) {
  // bias corrections in double, as torch computes them on the host
  const double bc1 = 1.0 - __builtin_pow(static_cast<double>(beta1), static_cast<double>(step));
  const double bc2 = 1.0 - __builtin_pow(static_cast<double>(beta2), static_cast<double>(step));
  Hyper h;
  h.decay = 1.f - lr * weight_decay;
  h.one_minus_b1 = 1.f - beta1;
  h.b2 = beta2;
  h.one_minus_b2 = 1.f - beta2;
  h.step_size = static_cast<float>(static_cast<double>(lr) / bc1);
  h.inv_sqrt_bc2 = static_cast<float>(1.0 / __builtin_sqrt(bc2));
  h.eps = eps;
  h.grad_scale = grad_scale;
  return h;
}

int64_t blocks_of(int64_t n, bool stream) {
  const int64_t per_block = kThreads * (stream ? kPerThread<true> : kPerThread<false>);
  return (n + per_block - 1) / per_block;
}
// A launch has less than 2^32 threads; tensors of more than this many elements (a whole number of blocks) go in slices.
constexpr int64_t kMostBlocks = 0xffffffff / kThreads, kSlice = int64_t(1) << 31;

template <typename TW, typename TM>
int64_t state_bytes(int grad_dtype, bool copy) {   // per parameter, each array once
  return static_cast<int64_t>(sizeof(TW) + 2 * sizeof(TM)) + (grad_dtype == PICO_BF16 ? 2 : 4) + (copy ? 2 : 0);
}
bool streams(int64_t bytes) { return bytes > kCacheBytes; }
template <typename Fn>
void with_kernel_types(int grad_dtype, bool stream, const Fn& fn) {
  auto by_grad = [&](auto stream_it) {
    if (grad_dtype == PICO_BF16) fn(stream_it, __bf16());
    else fn(stream_it, float());
  };
  if (stream) by_grad(std::true_type());
  else by_grad(std::false_type());
}

template <typename TW, typename TM>
int adamw_launch(const char* who, void* param_lp, TW* master, const void* grad, int grad_dtype, TM* exp_avg,
                 TM* exp_avg_sq, int64_t n, float lr, float beta1, float beta2, float eps, float weight_decay,
                 int64_t step, float grad_scale, void* stream) {
  if (int rc = hyper_check(who, grad_dtype, step)) return rc;
  if (n < 0) return fail(PICO_ERR_SHAPE, "%s: n=%lld must be >= 0", who, static_cast<long long>(n));
  if (n == 0) return PICO_OK;
  if (!master || !grad || !exp_avg || !exp_avg_sq)
    return fail(PICO_ERR_NULL, "%s: the weight, grad, exp_avg and exp_avg_sq are required", who);
  if (!aligned16(param_lp) || !aligned16(master) || !aligned16(grad) || !aligned16(exp_avg) || !aligned16(exp_avg_sq))
    return fail(PICO_ERR_ALIGN, "%s: pointers must be 16-byte aligned", who);
  const Hyper h = make_hyper(lr, beta1, beta2, eps, weight_decay, step, grad_scale);
  const bool stream_all = streams(n * state_bytes<TW, TM>(grad_dtype, param_lp != nullptr));
  hipStream_t s = static_cast<hipStream_t>(stream);
  for (int64_t at = 0; at < n; at += kSlice) {
    const int64_t count = std::min(n - at, kSlice);
    with_kernel_types(grad_dtype, stream_all, [&](auto stream_it, auto grad_type) {
      using TG = decltype(grad_type);
      hipLaunchKernelGGL((adamw_kernel<decltype(stream_it)::value, TW, TM, TG>), dim3(static_cast<unsigned>(blocks_of(count, stream_all))), dim3(kThreads), 0, s,
                         param_lp ? static_cast<__bf16*>(param_lp) + at : nullptr, master + at, static_cast<const TG*>(grad) + at, exp_avg + at,
                         exp_avg_sq + at, count, h);
    });
    if (int rc = check_launch(who)) return rc;
  }
  return PICO_OK;
}

template <typename TW, typename TM>
int adamw_multi_launch(int count, void* const* weights, void* const* param_lps, const void* const* grads,
                       void* const* exp_avgs, void* const* exp_avg_sqs, const int64_t* sizes, int grad_dtype,
                       const Hyper& h, hipStream_t s) {
  const char* who = "pico_adamw_multi";
  // validate everything before the first launch so that a rejected call has changed nothing
  for (int i = 0; i < count; ++i) {
    if (sizes[i] < 0) return fail(PICO_ERR_SHAPE, "%s: tensor %d has n=%lld", who, i, static_cast<long long>(sizes[i]));
    if (sizes[i] == 0) continue;
    if (!weights[i] || !grads[i] || !exp_avgs[i] || !exp_avg_sqs[i])
      return fail(PICO_ERR_NULL, "%s: tensor %d: the weight, grad, exp_avg and exp_avg_sq are required", who, i);
    if (!aligned16(weights[i]) || !aligned16(grads[i]) || !aligned16(exp_avgs[i]) || !aligned16(exp_avg_sqs[i]) ||
        (param_lps && !aligned16(param_lps[i])))
      return fail(PICO_ERR_ALIGN, "%s: tensor %d: pointers must be 16-byte aligned", who, i);
    if (blocks_of(sizes[i], false) > 0x7fffffff)
      return fail(PICO_ERR_SHAPE, "%s: tensor %d is too large for one launch", who, i);
  }
  int64_t elements = 0;
  for (int i = 0; i < count; ++i) elements += sizes[i];
  const bool stream_all = streams(elements * state_bytes<TW, TM>(grad_dtype, param_lps != nullptr));
  TensorTable t;
  t.count = 0;
  t.block_start[0] = 0;
  auto flush = [&]() -> int {
    if (t.count == 0) return PICO_OK;
    const unsigned grid = t.block_start[t.count];
    with_kernel_types(grad_dtype, stream_all, [&](auto stream_it, auto grad_type) {
      hipLaunchKernelGGL((adamw_multi_kernel<decltype(stream_it)::value, TW, TM, decltype(grad_type)>), dim3(grid), dim3(kThreads), 0, s, t, h);
    });
    t.count = 0;
    return check_launch(who);
  };
  for (int i = 0; i < count; ++i) {
    if (sizes[i] == 0) continue;
    for (int64_t at = 0; at < sizes[i]; at += kSlice) {
      const int64_t n = std::min(sizes[i] - at, kSlice), blocks = blocks_of(n, stream_all);
      if (t.count == kMaxTensors || t.block_start[t.count] + blocks > kMostBlocks)
        if (int rc = flush()) return rc;
      const int j = t.count++;
      t.weight[j] = static_cast<TW*>(weights[i]) + at;
      t.param_lp[j] = param_lps && param_lps[i] ? static_cast<__bf16*>(param_lps[i]) + at : nullptr;
      t.grad[j] = static_cast<const char*>(grads[i]) + at * (grad_dtype == PICO_BF16 ? 2 : 4);
      t.exp_avg[j] = static_cast<TM*>(exp_avgs[i]) + at;
      t.exp_avg_sq[j] = static_cast<TM*>(exp_avg_sqs[i]) + at;
      t.n[j] = n;
      t.block_start[j + 1] = t.block_start[j] + static_cast<unsigned>(blocks);
    }
  }
  return flush();
}

}  // namespace

extern "C" int pico_adamw_multi(int count, void* const* weights, void* const* param_lps, const void* const* grads,
                                void* const* exp_avgs, void* const* exp_avg_sqs, const int64_t* sizes, int weight_dtype,
                                int state_dtype, int grad_dtype, float lr, float beta1, float beta2, float eps,
                                float weight_decay, int64_t step, float grad_scale, void* stream) {
  const char* who = "pico_adamw_multi";
  if (int rc = hyper_check(who, grad_dtype, step)) return rc;
  if (count < 0) return fail(PICO_ERR_SHAPE, "%s: count=%d must be >= 0", who, count);
  if (count == 0) return PICO_OK;
  if (!weights || !grads || !exp_avgs || !exp_avg_sqs || !sizes)
    return fail(PICO_ERR_NULL, "%s: the pointer tables and sizes are required", who);
  const Hyper h = make_hyper(lr, beta1, beta2, eps, weight_decay, step, grad_scale);
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (weight_dtype == PICO_F32 && state_dtype == PICO_F32)
    return adamw_multi_launch<float, float>(count, weights, param_lps, grads, exp_avgs, exp_avg_sqs, sizes, grad_dtype, h, s);
  if (weight_dtype == PICO_BF16 && (state_dtype == PICO_BF16 || state_dtype == PICO_F32)) {
    if (param_lps) return fail(PICO_ERR_NULL, "%s: param_lps must be NULL when the weights are bf16 (they are the parameters)", who);
    if (state_dtype == PICO_BF16)
      return adamw_multi_launch<__bf16, __bf16>(count, weights, nullptr, grads, exp_avgs, exp_avg_sqs, sizes, grad_dtype, h, s);
    return adamw_multi_launch<__bf16, float>(count, weights, nullptr, grads, exp_avgs, exp_avg_sqs, sizes, grad_dtype, h, s);
  }
  return fail(PICO_ERR_DTYPE, "%s: weight dtype code %d with state dtype code %d not supported", who, weight_dtype, state_dtype);
}

extern "C" int pico_adamw(void* param_lp, float* master, const void* grad, int grad_dtype, float* exp_avg,
                          float* exp_avg_sq, int64_t n, float lr, float beta1, float beta2, float eps,
                          float weight_decay, int64_t step, float grad_scale, void* stream) {
  return adamw_launch<float, float>("pico_adamw", param_lp, master, grad, grad_dtype, exp_avg, exp_avg_sq, n, lr, beta1,
                                    beta2, eps, weight_decay, step, grad_scale, stream);
}

extern "C" int pico_adamw_lp(void* param, const void* grad, int grad_dtype, void* exp_avg, void* exp_avg_sq,
                             int64_t n, int param_dtype, int state_dtype, float lr, float beta1, float beta2, float eps,
                             float weight_decay, int64_t step, float grad_scale, void* stream) {
  if (param_dtype != PICO_BF16)
    return fail(PICO_ERR_DTYPE, "pico_adamw_lp: parameter dtype code %d not supported (bf16 only)", param_dtype);
  if (state_dtype == PICO_BF16)
    return adamw_launch<__bf16, __bf16>("pico_adamw_lp", nullptr, static_cast<__bf16*>(param), grad, grad_dtype,
                                        static_cast<__bf16*>(exp_avg), static_cast<__bf16*>(exp_avg_sq), n, lr, beta1,
                                        beta2, eps, weight_decay, step, grad_scale, stream);
  if (state_dtype == PICO_F32)
    return adamw_launch<__bf16, float>("pico_adamw_lp", nullptr, static_cast<__bf16*>(param), grad, grad_dtype,
                                       static_cast<float*>(exp_avg), static_cast<float*>(exp_avg_sq), n, lr, beta1, beta2,
                                       eps, weight_decay, step, grad_scale, stream);
  return fail(PICO_ERR_DTYPE, "pico_adamw_lp: state dtype code %d not supported", state_dtype);
}
