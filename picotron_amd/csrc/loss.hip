// Cross-entropy over the vocabulary: one workgroup per token row.
//   forward : lse = logsumexp(row), loss = lse - row[target]      (one read of the logits)
//   backward: dlogits = (exp(row - lse) - onehot(target)) * scale  (one read, one write)
//   both    : the row stays in registers between the two, so forward and backward together read the logits once
// fp32 arithmetic on bf16 or fp32 logits; rows whose target equals ignore_index -- or lies outside [0, vocab), which
// no load may follow -- contribute nothing: loss 0, gradient row 0.
#include "common.h"

namespace pico {
namespace {

constexpr int kThreads = 512;
constexpr int kWaves = kThreads / kWave;
// The logits of a training step are far larger than the caches, so they are read with streaming loads and dlogits
// leave with streaming stores (forward +13 %, backward +6 % at [4096, 49152]); a thread requests several pieces of its
// row before it uses the first (bytes in flight per thread: forward 2, backward 4 pieces).
constexpr bool kStreamLoads = true, kStreamStores = true;
constexpr int kFwdUnroll = 2, kBwdUnroll = 4;

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
  return v;
}

template <typename T>
__global__ __launch_bounds__(kThreads) void ce_fwd_kernel(const T* __restrict__ logits, const int64_t* __restrict__ targets,
                                                          float* __restrict__ loss, float* __restrict__ lse_out,
                                                          int vocab, int64_t ld, int64_t ignore_index) {
  constexpr int V = io<T>::kVec;
  __shared__ float red_m[kWaves], red_s[kWaves];
  const int64_t row = blockIdx.x;
  const T* x = logits + row * ld;
  const int nvec = vocab / V;
  // online (max, sum of exp) per thread, in the log2 domain
  float m = -INFINITY, s = 0.f;
  auto absorb = [&](const float (&e)[V]) {
    float mx = e[0];
#pragma unroll
    for (int i = 1; i < V; ++i) mx = fmaxf(mx, e[i]);
    mx *= kLog2e;
    if (mx > m) { s *= fast_exp2(m - mx); m = mx; }
#pragma unroll
    for (int i = 0; i < V; ++i) s += fast_exp2(e[i] * kLog2e - m);
  };
  constexpr int U = kFwdUnroll;   // pieces of the row requested together (bytes in flight per thread)
  int v = threadIdx.x;
  for (; v + (U - 1) * kThreads < nvec; v += U * kThreads) {
    float e[U][V];
#pragma unroll
    for (int u = 0; u < U; ++u) load_as<T, kStreamLoads>(x + static_cast<int64_t>(v + u * kThreads) * V, e[u]);
#pragma unroll
    for (int u = 0; u < U; ++u) absorb(e[u]);
  }
  for (; v < nvec; v += kThreads) {
    float e[V];
    load_as<T, kStreamLoads>(x + static_cast<int64_t>(v) * V, e);
    absorb(e);
  }
  for (int j = nvec * V + threadIdx.x; j < vocab; j += kThreads) {  // tail when vocab is not a multiple of V
    const float e = static_cast<float>(x[j]) * kLog2e;
    if (e > m) { s *= fast_exp2(m - e); m = e; }
    s += fast_exp2(e - m);
  }
  const float wm = wave_max(m);
  s = (m == -INFINITY) ? 0.f : s * fast_exp2(m - wm);
  s = wave_sum(s);
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  if (lane == 0) { red_m[wave] = wm; red_s[wave] = s; }
  __syncthreads();
  if (threadIdx.x == 0) {
    float bm = red_m[0];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) bm = fmaxf(bm, red_m[w]);
    float bs = 0.f;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) bs += (red_m[w] == -INFINITY) ? 0.f : red_s[w] * fast_exp2(red_m[w] - bm);
    const float lse = (bm + fast_log2(bs)) * kLn2;
    const int64_t t = targets[row];
    lse_out[row] = lse;
    const bool counts = t != ignore_index && t >= 0 && t < vocab;
    loss[row] = counts ? lse - static_cast<float>(x[t]) : 0.f;
  }
}

template <typename T>
__global__ __launch_bounds__(kThreads) void ce_bwd_kernel(const T* __restrict__ logits, const int64_t* __restrict__ targets,
                                                          const float* __restrict__ lse, const float* __restrict__ scale_ptr,
                                                          const float* __restrict__ grad_out, int skip_unit,
                                                          T* __restrict__ dlogits, int64_t rows, int vocab, int64_t ld, int64_t dld,
                                                          int64_t ignore_index) {
  constexpr int V = io<T>::kVec;
  const float up = grad_out != nullptr ? *grad_out : 1.f;
  if (skip_unit && up == 1.f) return;   // dlogits holds the gradient for a unit upstream gradient already
  for (int64_t row = blockIdx.x; row < rows; row += gridDim.x) {
    const T* x = logits + row * ld;
    T* d = dlogits + row * dld;
    const int64_t t = targets[row];
    const float scale = (t != ignore_index && t >= 0 && t < vocab) ? *scale_ptr * up : 0.f;
    const float l2 = lse[row] * kLog2e;
    const int nvec = vocab / V;
    // kCeUnroll pieces of the row per thread are requested before the first is used: one 16-byte load per thread at a
    // time leaves too few bytes in flight to cover the memory latency
    constexpr int U = kBwdUnroll;
    int v = threadIdx.x;
    for (; v + (U - 1) * kThreads < nvec; v += U * kThreads) {
      float e[U][V];
#pragma unroll
      for (int u = 0; u < U; ++u) load_as<T, kStreamLoads>(x + static_cast<int64_t>(v + u * kThreads) * V, e[u]);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        float o[V];
        const int j0 = (v + u * kThreads) * V;
#pragma unroll
        for (int i = 0; i < V; ++i) {
          const float p = fast_exp2(e[u][i] * kLog2e - l2);
          o[i] = (p - ((j0 + i) == t ? 1.f : 0.f)) * scale;
        }
        store_as<T, kStreamStores>(d + static_cast<int64_t>(v + u * kThreads) * V, o);
      }
    }
    for (; v < nvec; v += kThreads) {
      float e[V], o[V];
      load_as<T, kStreamLoads>(x + static_cast<int64_t>(v) * V, e);
      const int j0 = v * V;
#pragma unroll
      for (int i = 0; i < V; ++i) {
        const float p = fast_exp2(e[i] * kLog2e - l2);
        o[i] = (p - ((j0 + i) == t ? 1.f : 0.f)) * scale;
      }
      store_as<T, kStreamStores>(d + static_cast<int64_t>(v) * V, o);
    }
    for (int j = nvec * V + threadIdx.x; j < vocab; j += kThreads) {
      const float p = fast_exp2(static_cast<float>(x[j]) * kLog2e - l2);
      d[j] = static_cast<T>((p - (j == t ? 1.f : 0.f)) * scale);
    }
  }
}

// ---- forward and backward in one pass over the logits.  Bound by HBM: the row (96 KiB at vocab 49152 in bf16) is read
// once into registers, 16 bytes per lane and piece, reduced, turned into its gradient and written: 2 x rows x vocab
// elements of traffic where forward and backward apart move 3 x.  NT threads hold NV pieces each; with at most 8 pieces
// (32 registers for the row, 64 in all, none in scratch) two 1024-thread workgroups share a CU and one reads while the other
// writes.  Measured, forward
// + backward through autograd, against the two streaming kernels and torch's reductions between them: [4096, 49152] bf16
// 232 -> 146 us (5.5 TB/s), [4096, 49152] fp32 414 -> 301, [16384, 2000] bf16 63 -> 40 (kernels alone).
template <typename T>
__device__ __forceinline__ void unpack_piece(const u32x4& raw, float (&out)[io<T>::kVec]) {
  if constexpr (sizeof(T) == 2) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      out[2 * i] = __uint_as_float(raw[i] << 16);
      out[2 * i + 1] = __uint_as_float(raw[i] & 0xffff0000u);
    }
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) out[i] = __uint_as_float(raw[i]);
  }
}

// Up to kCountMost rows per thread every workgroup counts the rows that count for itself, instead of a launch in front of it
// (forward + backward [512, 49152] bf16 22.9 -> 20.6 us, fp32 41.4 -> 39.0; with four rows per thread [4096, 49152] 143.6 -> 146.5).  Where
// the row leaves no registers for that (28 bytes of scratch), the launch stays.
constexpr int kCountMost = 1;
template <int NT, int NV> constexpr bool kCountsItself = NT < 1024 || NV != 8;
template <typename T, int NT, int NV, bool kGrad>
__global__ __launch_bounds__(NT, NV <= 8 ? 8 : 4) void ce_one_pass_kernel(const T* __restrict__ logits, const int64_t* __restrict__ targets,
                                                         float* __restrict__ loss, float* __restrict__ lse_out,
                                                         const float* __restrict__ inv_count, T* __restrict__ dlogits, int vocab,
                                                         int64_t ld, int64_t dld, int64_t ignore_index, int count_rows, float unit) {
  constexpr int V = io<T>::kVec, W = NT / kWave;
  __shared__ float red_m[W], red_s[W];
  __shared__ int red_n[W];
  const int64_t row = blockIdx.x;
  const T* x = logits + row * ld;
  T* d = kGrad ? dlogits + row * dld : nullptr;
  const int nvec = vocab / V, tail = nvec * V + static_cast<int>(threadIdx.x);   // tail: vocab that is no multiple of V
  const int64_t t = targets[row];
  const bool counts = t != ignore_index && t >= 0 && t < vocab;
  if (kGrad && !counts) {   // nothing of the row is needed
    const u32x4 zero = {0u, 0u, 0u, 0u};
    for (int v = threadIdx.x; v < nvec; v += NT) __builtin_nontemporal_store(zero, reinterpret_cast<u32x4*>(d + static_cast<int64_t>(v) * V));
    if (tail < vocab) d[tail] = static_cast<T>(0.f);
    if (threadIdx.x == 0) { loss[row] = 0.f; lse_out[row] = 0.f; }
    return;
  }
  // lanes past the end of the row hold -inf, whose exponential is 0
  constexpr uint32_t kNegInf = sizeof(T) == 2 ? 0xff80ff80u : 0xff800000u;
  u32x4 raw[NV];
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int v = threadIdx.x + j * NT;
    raw[j] = u32x4{kNegInf, kNegInf, kNegInf, kNegInf};
    if (v < nvec) raw[j] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(x + static_cast<int64_t>(v) * V));
  }
  // the row stays packed: each phase unpacks it again (the empty asm hides that it is the same value, or the compiler would
  // keep the unpacked row, two to four times the registers, from phase to phase)
  auto hide = [&]() {
#pragma unroll
    for (int j = 0; j < NV; ++j) asm volatile("" : "+v"(raw[j]));
  };
  // the rows that count, by every workgroup for itself where they are few (count_rows > 0), behind the requests for its row
  if constexpr (kGrad && kCountsItself<NT, NV>) {
    if (count_rows > 0) {
      int n = 0;
#pragma unroll
      for (int u = 0; u < kCountMost; ++u) {
        const int r = threadIdx.x + u * NT;
        const int64_t tr = r < count_rows ? targets[r] : ignore_index;
        n += __popcll(__ballot(tr != ignore_index && tr >= 0 && tr < vocab));
      }
      if (threadIdx.x % kWave == 0) red_n[threadIdx.x / kWave] = n;
    }
  }
  const float given = kGrad && (!kCountsItself<NT, NV> || count_rows == 0) ? *inv_count : 0.f, xt = counts ? static_cast<float>(x[t]) : 0.f, xe = tail < vocab ? static_cast<float>(x[tail]) : -INFINITY;
  float m = xe;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    float e[V];
    unpack_piece<T>(raw[j], e);
#pragma unroll
    for (int i = 0; i < V; ++i) m = fmaxf(m, e[i]);
  }
  hide();
  m *= kLog2e;   // (log2 domain)
  float s = tail < vocab ? fast_exp2(xe * kLog2e - m) : 0.f;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    float e[V];
    unpack_piece<T>(raw[j], e);
#pragma unroll
    for (int i = 0; i < V; ++i) s += fast_exp2(e[i] * kLog2e - m);
    __builtin_amdgcn_sched_barrier(0);
  }
  hide();
  const float wm = wave_max(m);
  s = wave_sum(m == -INFINITY ? 0.f : s * fast_exp2(m - wm));
  const int wave = threadIdx.x / kWave;
  if (threadIdx.x % kWave == 0) { red_m[wave] = wm; red_s[wave] = s; }
  __syncthreads();
  // Rows of eight pieces and more in eight waves and more: one wave's share per lane, reduced by exchanges.  Read whole by every
  // lane the shares take 2 W registers beside the row, and those rows went to scratch ([4096, 32000] bf16 forward + backward
  // 110 -> 103 us, [2048, 65536] 114 -> 105, [8192, 20000] 139 -> 132, fp32 the same).  Elsewhere there is room, and reading
  // them is 2 to 3 % faster (kernel alone, 4096 rows of 2040 pieces 54.4 us, by exchanges 56.1).
  float bm, bs;
  if constexpr (NV >= 8 && W >= 8) {
    const float pm = red_m[threadIdx.x % W];
    bm = pm;
#pragma unroll
    for (int off = W / 2; off > 0; off >>= 1) bm = fmaxf(bm, __shfl_xor(bm, off, kWave));
    bs = pm == -INFINITY ? 0.f : red_s[threadIdx.x % W] * fast_exp2(pm - bm);
#pragma unroll
    for (int off = W / 2; off > 0; off >>= 1) bs += __shfl_xor(bs, off, kWave);
  } else {
    bm = red_m[0];
    bs = 0.f;
#pragma unroll
    for (int w = 1; w < W; ++w) bm = fmaxf(bm, red_m[w]);
#pragma unroll
    for (int w = 0; w < W; ++w) bs += red_m[w] == -INFINITY ? 0.f : red_s[w] * fast_exp2(red_m[w] - bm);
  }
  const float l2 = bm + fast_log2(bs);
  if (threadIdx.x == 0) {
    const float lse = l2 * kLn2;
    lse_out[row] = lse;
    loss[row] = counts ? lse - xt : 0.f;
  }
  if constexpr (!kGrad) return;
  float scale = given;
  if (kCountsItself<NT, NV> && count_rows > 0) {
    int n = 0;
#pragma unroll
    for (int w = 0; w < W; ++w) n += red_n[w];
    scale = unit / static_cast<float>(n > 0 ? n : 1);
  }
  const int t_piece = static_cast<int>(t) / V, t_elem = static_cast<int>(t) % V;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int v = threadIdx.x + j * NT;
    if (v < nvec) {
      float e[V];
      unpack_piece<T>(raw[j], e);
#pragma unroll
      for (int i = 0; i < V; ++i) e[i] = fast_exp2(e[i] * kLog2e - l2);
      if (v == t_piece) {   // one lane of the workgroup
#pragma unroll
        for (int i = 0; i < V; ++i) e[i] -= i == t_elem ? 1.f : 0.f;
      }
#pragma unroll
      for (int i = 0; i < V; ++i) e[i] *= scale;
      io<T>::store_stream(d + static_cast<int64_t>(v) * V, e);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  if (tail < vocab) d[tail] = static_cast<T>((fast_exp2(xe * kLog2e - l2) - (tail == t ? 1.f : 0.f)) * scale);
}

// inv_count = scale / max(rows that count, 1) and, with `loss`, mean = scale * sum(loss) / count: one workgroup, a fixed order
// of summation.  (A few microseconds of launch and latency; the eight elementwise and reduction launches torch needs for
// the same took 30.)
constexpr int kMeanThreads = 1024;
__global__ __launch_bounds__(kMeanThreads) void ce_mean_kernel(const float* __restrict__ loss, const int64_t* __restrict__ targets,
                                                               float* __restrict__ mean, float* __restrict__ inv_count, float scale,
                                                               int64_t rows, int64_t vocab, int64_t ignore_index) {
  __shared__ float red_s[kMeanThreads / kWave];
  __shared__ int red_n[kMeanThreads / kWave];
  float s = 0.f;
  int n = 0;
  for (int64_t r = threadIdx.x; r < rows; r += kMeanThreads) {
    const int64_t t = targets[r];
    n += t != ignore_index && t >= 0 && t < vocab;
    if (loss != nullptr) s += loss[r];
  }
  s = wave_sum(s);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) n += __shfl_xor(n, off, kWave);
  if (threadIdx.x % kWave == 0) { red_s[threadIdx.x / kWave] = s; red_n[threadIdx.x / kWave] = n; }
  __syncthreads();
  if (threadIdx.x == 0) {
    float total = 0.f;
    int count = 0;
    for (int w = 0; w < kMeanThreads / kWave; ++w) { total += red_s[w]; count += red_n[w]; }
    const float c = static_cast<float>(count > 0 ? count : 1);
    *inv_count = scale / c;
    if (loss != nullptr) *mean = total / c * scale;
  }
}

// Pieces of 16 bytes per row that the one-pass kernel can hold: 1024 threads x 16.
constexpr int kOnePassMaxPieces = 1024 * 16;
bool one_pass_fits(int64_t vocab, int dtype) { return vocab / (dtype == PICO_BF16 ? 8 : 4) <= kOnePassMaxPieces; }

// count(): the launch that fills inv_count, where the kernel does not count by itself
template <typename T, bool kGrad, typename Count>
void launch_one_pass(const void* logits, const int64_t* targets, float* loss, float* lse, const float* inv_count, void* dlogits,
                     int64_t rows, int vocab, int64_t ld, int64_t dld, int64_t ignore_index, float unit, const Count& count, hipStream_t s) {
  auto go = [&](auto kern, int threads, bool can_count = true) {
    const bool itself = can_count && rows <= kCountMost * threads;
    if (kGrad && !itself) count();
    hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(rows)), dim3(threads), 0, s, static_cast<const T*>(logits), targets, loss, lse,
                       inv_count, static_cast<T*>(dlogits), vocab, ld, dld, ignore_index, kGrad && itself ? static_cast<int>(rows) : 0, unit);
  };
  // the narrowest workgroup that holds the row in 4 pieces per lane, 8 from 256 threads on: in a wider one most lanes of a
  // short row would idle, and every row pays for a barrier over all its waves
  const int pieces = (vocab + io<T>::kVec - 1) / io<T>::kVec;
  if (pieces <= 64 * 4) go(ce_one_pass_kernel<T, 64, 4, kGrad>, 64);
  else if (pieces <= 128 * 4) go(ce_one_pass_kernel<T, 128, 4, kGrad>, 128);
  else if (pieces <= 256 * 4) go(ce_one_pass_kernel<T, 256, 4, kGrad>, 256);
  else if constexpr (kGrad) {
    if (pieces <= 256 * 8) go(ce_one_pass_kernel<T, 256, 8, true>, 256);
    else if (pieces <= 512 * 8) go(ce_one_pass_kernel<T, 512, 8, true>, 512);
    else if (pieces <= 1024 * 6) go(ce_one_pass_kernel<T, 1024, 6, true>, 1024);
    else if (pieces <= 1024 * 8) go(ce_one_pass_kernel<T, 1024, 8, true>, 1024, kCountsItself<1024, 8>);
    else go(ce_one_pass_kernel<T, 1024, 16, true>, 1024);
  }
}
// the forward alone streams long rows through its 512 threads at 6.3 TB/s; rows of up to this many pieces take the kernel
// above with the gradient left out (16384 x 2000 in bf16: 37 us with the streaming kernel)
constexpr int kForwardShortPieces = 256 * 4;

int check_ce(const char* fn, int64_t rows, int64_t vocab, int64_t ld, int dtype) {
  if (dtype != PICO_BF16 && dtype != PICO_F32) return fail(PICO_ERR_DTYPE, "%s: dtype code %d not supported", fn, dtype);
  const int vec = dtype == PICO_BF16 ? 8 : 4;
  if (rows < 0 || vocab <= 0 || vocab > 0x7fffffff) return fail(PICO_ERR_SHAPE, "%s: rows=%lld vocab=%lld", fn,
                                                                static_cast<long long>(rows), static_cast<long long>(vocab));
  if (ld < vocab || ld % vec != 0) return fail(PICO_ERR_STRIDE, "%s: row pitch %lld must be >= vocab and a multiple of %d",
                                               fn, static_cast<long long>(ld), vec);
  return PICO_OK;
}

}  // namespace
}  // namespace pico

using namespace pico;

extern "C" int pico_cross_entropy_fwd(const void* logits, const int64_t* targets, float* loss, float* lse, int64_t rows,
                                      int64_t vocab, int64_t ld, int64_t ignore_index, int dtype, void* stream) {
  if (int rc = check_ce("pico_cross_entropy_fwd", rows, vocab, ld, dtype)) return rc;
  if (rows == 0) return PICO_OK;
  if (!logits || !targets || !loss || !lse) return fail(PICO_ERR_NULL, "pico_cross_entropy_fwd: logits, targets, loss and lse are required");
  if (!aligned16(logits)) return fail(PICO_ERR_ALIGN, "pico_cross_entropy_fwd: logits must be 16-byte aligned");
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (vocab <= kForwardShortPieces * (dtype == PICO_BF16 ? 8 : 4)) {
    if (dtype == PICO_BF16)
      launch_one_pass<__bf16, false>(logits, targets, loss, lse, nullptr, nullptr, rows, static_cast<int>(vocab), ld, 0, ignore_index, 1.f, [] {}, s);
    else
      launch_one_pass<float, false>(logits, targets, loss, lse, nullptr, nullptr, rows, static_cast<int>(vocab), ld, 0, ignore_index, 1.f, [] {}, s);
  } else if (dtype == PICO_BF16)
    hipLaunchKernelGGL(ce_fwd_kernel<__bf16>, dim3(static_cast<unsigned>(rows)), dim3(kThreads), 0, s,
                       static_cast<const __bf16*>(logits), targets, loss, lse, static_cast<int>(vocab), ld, ignore_index);
  else
    hipLaunchKernelGGL(ce_fwd_kernel<float>, dim3(static_cast<unsigned>(rows)), dim3(kThreads), 0, s,
                       static_cast<const float*>(logits), targets, loss, lse, static_cast<int>(vocab), ld, ignore_index);
  return check_launch("pico_cross_entropy_fwd");
}

extern "C" int pico_cross_entropy_bwd(const void* logits, const int64_t* targets, const float* lse, const float* scale,
                                      void* dlogits, int64_t rows, int64_t vocab, int64_t ld, int64_t dld,
                                      int64_t ignore_index, int dtype, void* stream) {
  if (int rc = check_ce("pico_cross_entropy_bwd", rows, vocab, ld, dtype)) return rc;
  if (int rc = check_ce("pico_cross_entropy_bwd", rows, vocab, dld, dtype)) return rc;
  if (rows == 0) return PICO_OK;
  if (!logits || !targets || !lse || !scale || !dlogits)
    return fail(PICO_ERR_NULL, "pico_cross_entropy_bwd: logits, targets, lse, scale and dlogits are required");
  if (!aligned16(logits) || !aligned16(dlogits)) return fail(PICO_ERR_ALIGN, "pico_cross_entropy_bwd: logits and dlogits must be 16-byte aligned");
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (dtype == PICO_BF16)
    hipLaunchKernelGGL(ce_bwd_kernel<__bf16>, dim3(static_cast<unsigned>(rows)), dim3(kThreads), 0, s,
                       static_cast<const __bf16*>(logits), targets, lse, scale, nullptr, 0, static_cast<__bf16*>(dlogits), rows,
                       static_cast<int>(vocab), ld, dld, ignore_index);
  else
    hipLaunchKernelGGL(ce_bwd_kernel<float>, dim3(static_cast<unsigned>(rows)), dim3(kThreads), 0, s,
                       static_cast<const float*>(logits), targets, lse, scale, nullptr, 0, static_cast<float*>(dlogits), rows,
                       static_cast<int>(vocab), ld, dld, ignore_index);
  return check_launch("pico_cross_entropy_bwd");
}

extern "C" int pico_cross_entropy_one_pass(int64_t vocab, int dtype) {
  return (dtype == PICO_BF16 || dtype == PICO_F32) && vocab > 0 && one_pass_fits(vocab, dtype);
}

namespace {
int run_mean_fwd(const char* fn, const void* logits, const int64_t* targets, float* loss, float* lse, float* mean, float* inv_count,
                 void* dlogits, float scale, int64_t rows, int64_t vocab, int64_t ld, int64_t dld, int64_t ignore_index, int dtype,
                 void* stream) {
  if (int rc = check_ce(fn, rows, vocab, ld, dtype)) return rc;
  if (!mean || !inv_count) return fail(PICO_ERR_NULL, "%s: mean and inv_count are required", fn);
  if (rows > 0 && (!logits || !targets || !loss || !lse)) return fail(PICO_ERR_NULL, "%s: logits, targets, loss and lse are required", fn);
  if (!aligned16(logits) || !aligned16(dlogits)) return fail(PICO_ERR_ALIGN, "%s: logits and dlogits must be 16-byte aligned", fn);
  hipStream_t s = static_cast<hipStream_t>(stream);
  auto finish = [&](const float* l) {
    hipLaunchKernelGGL(ce_mean_kernel, dim3(1), dim3(kMeanThreads), 0, s, l, targets, mean, inv_count, scale, rows, vocab, ignore_index);
  };
  if (dlogits != nullptr && rows > 0) {
    if (int rc = check_ce(fn, rows, vocab, dld, dtype)) return rc;
    if (!one_pass_fits(vocab, dtype))
      return fail(PICO_ERR_SHAPE, "%s: vocab=%lld does not fit one pass (see pico_cross_entropy_one_pass)", fn, static_cast<long long>(vocab));
    auto count = [&] { finish(nullptr); };   // the gradient needs scale / count
    if (dtype == PICO_BF16)
      launch_one_pass<__bf16, true>(logits, targets, loss, lse, inv_count, dlogits, rows, static_cast<int>(vocab), ld, dld, ignore_index, scale, count, s);
    else
      launch_one_pass<float, true>(logits, targets, loss, lse, inv_count, dlogits, rows, static_cast<int>(vocab), ld, dld, ignore_index, scale, count, s);
  } else if (rows > 0) {
    if (int rc = pico_cross_entropy_fwd(logits, targets, loss, lse, rows, vocab, ld, ignore_index, dtype, stream)) return rc;
  }
  finish(loss != nullptr ? loss : lse);   // (no rows: nothing is read, the mean is 0)
  return check_launch(fn);
}

}  // namespace

extern "C" int pico_cross_entropy_mean_fwd(const void* logits, const int64_t* targets, float* loss, float* lse, float* mean,
                                           float* inv_count, void* dlogits, int64_t rows, int64_t vocab, int64_t ld, int64_t dld,
                                           int64_t ignore_index, int dtype, void* stream) {
  return run_mean_fwd("pico_cross_entropy_mean_fwd", logits, targets, loss, lse, mean, inv_count, dlogits, 1.f, rows, vocab, ld, dld,
                      ignore_index, dtype, stream);
}

extern "C" int pico_cross_entropy_scaled_mean_fwd(const void* logits, const int64_t* targets, float* loss, float* lse, float* mean,
                                                  float* inv_count, void* dlogits, float scale, int64_t rows, int64_t vocab, int64_t ld,
                                                  int64_t dld, int64_t ignore_index, int dtype, void* stream) {
  return run_mean_fwd("pico_cross_entropy_scaled_mean_fwd", logits, targets, loss, lse, mean, inv_count, dlogits, scale, rows, vocab, ld,
                      dld, ignore_index, dtype, stream);
}

extern "C" int pico_cross_entropy_mean_bwd(const void* logits, const int64_t* targets, const float* lse, const float* inv_count,
                                           const float* grad_out, void* dlogits, int have_unit, int64_t rows, int64_t vocab, int64_t ld,
                                           int64_t dld, int64_t ignore_index, int dtype, void* stream) {
  const char* fn = "pico_cross_entropy_mean_bwd";
  if (int rc = check_ce(fn, rows, vocab, ld, dtype)) return rc;
  if (int rc = check_ce(fn, rows, vocab, dld, dtype)) return rc;
  if (rows == 0) return PICO_OK;
  if (!logits || !targets || !lse || !inv_count || !grad_out || !dlogits)
    return fail(PICO_ERR_NULL, "%s: logits, targets, lse, inv_count, grad_out and dlogits are required", fn);
  if (!aligned16(logits) || !aligned16(dlogits)) return fail(PICO_ERR_ALIGN, "%s: logits and dlogits must be 16-byte aligned", fn);
  hipStream_t s = static_cast<hipStream_t>(stream);
  // (with the gradient at hand the launch usually only looks at grad_out: few workgroups, which walk the rows if they must)
  const dim3 grid(static_cast<unsigned>(have_unit ? std::min<int64_t>(rows, 1024) : rows));
  if (dtype == PICO_BF16)
    hipLaunchKernelGGL(ce_bwd_kernel<__bf16>, grid, dim3(kThreads), 0, s,
                       static_cast<const __bf16*>(logits), targets, lse, inv_count, grad_out, have_unit, static_cast<__bf16*>(dlogits), rows,
                       static_cast<int>(vocab), ld, dld, ignore_index);
  else
    hipLaunchKernelGGL(ce_bwd_kernel<float>, grid, dim3(kThreads), 0, s,
                       static_cast<const float*>(logits), targets, lse, inv_count, grad_out, have_unit, static_cast<float*>(dlogits), rows,
                       static_cast<int>(vocab), ld, dld, ignore_index);
  return check_launch(fn);
}
