// Gradient of the token embedding: dw[v] = sum of dy[t] over the tokens t with id v, zero elsewhere.
//
// Bound by writing dw (vocab x hidden, mostly zeros) and reading dy once.  Three launches, all sums in a fixed order:
//   1. rank + fill: the fill of dw and, in the first workgroups of the same launch, a stable sort of the tokens by id.  A
//      token's place is the number of (id, token) pairs below its own, counted against every other token: tokens^2 integer
//      compares, which for the 32768 tokens the entry point takes at most is still a fraction of the fill's time, and
//      one pass instead of a radix sort's dozen launches.
//   2. runs: a workgroup takes 8 places of the sorted order, requests their rows of dy together, adds them up run by run in
//      fp32 and writes the runs that lie within its places; what belongs to a run that reaches over an edge is left in fp32.
//   3. joins: the workgroup in whose places such a run begins adds its pieces up.
// Measured (torch's embedding backward in brackets), bf16, vocabulary 49152: 4096 tokens of 2048 columns 38 us (155), 1024 of
// 576 18 us (44), 8192 of 2048 52 us (213); 8192 times the same token 129 us (344).
#include "common.h"

#include <type_traits>

namespace pico {
namespace {

constexpr int kPlaces = 8;            // sorted places of a workgroup of the second kernel
constexpr int kRankWaves = 8;         // waves that share the counting for 64 tokens
constexpr int kFillBytes = 32768;     // of dw that a workgroup of the first kernel clears
constexpr int kRankThreads = 64 * kRankWaves;

typedef __attribute__((ext_vector_type(4))) int i32x4;

struct EmbeddingParams {
  const void* ids;
  const void* dy;
  void* dw;
  int *order, *sorted;                // token and id of every place
  float* partial;                     // [group of places][run that came in / run that goes out][hidden]
  int tokens, vocab, hidden, skip;    // skip: an id whose row stays zero (-1: none)
};

// ids outside [0, vocab) are all one, -1, which no row belongs to (as they stand, wide ones would alias rows of the vocabulary
// when they are narrowed, and the largest would leave a place of the order unwritten)
template <typename I>
__device__ __forceinline__ int id_at(const I* ids, int t, int vocab) {
  const I id = ids[t];
  return static_cast<std::make_unsigned_t<I>>(id) < static_cast<std::make_unsigned_t<I>>(vocab) ? static_cast<int>(id) : -1;
}

template <typename I>
__global__ __launch_bounds__(kRankThreads) void embedding_rank_fill_kernel(const EmbeddingParams p, const I* __restrict__ ids, int rank_blocks,
                                                                           int64_t dw_bytes) {
  __shared__ int counts[kRankWaves][64];
  __shared__ __attribute__((aligned(16))) int shared_ids[kRankWaves][64];
  const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  if (static_cast<int>(blockIdx.x) >= rank_blocks) {
    const int64_t from = static_cast<int64_t>(blockIdx.x - rank_blocks) * kFillBytes;
    const u32x4 zero = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < kFillBytes / (16 * kRankThreads); ++i) {
      const int64_t at = from + (static_cast<int64_t>(i) * kRankThreads + threadIdx.x) * 16;
      if (at < dw_bytes) *reinterpret_cast<u32x4*>(static_cast<char*>(p.dw) + at) = zero;
    }
    return;
  }
  const int t0 = static_cast<int>(blockIdx.x) * 64, mine = t0 + lane;
  const int my_id = mine < p.tokens ? id_at(ids, mine, p.vocab) : p.vocab;
  // every wave counts a share of the tokens, 64 at a time: a lane fetches one of them (the next 64 while these are counted), the
  // wave's piece of LDS hands all of them to every lane
  const int groups = (p.tokens + 63) / 64, g_end = groups * (wave + 1) / kRankWaves;
  auto fetch = [&](int g) {
    const int j = g * 64 + lane;
    return g < g_end && j < p.tokens ? id_at(ids, j, p.vocab) : 0x7fffffff;   // (past the end: below nothing)
  };
  int* const share = shared_ids[wave];
  int below = 0, next = fetch(groups * wave / kRankWaves);
  for (int g = groups * wave / kRankWaves; g < g_end; ++g) {
    __builtin_amdgcn_wave_barrier();   // (LDS answers a wave in order)
    share[lane] = next;
    __builtin_amdgcn_wave_barrier();
    next = fetch(g + 1);
    const int j0 = g * 64;
    const int bound = my_id + (j0 < t0);   // of equal ids the earlier token comes first
#pragma unroll
    for (int j = 0; j < 64; j += 4) {
      const i32x4 id = *reinterpret_cast<const i32x4*>(share + j);
#pragma unroll
      for (int e = 0; e < 4; ++e) below += id[e] < bound;
    }
    if (j0 == t0)
      for (int j = 0; j < 64; ++j) below += share[j] == my_id && j < lane;
  }
  counts[wave][lane] = below;
  __syncthreads();
  if (wave > 0 || mine >= p.tokens) return;
  int place = 0;
#pragma unroll
  for (int w = 0; w < kRankWaves; ++w) place += counts[w][lane];
  p.order[place] = mine;
  p.sorted[place] = my_id;
}

template <typename T>
__device__ __forceinline__ void store_row(const EmbeddingParams& p, int id, int col, const float (&acc)[io<T>::kVec]) {
  if (id < 0 || id >= p.vocab || id == p.skip) return;
  io<T>::store(static_cast<T*>(p.dw) + static_cast<int64_t>(id) * p.hidden + col, acc);
}
__device__ __forceinline__ void store_partial(float* dst, const float* acc, int n) {
  for (int e = 0; e < n; e += 4) *reinterpret_cast<f32x4*>(dst + e) = f32x4{acc[e], acc[e + 1], acc[e + 2], acc[e + 3]};
}

template <typename T>
__global__ __launch_bounds__(256) void embedding_runs_kernel(const EmbeddingParams p) {
  constexpr int V = io<T>::kVec;
  const int p0 = static_cast<int>(blockIdx.x) * kPlaces, n = p.tokens - p0 < kPlaces ? p.tokens - p0 : kPlaces;
  const int col = (static_cast<int>(blockIdx.y * blockDim.x) + static_cast<int>(threadIdx.x)) * V;
  if (col >= p.hidden) return;
  float rows[kPlaces][V];
  int id[kPlaces];
#pragma unroll
  for (int i = 0; i < kPlaces; ++i) {
    const int at = p0 + (i < n ? i : n - 1);
    id[i] = p.sorted[at];
    io<T>::load(static_cast<const T*>(p.dy) + static_cast<int64_t>(p.order[at]) * p.hidden + col, rows[i]);
  }
  const int before = p0 > 0 ? p.sorted[p0 - 1] : -1, after = p0 + n < p.tokens ? p.sorted[p0 + n] : -1;
  bool own = p0 == 0 || before != id[0];   // the run being added up began here
  float* const left = p.partial + static_cast<int64_t>(blockIdx.x) * 2 * p.hidden + col;
  float acc[V];
#pragma unroll
  for (int e = 0; e < V; ++e) acc[e] = 0.f;
#pragma unroll
  for (int i = 0; i < kPlaces; ++i) {
    if (i >= n) break;
#pragma unroll
    for (int e = 0; e < V; ++e) acc[e] += rows[i][e];
    const bool last = i + 1 == n;
    const bool ends = last ? p0 + n >= p.tokens || after != id[i] : id[i + 1] != id[i];
    if (ends || last) {
      if (ends && own) store_row<T>(p, id[i], col, acc);
      else store_partial(left + (own ? p.hidden : 0), acc, V);
#pragma unroll
      for (int e = 0; e < V; ++e) acc[e] = 0.f;
      own = true;
    }
  }
}

template <typename T>
__global__ __launch_bounds__(256) void embedding_joins_kernel(const EmbeddingParams p) {
  constexpr int V = io<T>::kVec;
  const int p0 = static_cast<int>(blockIdx.x) * kPlaces, next = p0 + kPlaces;
  if (next >= p.tokens) return;
  const int id = p.sorted[next - 1];
  if (p.sorted[next] != id) return;                                                   // no run goes out,
  if (p.sorted[p0] == id && p0 > 0 && p.sorted[p0 - 1] == id) return;                 // or it began further up
  const int col = (static_cast<int>(blockIdx.y * blockDim.x) + static_cast<int>(threadIdx.x)) * V;
  if (col >= p.hidden) return;
  int lo = next, hi = p.tokens;   // first place past the run
  while (lo < hi) {
    const int mid = lo + (hi - lo) / 2;
    if (p.sorted[mid] <= id) lo = mid + 1;
    else hi = mid;
  }
  const int pieces = (lo - next + kPlaces - 1) / kPlaces;   // groups after this one that the run reaches into
  const float* src = p.partial + (static_cast<int64_t>(blockIdx.x) * 2 + 1) * p.hidden + col;
  float acc[V];
  for (int e = 0; e < V; ++e) acc[e] = src[e];
  src += p.hidden;
#pragma unroll 4
  for (int i = 0; i < pieces; ++i, src += 2 * p.hidden)
#pragma unroll
    for (int e = 0; e < V; e += 4) {
      const f32x4 v = *reinterpret_cast<const f32x4*>(src + e);
#pragma unroll
      for (int k = 0; k < 4; ++k) acc[e + k] += v[k];
    }
  store_row<T>(p, id, col, acc);
}

int64_t align256(int64_t n) { return (n + 255) / 256 * 256; }

template <typename T, typename I>
void launch(const EmbeddingParams& p, hipStream_t s) {
  constexpr int V = io<T>::kVec;
  const int64_t dw_bytes = static_cast<int64_t>(p.vocab) * p.hidden * sizeof(T);
  const int rank_blocks = (p.tokens + 63) / 64, groups = (p.tokens + kPlaces - 1) / kPlaces, lanes = p.hidden / V;
  hipLaunchKernelGGL((embedding_rank_fill_kernel<I>), dim3(static_cast<unsigned>(rank_blocks + (dw_bytes + kFillBytes - 1) / kFillBytes)),
                     dim3(kRankThreads), 0, s, p, static_cast<const I*>(p.ids), rank_blocks, dw_bytes);
  const int threads = std::min(256, (lanes + 63) / 64 * 64);
  hipLaunchKernelGGL(embedding_runs_kernel<T>, dim3(groups, (lanes + threads - 1) / threads), dim3(threads), 0, s, p);
  // (narrow workgroups: a run over thousands of places is spread over more CUs)
  hipLaunchKernelGGL(embedding_joins_kernel<T>, dim3(groups, (lanes + 63) / 64), dim3(64), 0, s, p);
}

}  // namespace
}  // namespace pico

using namespace pico;

extern "C" int64_t pico_embedding_bwd_workspace_bytes(int64_t tokens, int64_t hidden) {
  if (tokens < 0 || tokens > PICO_EMBEDDING_MAX_TOKENS || hidden < 0) return -1;
  const int64_t groups = (tokens + kPlaces - 1) / kPlaces;
  return 2 * align256(tokens * 4) + groups * 2 * hidden * 4;
}

extern "C" int pico_embedding_bwd(const void* ids, int id_bytes, const void* dy, void* dw, void* workspace, int64_t tokens, int64_t vocab,
                                  int64_t hidden, int64_t skip_id, int dtype, void* stream) {
  if (dtype != PICO_BF16 && dtype != PICO_F32) return fail(PICO_ERR_DTYPE, "pico_embedding_bwd: dtype code %d not supported", dtype);
  if (id_bytes != 4 && id_bytes != 8) return fail(PICO_ERR_DTYPE, "pico_embedding_bwd: ids of %d bytes not supported", id_bytes);
  if (tokens < 1 || tokens > PICO_EMBEDDING_MAX_TOKENS || vocab < 1 || vocab > 0x7ffffffe || hidden < 8 || hidden % 8 != 0 || hidden > (1 << 20))
    return fail(PICO_ERR_SHAPE, "pico_embedding_bwd: tokens=%lld (1 .. %d) vocab=%lld hidden=%lld (a multiple of 8)", (long long)tokens,
                PICO_EMBEDDING_MAX_TOKENS, (long long)vocab, (long long)hidden);
  if (!ids || !dy || !dw || !workspace) return fail(PICO_ERR_NULL, "pico_embedding_bwd: ids, dy, dw and workspace are required");
  if (!aligned16(dy) || !aligned16(dw) || !aligned16(workspace))
    return fail(PICO_ERR_ALIGN, "pico_embedding_bwd: dy, dw and workspace must be 16-byte aligned");
  EmbeddingParams p;
  p.ids = ids;
  p.dy = dy;
  p.dw = dw;
  p.tokens = static_cast<int>(tokens);
  p.vocab = static_cast<int>(vocab);
  p.hidden = static_cast<int>(hidden);
  p.skip = skip_id >= 0 && skip_id < vocab ? static_cast<int>(skip_id) : -1;
  p.order = static_cast<int*>(workspace);
  p.sorted = reinterpret_cast<int*>(static_cast<char*>(workspace) + align256(tokens * 4));
  p.partial = reinterpret_cast<float*>(static_cast<char*>(workspace) + 2 * align256(tokens * 4));
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (dtype == PICO_BF16) id_bytes == 8 ? launch<__bf16, int64_t>(p, s) : launch<__bf16, int32_t>(p, s);
  else id_bytes == 8 ? launch<float, int64_t>(p, s) : launch<float, int32_t>(p, s);
  return check_launch("pico_embedding_bwd");
}
