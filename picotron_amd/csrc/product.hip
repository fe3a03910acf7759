// Matrix products of small layers: C = op(A) op(B) in bf16 with fp32 accumulation, where the GEMM library's tiles leave most
// CUs idle and its time is that of one workgroup's walk along the contraction.
//
// What bounds them is latency: [512 x 576] @ [576 x 576] moves 2 MB and takes 0.3 GFLOP, half a microsecond of either, but
// every step of a walk waits for memory.  So: tiles of 64 x 64 (enough workgroups from few rows), three steps of 64 requested
// ahead in registers, two LDS buffers, and the walk dealt to KS groups of four waves inside the workgroup, whose fp32 sums
// meet in LDS in the order of the groups (the same result on every run, no second launch).  A step costs 0.4 us in one group
// and start plus end 2.5 us.  Over 135 shapes drawn from layers of 128 .. 4096 columns and 100 .. 6000 rows that the caller's
// rule sends here, the geometric mean of the time over the library's is 0.61 for weight gradients, 0.78 for input gradients
// and 0.82 for the forward, 0.99 at worst; the error against 64 bits is the library's (1.66e-3, the rounding to bf16).
#include "attn_common.h"

namespace pico {
namespace {

constexpr int kTile = 64, kStep = 64;      // rows / columns of a tile, contraction per step
constexpr int kPitch = kTile + 8;          // elements between the rows of a staged tile (16 bytes of padding against bank conflicts)
constexpr int kTileBytes = kTile * kPitch * 2;
constexpr int kAhead = 3;

struct ProductParams {
  const __bf16 *a, *b;
  __bf16* c;
  int M, N, K;
  int64_t lda, ldb;   // elements between the rows of a and b as they lie in memory
  int tiles_n;
};

// One operand's 64 x 64 piece: kSlow false: rows of the tile are rows of the matrix (contraction contiguous), true: the matrix
// lies with its contraction as the slow axis and is staged that way.
template <bool kSlow>
struct Operand {
  buffer_rsrc window;
  uint32_t off[2];        // byte offset of this thread's two 16-byte pieces at contraction 0
  int k[2];               // their first contraction index
  uint32_t step_bytes;    // from one contraction index to the next
  bool out[2];            // columns past the matrix (kSlow)

  __device__ __forceinline__ void open(const __bf16* base, int64_t ld, int first, int rows, int K, int tid) {
    const int left = min(kTile, rows - first);
    if constexpr (kSlow) window = make_buffer(base + first, static_cast<uint32_t>(((K - 1) * ld + left) * 2));
    else window = make_buffer(base + first * ld, span_bytes(left, ld, K));
    step_bytes = kSlow ? static_cast<uint32_t>(ld * 2) : 2u;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int idx = tid + 256 * i, r = idx / 8, cv = idx % 8;
      off[i] = static_cast<uint32_t>((r * ld + cv * 8) * 2);
      k[i] = kSlow ? r : cv * 8;
      out[i] = kSlow && cv * 8 >= left;
    }
  }
  // pieces past the contraction's end or the matrix' edge read as zeros
  __device__ __forceinline__ void load(int k0, int k_end, u32x4 (&r)[2]) const {
#pragma unroll
    for (int i = 0; i < 2; ++i) r[i] = buffer_load_b128(window, k0 + k[i] < k_end && !out[i] ? off[i] + static_cast<uint32_t>(k0) * step_bytes : 0xfffffff0u);
  }
  static __device__ __forceinline__ void stage(unsigned char* tile, int tid, const u32x4 (&r)[2]) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int idx = tid + 256 * i;
      *reinterpret_cast<u32x4*>(tile + (idx / 8) * kPitch * 2 + (idx % 8) * 16) = r[i];
    }
  }
  // lane n gets row `first` + n % 32 of the operand, contraction 16 s + 8 (n / 32) ..+7
  static __device__ __forceinline__ bf16x8 fragment(const unsigned char* tile, int first, int s, int lane) {
    const __bf16* t = reinterpret_cast<const __bf16*>(tile);
    const int h = lane / 32;
    if constexpr (kSlow)
      return lds_read_tr_pair_step(t + (16 * s + 8 * h + (lane % 16) / 4) * kPitch + first + 16 * ((lane % 32) / 16) + 4 * (lane % 4), 4 * kPitch);
    else
      return *reinterpret_cast<const bf16x8*>(t + (first + lane % 32) * kPitch + 16 * s + 8 * h);
  }
};

template <bool kSlowA, bool kSlowB, int KS>
__global__ __launch_bounds__(256 * KS) void product_kernel(const ProductParams p) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int group = wave / 4, tid = threadIdx.x % 256, wm = (wave % 4) / 2 * 32, wn = (wave % 4) % 2 * 32;
  const int m0 = blockIdx.x / p.tiles_n * kTile, n0 = blockIdx.x % p.tiles_n * kTile;
  const int steps = (p.K + kStep - 1) / kStep, trips = (steps + KS - 1) / KS;   // every group makes the same number of trips
  const int k_first = group * trips * kStep, k_end = min(p.K, k_first + trips * kStep);
  unsigned char* buf = lds + group * 4 * kTileBytes;
  Operand<kSlowA> a;
  Operand<kSlowB> b;
  a.open(p.a, p.lda, m0, p.M, p.K, tid);
  b.open(p.b, p.ldb, n0, p.N, p.K, tid);
  u32x4 ra[kAhead][2], rb[kAhead][2];
#pragma unroll
  for (int u = 0; u < kAhead; ++u) {
    a.load(k_first + u * kStep, k_end, ra[u]);
    b.load(k_first + u * kStep, k_end, rb[u]);
  }
  Operand<kSlowA>::stage(buf, tid, ra[0]);
  Operand<kSlowB>::stage(buf + kTileBytes, tid, rb[0]);
  __syncthreads();
  f32x16 acc;
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] = 0.f;
  for (int t0 = 0; t0 < trips; t0 += kAhead) {
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      const int t = t0 + u;
      if (t < trips) {   // (uniform over the workgroup)
        const int next = (u + 1) % kAhead;
        unsigned char *now = buf + (t & 1) * 2 * kTileBytes, *then = buf + (~t & 1) * 2 * kTileBytes;
        bf16x8 fa[kStep / 16], fb[kStep / 16];   // requested before the next step's tile is written: LDS answers in order
#pragma unroll
        for (int s = 0; s < kStep / 16; ++s) {
          fa[s] = Operand<kSlowA>::fragment(now, wm, s, lane);
          fb[s] = Operand<kSlowB>::fragment(now + kTileBytes, wn, s, lane);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (t + 1 < trips) {
          Operand<kSlowA>::stage(then, tid, ra[next]);
          Operand<kSlowB>::stage(then + kTileBytes, tid, rb[next]);
        }
        if (t + kAhead < trips) {
          a.load(k_first + (t + kAhead) * kStep, k_end, ra[u]);
          b.load(k_first + (t + kAhead) * kStep, k_end, rb[u]);
        }
#pragma unroll
        for (int s = 0; s < kStep / 16; ++s) acc = mfma32(fb[s], fa[s], acc);   // C^T: a lane holds one row of C, its registers columns 8 j + 4 h ..+3
        __syncthreads();   // `now` may be filled again, `then` is complete
      }
    }
  }
  if constexpr (KS > 1) {
    float* sums = reinterpret_cast<float*>(lds);
    if (group > 0) {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        *reinterpret_cast<f32x4*>(sums + (((wave - 4) * 4 + j) * kWave + lane) * 4) = f32x4{acc[4 * j], acc[4 * j + 1], acc[4 * j + 2], acc[4 * j + 3]};
    }
    __syncthreads();
    if (group == 0) {
#pragma unroll
      for (int g = 0; g < KS - 1; ++g)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const f32x4 v = *reinterpret_cast<const f32x4*>(sums + (((g * 4 + wave) * 4 + j) * kWave + lane) * 4);
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[4 * j + e] += v[e];
        }
    }
  }
  // the tile leaves through LDS as whole lines (behind the groups' sums, which may still be read)
  unsigned char* out = lds + (KS - 1) * 4 * 4 * kWave * 16;
  if (group == 0) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      bf16x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = static_cast<__bf16>(acc[4 * j + e]);
      *reinterpret_cast<bf16x4*>(out + ((wm + lane % 32) * kPitch + wn + 8 * j + 4 * (lane / 32)) * 2) = v;
    }
  }
  __syncthreads();
  for (int idx = threadIdx.x; idx < kTile * kTile / 8; idx += 256 * KS) {
    const int r = idx / 8, cv = idx % 8;
    if (m0 + r < p.M && n0 + cv * 8 < p.N)
      *reinterpret_cast<u32x4*>(p.c + static_cast<int64_t>(m0 + r) * p.N + n0 + cv * 8) = *reinterpret_cast<const u32x4*>(out + r * kPitch * 2 + cv * 16);
  }
}

template <bool kSlowA, bool kSlowB, int KS>
int launch(const ProductParams& p, int64_t tiles, hipStream_t s) {
  constexpr int kStaging = KS * 4 * kTileBytes, kEnd = (KS - 1) * 4 * 4 * kWave * 16 + kTileBytes;
  constexpr int kLds = kStaging > kEnd ? kStaging : kEnd;
  static LdsOnce reserved;
  if (kLds > 48 * 1024 && !reserve_lds_once(reserved, reinterpret_cast<const void*>(&product_kernel<kSlowA, kSlowB, KS>), kLds))
    return fail(PICO_ERR_LAUNCH, "pico_product: cannot reserve %d bytes of LDS", kLds);
  hipLaunchKernelGGL((product_kernel<kSlowA, kSlowB, KS>), dim3(static_cast<unsigned>(tiles)), dim3(256 * KS), kLds, s, p);
  return check_launch("pico_product");
}
template <bool kSlowA, bool kSlowB>
int launch_groups(const ProductParams& p, int64_t tiles, int groups, hipStream_t s) {
  switch (groups) {
    case 1: return launch<kSlowA, kSlowB, 1>(p, tiles, s);
    case 2: return launch<kSlowA, kSlowB, 2>(p, tiles, s);
    default: return launch<kSlowA, kSlowB, 4>(p, tiles, s);
  }
}

}  // namespace
}  // namespace pico

using namespace pico;

extern "C" int pico_product(const void* a, const void* b, void* c, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int a_slow,
                            int b_slow, int groups, void* stream) {
  constexpr int64_t kMost = 0x7fffffff;
  if (M < 1 || N < 1 || K < 1 || M > kMost || N > kMost || K > kMost - 4 * 64 * 4 || N % 8 != 0 || (a_slow ? M : K) % 8 != 0 ||
      (b_slow ? N : K) % 8 != 0 || lda % 8 != 0 || ldb % 8 != 0 || lda < (a_slow ? M : K) || ldb < (b_slow ? N : K))
    return fail(PICO_ERR_SHAPE, "pico_product: M=%lld N=%lld K=%lld row pitches %lld, %lld (rows of a, b and c must be multiples of 8 elements)",
                (long long)M, (long long)N, (long long)K, (long long)lda, (long long)ldb);
  // the windows of the buffer loads: 64 rows, or the whole contraction where that is the slow axis
  if (lda > kMost / 2 || ldb > kMost / 2 || ((a_slow ? K + 1024 : 64) * lda + K) * 2 > kMost || ((b_slow ? K + 1024 : 64) * ldb + K) * 2 > kMost)
    return fail(PICO_ERR_SHAPE, "pico_product: an operand is too large");
  if (groups != 1 && groups != 2 && groups != 4) return fail(PICO_ERR_SHAPE, "pico_product: groups=%d (1, 2 or 4)", groups);
  if (!a || !b || !c) return fail(PICO_ERR_NULL, "pico_product: a, b and c are required");
  if (!aligned16(a) || !aligned16(b) || !aligned16(c)) return fail(PICO_ERR_ALIGN, "pico_product: pointers must be 16-byte aligned");
  const int64_t tm = (M + kTile - 1) / kTile, tn = (N + kTile - 1) / kTile;
  if (tm * tn > kMost) return fail(PICO_ERR_SHAPE, "pico_product: too many tiles");
  const ProductParams p = {static_cast<const __bf16*>(a), static_cast<const __bf16*>(b), static_cast<__bf16*>(c), (int)M, (int)N, (int)K, lda, ldb, (int)tn};
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (a_slow) return b_slow ? launch_groups<true, true>(p, tm * tn, groups, s) : launch_groups<true, false>(p, tm * tn, groups, s);
  return b_slow ? launch_groups<false, true>(p, tm * tn, groups, s) : launch_groups<false, false>(p, tm * tn, groups, s);
}
