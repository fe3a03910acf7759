// Matrix products of small layers: C = op(A) op(B) in bf16 with fp32 accumulation, where the GEMM library's tiles leave most
// CUs idle and its time is that of one workgroup's walk along the contraction.
//
// What bounds them is latency: [512 x 576] @ [576 x 576] moves 2 MB and takes 0.3 GFLOP, half a microsecond of either, but
// every step of a walk waits for memory.  So: tiles of 64 x 64 (enough workgroups from few rows), three steps of 64 requested
// ahead in registers, two LDS buffers, and the walk dealt to KS groups of four waves inside the workgroup, whose fp32 sums
// meet in LDS in the order of the groups (the same result on every run, no second launch).  A step costs 0.3 us in one group
// and start plus end 3 us: [512 x 960]^T [512 x 576] takes 6.0 us (library 9.2).
// With more tiles than CUs the reads of LDS are the bound, 3 KiB per MFMA of a tile of 64; tiles of 128 take 2 KiB, and two
// workgroups fit a CU: [451 x 9792]^T [451 x 3264] 44 us = 655 TFLOP/s.  (A walk dealt to four groups was level with two or behind
// where pico_product_mid leaves it here: [3950 x 15800]^T [3950 x 40] 22.7 us, in two 21.3.)  The error against 64
// bits is the library's (1.66e-3, the rounding to bf16).
#include "attn_common.h"

namespace pico {
namespace {

constexpr int kStep = 64;   // contraction per step
constexpr int kAhead = 3;

struct ProductParams {
  const __bf16 *a, *b;
  __bf16* c;
  int M, N, K;
  int64_t lda, ldb;   // elements between the rows of a and b as they lie in memory
  int tiles_m, tiles_n;
};

// One operand's piece of 64 W rows and 64 of contraction.  kSlow false: rows of the piece are rows of the matrix (contraction
// contiguous), true: the matrix lies with its contraction as the slow axis and is staged that way.  The staged rows' pitch
// spreads the reads of a fragment over the banks: 16-byte reads down a column, or transposing reads of four rows at once.
template <bool kSlow, int W>
struct Operand {
  static constexpr int kRows = 64 * W, kPieces = 2 * W, kPerRow = kSlow ? 8 * W : 8, kPitch = kSlow ? kRows + 16 * W : kStep + 8;
  static constexpr int kBytes = (kSlow ? kStep : kRows) * kPitch * 2;
  buffer_rsrc window;
  uint32_t off[kPieces];   // byte offset of this thread's 16-byte pieces at contraction 0
  int k[kPieces];          // their first contraction index
  uint32_t step_bytes;     // from one contraction index to the next
  bool out[kPieces];       // columns past the matrix (kSlow)

  __device__ __forceinline__ void open(const __bf16* base, int64_t ld, int first, int rows, int K, int tid) {
    const int left = min(kRows, rows - first);
    if constexpr (kSlow) window = make_buffer(base + first, static_cast<uint32_t>(((K - 1) * ld + left) * 2));
    else window = make_buffer(base + first * ld, span_bytes(left, ld, K));
    step_bytes = kSlow ? static_cast<uint32_t>(ld * 2) : 2u;
#pragma unroll
    for (int i = 0; i < kPieces; ++i) {
      const int idx = tid + 256 * i, r = idx / kPerRow, cv = idx % kPerRow;
      off[i] = static_cast<uint32_t>((r * ld + cv * 8) * 2);
      k[i] = kSlow ? r : cv * 8;
      out[i] = kSlow && cv * 8 >= left;
    }
  }
  // pieces past the contraction's end or the matrix' edge read as zeros
  __device__ __forceinline__ void load(int k0, int k_end, u32x4 (&r)[kPieces]) const {
#pragma unroll
    for (int i = 0; i < kPieces; ++i)
      r[i] = buffer_load_b128(window, k0 + k[i] < k_end && !out[i] ? off[i] + static_cast<uint32_t>(k0) * step_bytes : 0xfffffff0u);
  }
  static __device__ __forceinline__ void stage(unsigned char* tile, int tid, const u32x4 (&r)[kPieces]) {
#pragma unroll
    for (int i = 0; i < kPieces; ++i) {
      const int idx = tid + 256 * i;
      *reinterpret_cast<u32x4*>(tile + (idx / kPerRow) * kPitch * 2 + (idx % kPerRow) * 16) = r[i];
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

template <bool kSlowA, bool kSlowB, int W, int KS>
struct Shape {
  using A = Operand<kSlowA, W>;
  using B = Operand<kSlowB, W>;
  static constexpr int kTile = 64 * W, kOutPitch = kTile + 8;
  static constexpr int kBuffer = A::kBytes + B::kBytes;
  static constexpr int kSums = (KS - 1) * 4 * W * W * 16 * kWave * 4;   // the other groups' accumulators
  static constexpr int kStaging = KS * 2 * kBuffer, kEnd = kSums + kTile * kOutPitch * 2;
  static constexpr int kLds = kStaging > kEnd ? kStaging : kEnd;
};

template <bool kSlowA, bool kSlowB, int W, int KS>
__global__ __launch_bounds__(256 * KS, 2) void product_kernel(const ProductParams p) {
  using S = Shape<kSlowA, kSlowB, W, KS>;
  using A = typename S::A;
  using B = typename S::B;
  constexpr int kTile = S::kTile;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int group = wave / 4, tid = threadIdx.x % 256, wm = (wave % 4) / 2 * 32 * W, wn = (wave % 4) % 2 * 32 * W;
  // workgroups go round the eight XCDs: each takes a run of neighbouring tiles, along the shorter side of the output, whose
  // operand then stays in its L2 ([577 x 2048]^T [577 x 8192] 42 us along the longer side, 34 along the shorter)
  const int tiles = p.tiles_m * p.tiles_n, xcd = blockIdx.x % 8, id = xcd * (tiles / 8) + min(xcd, tiles % 8) + blockIdx.x / 8;
  const bool down = p.tiles_m < p.tiles_n;
  const int m0 = (down ? id % p.tiles_m : id / p.tiles_n) * kTile, n0 = (down ? id / p.tiles_m : id % p.tiles_n) * kTile;
  const int steps = (p.K + kStep - 1) / kStep, trips = (steps + KS - 1) / KS;   // every group makes the same number of trips
  const int k_first = group * trips * kStep, k_end = min(p.K, k_first + trips * kStep);
  unsigned char* buf = lds + group * 2 * S::kBuffer;
  A a;
  B b;
  a.open(p.a, p.lda, m0, p.M, p.K, tid);
  b.open(p.b, p.ldb, n0, p.N, p.K, tid);
  constexpr int kDeep = W == 1 || KS == 1 ? kAhead : 2;   // (steps requested ahead; two groups of a tile of 128 gain nothing from a third)
  u32x4 ra[kDeep][A::kPieces], rb[kDeep][B::kPieces];
#pragma unroll
  for (int u = 0; u < kDeep; ++u) {
    a.load(k_first + u * kStep, k_end, ra[u]);
    b.load(k_first + u * kStep, k_end, rb[u]);
  }
  A::stage(buf, tid, ra[0]);
  B::stage(buf + A::kBytes, tid, rb[0]);
  __syncthreads();
  f32x16 acc[W][W];
#pragma unroll
  for (int i = 0; i < W; ++i)
#pragma unroll
    for (int j = 0; j < W; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
  constexpr int kSub = kStep / 16;
  constexpr int kEarly = W == 1 ? kSub : 1;   // fragments requested before the next step's tile is written: LDS answers in order
  bf16x8 fa[kSub][W], fb[kSub][W];
  unsigned char* now = buf;
  auto request = [&](int s) {
#pragma unroll
    for (int i = 0; i < W; ++i) {
      fa[s][i] = A::fragment(now, wm + 32 * i, s, lane);
      fb[s][i] = B::fragment(now + A::kBytes, wn + 32 * i, s, lane);
    }
  };
  auto multiply = [&] {
#pragma unroll
    for (int s = 0; s < kSub; ++s) {
      if (s + kEarly < kSub) request(s + kEarly);
#pragma unroll
      for (int i = 0; i < W; ++i)
#pragma unroll
        for (int j = 0; j < W; ++j) acc[i][j] = mfma32(fb[s][j], fa[s][i], acc[i][j]);   // C^T: a lane holds one row of C, its registers columns 8 q + 4 h ..+3
    }
  };
  // Straight-line code with nothing but one exit: requests are not skipped towards the walk's end (past it they read no
  // memory).  Skipped under a condition they would leave the compiler unsure how many are in flight, and it would wait for all
  // of them in every step instead of for the oldest ([2331 x 1024]^T [2331 x 1024] 15.8 us, as it is 14.8; [512 x 3072] @ [3072
  // x 576] 16.9, 14.4).
  for (int t = 0;;) {
#pragma unroll
    for (int u = 0; u < 2 * kDeep; ++u) {
      const int next = (u + 1) % kDeep, here = u % kDeep;
      now = buf + (u & 1) * S::kBuffer;
      unsigned char* then = buf + (~u & 1) * S::kBuffer;
#pragma unroll
      for (int s = 0; s < kEarly; ++s) request(s);
      if (++t >= trips) goto last;   // (uniform over the workgroup)
      __builtin_amdgcn_sched_barrier(0);
      A::stage(then, tid, ra[next]);
      B::stage(then + A::kBytes, tid, rb[next]);
      a.load(k_first + (t + kDeep - 1) * kStep, k_end, ra[here]);
      b.load(k_first + (t + kDeep - 1) * kStep, k_end, rb[here]);
      multiply();
      __syncthreads();   // `now` may be filled again, `then` is complete
    }
  }
last:
  multiply();
  __syncthreads();
  if constexpr (KS > 1) {
    float* sums = reinterpret_cast<float*>(lds);
    auto place = [&](int w, int i, int j, int q) { return sums + ((((w * W + i) * W + j) * 4 + q) * kWave + lane) * 4; };
    if (group > 0) {
#pragma unroll
      for (int i = 0; i < W; ++i)
#pragma unroll
        for (int j = 0; j < W; ++j)
#pragma unroll
          for (int q = 0; q < 4; ++q)
            *reinterpret_cast<f32x4*>(place(wave - 4, i, j, q)) = f32x4{acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
    }
    __syncthreads();
    if (group == 0) {
#pragma unroll
      for (int g = 0; g < KS - 1; ++g)
#pragma unroll
        for (int i = 0; i < W; ++i)
#pragma unroll
          for (int j = 0; j < W; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              const f32x4 v = *reinterpret_cast<const f32x4*>(place(g * 4 + wave, i, j, q));
#pragma unroll
              for (int e = 0; e < 4; ++e) acc[i][j][4 * q + e] += v[e];
            }
    }
  }
  // the tile leaves through LDS as whole lines (behind the groups' sums, which may still be read)
  unsigned char* out = lds + S::kSums;
  if (group == 0) {
#pragma unroll
    for (int i = 0; i < W; ++i)
#pragma unroll
      for (int j = 0; j < W; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          bf16x4 v;
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = static_cast<__bf16>(acc[i][j][4 * q + e]);
          *reinterpret_cast<bf16x4*>(out + ((wm + 32 * i + lane % 32) * S::kOutPitch + wn + 32 * j + 8 * q + 4 * (lane / 32)) * 2) = v;
        }
  }
  __syncthreads();
  for (int idx = threadIdx.x; idx < kTile * kTile / 8; idx += 256 * KS) {
    const int r = idx / (kTile / 8), cv = idx % (kTile / 8);
    if (m0 + r < p.M && n0 + cv * 8 < p.N)
      *reinterpret_cast<u32x4*>(p.c + static_cast<int64_t>(m0 + r) * p.N + n0 + cv * 8) = *reinterpret_cast<const u32x4*>(out + r * S::kOutPitch * 2 + cv * 16);
  }
}

template <bool kSlowA, bool kSlowB, int W, int KS>
int launch(const ProductParams& p, hipStream_t s) {
  constexpr int kLds = Shape<kSlowA, kSlowB, W, KS>::kLds;
  static_assert(kLds <= 160 * 1024);
  static LdsOnce reserved;
  if (kLds > 48 * 1024 && !reserve_lds_once(reserved, reinterpret_cast<const void*>(&product_kernel<kSlowA, kSlowB, W, KS>), kLds))
    return fail(PICO_ERR_LAUNCH, "pico_product: cannot reserve %d bytes of LDS", kLds);
  hipLaunchKernelGGL((product_kernel<kSlowA, kSlowB, W, KS>), dim3(static_cast<unsigned>(p.tiles_m) * p.tiles_n), dim3(256 * KS), kLds, s, p);
  return check_launch("pico_product");
}
template <bool kSlowA, bool kSlowB>
int launch_shape(const ProductParams& p, int tile, int groups, hipStream_t s) {
  if (tile == 128) return groups == 1 ? launch<kSlowA, kSlowB, 2, 1>(p, s) : launch<kSlowA, kSlowB, 2, 2>(p, s);
  return groups == 1 ? launch<kSlowA, kSlowB, 1, 1>(p, s) : launch<kSlowA, kSlowB, 1, 2>(p, s);   // (4: as 2)
}

}  // namespace
}  // namespace pico

using namespace pico;

extern "C" int pico_product_takes(int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int a_slow, int b_slow) {
  constexpr int64_t kMost = 0x7fffffff;
  if (M < 1 || N < 1 || K < 1 || M > kMost || N > kMost || K > kMost - 4096 || N % 8 != 0 || (a_slow ? M : K) % 8 != 0 ||
      (b_slow ? N : K) % 8 != 0 || lda % 8 != 0 || ldb % 8 != 0 || lda < (a_slow ? M : K) || ldb < (b_slow ? N : K))
    return 0;
  // the windows of the buffer loads: a tile's rows, or the whole contraction where that is the slow axis
  if (lda > kMost / 2 || ldb > kMost / 2 || ((a_slow ? K + 1024 : 128) * lda + K) * 2 > kMost || ((b_slow ? K + 1024 : 128) * ldb + K) * 2 > kMost)
    return 0;
  return ((M + 63) / 64) * ((N + 63) / 64) <= kMost;
}

extern "C" int pico_product(const void* a, const void* b, void* c, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int a_slow,
                            int b_slow, int tile, int groups, void* stream) {
  if (!pico_product_takes(M, N, K, lda, ldb, a_slow, b_slow))
    return fail(PICO_ERR_SHAPE, "pico_product: M=%lld N=%lld K=%lld row pitches %lld, %lld (rows of a, b and c and the pitches must be multiples of 8 elements, a tile's rows span less than 2 GiB)",
                (long long)M, (long long)N, (long long)K, (long long)lda, (long long)ldb);
  if (!(tile == 64 && (groups == 1 || groups == 2 || groups == 4)) && !(tile == 128 && (groups == 1 || groups == 2)))
    return fail(PICO_ERR_SHAPE, "pico_product: tile=%d groups=%d (64 with 1, 2 or 4 groups, 128 with 1 or 2)", tile, groups);
  if (!a || !b || !c) return fail(PICO_ERR_NULL, "pico_product: a, b and c are required");
  if (!aligned16(a) || !aligned16(b) || !aligned16(c)) return fail(PICO_ERR_ALIGN, "pico_product: pointers must be 16-byte aligned");
  const int64_t tm = (M + tile - 1) / tile, tn = (N + tile - 1) / tile;
  const ProductParams p = {static_cast<const __bf16*>(a), static_cast<const __bf16*>(b), static_cast<__bf16*>(c), (int)M, (int)N, (int)K, lda, ldb, (int)tm, (int)tn};
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (a_slow) return b_slow ? launch_shape<true, true>(p, tile, groups, s) : launch_shape<true, false>(p, tile, groups, s);
  return b_slow ? launch_shape<false, true>(p, tile, groups, s) : launch_shape<false, false>(p, tile, groups, s);
}
