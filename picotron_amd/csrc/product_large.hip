// Matrix products that fill the GPU: C = op(A) op(B) in bf16 with fp32 accumulation, in any of the three layouts of a linear
// layer (forward, input gradient, weight gradient).
//
// What bounds them is the matrix pipe and the power it draws: sustained products hold the clock at 1.6 .. 1.8 GHz, so an
// instruction that moves less through the registers per product is faster as well as cheaper.  Tiles of 256 x 256 (or one side
// 192 or 128, where that fills the CUs better) by eight waves, two per SIMD, one workgroup per CU that walks its tiles; 64 of
// contraction per step, two LDS buffers.  What the forms that were built reach, TFLOP/s at [8192 x 4096] @ [4096 x 8192]:
//   * products of 16 x 16 x 32 instead of 32 x 32 x 16: 1350 -> 1430 (half the accumulator traffic);
//   * one instruction between two products, whatever it is: a request of the next tile is one `buffer_load ... lds` (its place
//     in LDS goes into m0 one product earlier, the masks of a ragged contraction are made once per tile): 1290 -> 1350;
//   * operands go to LDS without passing the registers, 16 bytes per lane, all of them requested in the half step behind the
//     one that frees the buffer; fragments are read half a step ahead;
//   * a barrier whose two halves lie apart, with products between a wave's arrival and its wait: 102 -> 98 us at [4096 x 4096] @
//     [4096 x 4096], 423 -> 395 with a contraction of 16384, whose requests take longer;
//   * four waves of 128 x 128 (a third less LDS traffic): level with long contractions, 10 % behind with short ones; the two
//     waves of a SIMD in opposite phases of memory and products: 1300.
// LDS rows are swizzled so that neither the 16-byte reads down a column (fast contraction) nor the transposing reads (slow
// contraction) have bank conflicts; all three layouts run at the same rate (98 .. 103 us at 4096 cubed), where the GEMM library
// takes 91 in the forward's, 104 in the input gradient's and 137 in the weight gradient's.  The error against 64 bits is the
// library's (1.66e-3, the rounding to bf16).
#include <type_traits>
#include <utility>
#include "product_tile.h"

namespace pico {
namespace {

struct LargeParams {
  const __bf16 *a, *b;
  void* c;            // bf16 [M, N], or fp32 [parts, M, N]
  int M, N, K;
  int64_t lda, ldb;   // elements between the rows of a and b as they lie in memory
  int tiles_m, tiles_n, parts;
  bool streaming;     // the output is written past the caches
};

__device__ __forceinline__ void wait_lds() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// A barrier in two halves, so that products go on between a wave's arrival and the point where it needs the others: a count in
// LDS, to which every wave adds one (with all 64 lanes on).
__device__ __forceinline__ void arrive(uint32_t count) {
  asm volatile("s_mov_b64 exec, 1\n\tds_add_u32 %0, %1\n\ts_mov_b64 exec, -1" ::"v"(count), "v"(1) : "memory");
}
__device__ __forceinline__ void wait_for(uint32_t count, int arrivals) {
  uint32_t v;
  int now;
  asm volatile("pico_wait_%=:\n\tds_read_b32 %0, %2\n\ts_waitcnt lgkmcnt(0)\n\tv_readfirstlane_b32 %1, %0\n\ts_cmp_lt_i32 %1, %3\n\ts_cbranch_scc1 pico_wait_%="
               : "=&v"(v), "=&s"(now) : "v"(count), "s"(arrivals) : "scc", "memory");
}

// What a workgroup works on in a round of the grid: a tile of the output and a run of steps.  The workgroups of a round go
// round the eight XCDs; each XCD takes a run of neighbouring tiles, eight tile rows deep, whose operands then meet in its L2.
struct Unit {
  int m0, n0, part, first, steps;   // (steps: first .. first + steps - 1)
};
template <int TM, int TN>
__device__ __forceinline__ bool unit_at(const LargeParams& p, int round, Unit& u) {
  const int tiles = p.tiles_m * p.tiles_n, grid = gridDim.x, start = round * grid, count = min(grid, tiles * p.parts - start);
  if (static_cast<int>(blockIdx.x) >= count) return false;
  const int xcd = blockIdx.x % 8, id = start + xcd * (count / 8) + min(xcd, count % 8) + blockIdx.x / 8;
  constexpr int kDeep = 8;
  u.part = id / tiles;
  const int t = id % tiles, block = t / (kDeep * p.tiles_n), in = t % (kDeep * p.tiles_n), deep = min(kDeep, p.tiles_m - block * kDeep);
  u.m0 = (block * kDeep + in % deep) * TM;
  u.n0 = in / deep * TN;
  const int steps = (p.K + kStep - 1) / kStep;
  u.first = static_cast<int>(static_cast<int64_t>(u.part) * steps / p.parts);
  u.steps = static_cast<int>(static_cast<int64_t>(u.part + 1) * steps / p.parts) - u.first;
  return true;
}

template <int... m, typename Fn>
__device__ __forceinline__ void each(std::integer_sequence<int, m...>, const Fn& fn) {
  (fn(std::integral_constant<int, m>()), ...);
}

// 2 x 4 waves of 16 I x 16 J
template <bool kSlowA, bool kSlowB, int I, int J>
struct Shape {
  static constexpr int kThreads = 512, TM = 32 * I, TN = 64 * J;
  using A = Tile<kSlowA, TM, kThreads>;
  using B = Tile<kSlowB, TN, kThreads>;
  static constexpr int kBuffer = A::kBytes + B::kBytes;
  static constexpr int kRowRegion = 16 * 128;   // per wave, where a tile's rows are put together
  static constexpr int kCounts = 2 * kBuffer + 8 * kRowRegion, kLds = kCounts + 16;
  static_assert(kLds <= 160 * 1024);
};

template <bool kSlowA, bool kSlowB, int I, int J, bool kParts>
__global__ __launch_bounds__(512, 2) void product_large_kernel(const LargeParams p) {
  using S = Shape<kSlowA, kSlowB, I, J>;
  using A = typename S::A;
  using B = typename S::B;
  constexpr int TM = S::TM, TN = S::TN, kPA = A::kPieces, kPB = B::kPieces, kPieces = kPA + kPB;
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
  const int tid = threadIdx.x, lane = tid % kWave, wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int wm = wave / 4 * 16 * I, wn = wave % 4 * 16 * J;

  // ---- requests
  uint32_t oa[kPA], ob[kPB];
#pragma unroll
  for (int i = 0; i < kPA; ++i) oa[i] = A::offset(p.lda, tid, i);
#pragma unroll
  for (int i = 0; i < kPB; ++i) ob[i] = B::offset(p.ldb, tid, i);
  const int k_piece = (tid % 8 ^ (tid / 16 & 7)) * 8;   // contraction index of this thread's pieces (fast axis)
  const bool ragged = p.K % kStep != 0;
  const uint32_t step_a = static_cast<uint32_t>(kSlowA ? kStep * p.lda * 2 : kStep * 2), step_b = static_cast<uint32_t>(kSlowB ? kStep * p.ldb * 2 : kStep * 2);
  Unit load;   // where the requests stand
  int load_round = 0, load_step = 0;
  unit_at<TM, TN>(p, 0, load);   // (the grid is no larger than the work)
  Window wa = open_window<kSlowA>(p.a, p.lda, load.m0, TM, p.M, load.first * kStep, p.K);
  Window wb = open_window<kSlowB>(p.b, p.ldb, load.n0, TN, p.N, load.first * kStep, p.K);
  u32x4 ra = resource(wa), rb = resource(wb);
  // to the next step, in four parts that are dealt out between products (the third, a tile's end, branches)
  auto go_on = [&](int part) __attribute__((always_inline)) {
    if (part == 0) {
      ++load_step;
      advance(wa, step_a);
    }
    if (part == 1) advance(wb, step_b);
    if (part == 2 && load_step >= load.steps - 1) {
      if (load_step == load.steps) {
        load_step = 0;
        const bool more = unit_at<TM, TN>(p, ++load_round, load);
        wa = open_window<kSlowA>(p.a, p.lda, load.m0, TM, p.M, load.first * kStep, p.K);
        wb = open_window<kSlowB>(p.b, p.ldb, load.n0, TN, p.N, load.first * kStep, p.K);
        if (!more) wa.bytes = wb.bytes = 0;   // requests past the work's end read no memory
      }
      if (ragged && !(kSlowA && kSlowB)) {   // pieces past the contraction's end read as zeros
        const bool in = k_piece < p.K - (load.first + load_step) * kStep;
#pragma unroll
        for (int i = 0; i < kPA; ++i) oa[i] = kSlowA || in ? A::offset(p.lda, tid, i) : 0xfffffff0u;
#pragma unroll
        for (int i = 0; i < kPB; ++i) ob[i] = kSlowB || in ? B::offset(p.ldb, tid, i) : 0xfffffff0u;
      }
    }
    if (part == 3) {
      ra = resource(wa);
      rb = resource(wb);
    }
  };
  const uint32_t lds_wave = wave * 1024;   // (dynamic LDS starts at 0: the build looks)
  auto aim = [&](auto piece, uint32_t buffer) __attribute__((always_inline)) {
    constexpr int i = decltype(piece)::value;
    return aim_request<(i < kPA ? i * S::kThreads * 16 : A::kBytes + (i - kPA) * S::kThreads * 16)>(lds_wave + buffer);
  };
  auto request = [&](auto piece, uint32_t aimed) __attribute__((always_inline)) {
    constexpr int i = decltype(piece)::value;
    if constexpr (i < kPA) request16(aimed, ra, oa[i]);
    else request16(aimed, rb, ob[i - kPA]);
  };

  // ---- half a step: its products, and behind each at most one other thing: a fragment of the half step that follows, a
  // request (the second half), or the way to the next step (the first half)
  constexpr int kFragments = I + J, kProducts = I * J;
  bf16x8 fa[2][I], fb[2][J];
  f32x4 acc[I][J];
  auto fetch = [&](const unsigned char* buffer, int s, int f) __attribute__((always_inline)) {
    if (f < J) fb[s][f < J ? f : 0] = B::fragment(buffer + A::kBytes, wn + 16 * f, s, lane);
    else fa[s][f < J ? 0 : f - J] = A::fragment(buffer, wm + 16 * (f - J), s, lane);
  };
  constexpr uint32_t kFree = S::kCounts, kThere = S::kCounts + 4;
  int arrivals = 0;   // that the waits of this step look for
  auto half_step = [&](auto half, const unsigned char* next, uint32_t free) __attribute__((always_inline)) {
    constexpr int s = decltype(half)::value;
    each(std::make_integer_sequence<int, kProducts>(), [&](auto product) __attribute__((always_inline)) {
      // Columns there and back, so that from each product to the next one of the operands stays (with all rows from left to right both change
      // at every row's end): the products of whole tiles run at the power limit, and an operand that does not change takes less.  us, one way and
      // there and back: [16384 x 4096] @ [4096 x 2048] transposed operands 200.9, 199.5; [4096 x 16384] @ [16384 x 2048] in two 195.6, 193.4; [8192 x 8192]
      // @ [8192 x 8192]^T 740.4, 734.2; 33 launches, 30 of them drawn, 0.984 to 1.002 of the time, 0.995 over all; where CUs idle, level.
      constexpr int m = decltype(product)::value, i = m / J, j = i % 2 ? J - 1 - m % J : m % J;
      // requests lie behind every second product (every one where there are few)
      constexpr int kGap = kProducts >= 32 ? 2 : 1, kPlaces = kProducts / kGap, place = m / kGap;
      constexpr bool here = s == 1 && m % kGap == kGap - 1;
      constexpr int first = here ? (place * kPieces + kPlaces - 1) / kPlaces : 0, last = here ? ((place + 1) * kPieces + kPlaces - 1) / kPlaces : 0;
      static_assert(last <= first + 1);
      using Piece = std::integral_constant<int, first>;
      [[maybe_unused]] uint32_t aimed = 0;
      if constexpr (last > first) aimed = aim(Piece(), free);
      __builtin_amdgcn_sched_barrier(0);
      acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[s][j], fa[s][i], acc[i][j], 0, 0, 0);   // C^T: a lane holds four columns of a row of C
      __builtin_amdgcn_sched_barrier(0);
      constexpr int kFrom = s == 0 ? 0 : kProducts * 10 / 32, kTo = s == 0 ? kProducts * 18 / 32 : kProducts;
      if constexpr (s == 1 && m == kFrom) wait_for(kThere, arrivals);
#pragma unroll
      for (int f = 0; f < kFragments; ++f)
        if (kFrom + f * (kTo - kFrom) / kFragments == m) fetch(next, 1 - s, f);
      if constexpr (s == 0 && m == kProducts * 24 / 32) {
        wait_lds();
        arrive(kFree);
      }
      if constexpr (last > first) request(Piece(), aimed);
      if constexpr (s == 0 && m % (kProducts / 4) == 1) go_on(m / (kProducts / 4));
      __builtin_amdgcn_sched_barrier(0);
    });
  };

  auto all_requests = [&](uint32_t buffer) __attribute__((always_inline)) {
    each(std::make_integer_sequence<int, kPieces>(), [&](auto piece) __attribute__((always_inline)) {
      const uint32_t aimed = aim(piece, buffer);
      asm volatile("s_nop 0");
      request(piece, aimed);
    });
  };
  all_requests(0);
#pragma unroll
  for (int i = 0; i < 4; ++i) go_on(i);
  all_requests(S::kBuffer);
  if (tid < 2) reinterpret_cast<uint32_t*>(lds + S::kCounts)[tid] = 0;
  wait_lds();
  wait_requests<kPieces>();
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
#pragma unroll
  for (int f = 0; f < kFragments; ++f) fetch(lds, 0, f);

  constexpr int kStores = I * (kParts ? (J + 1) / 2 : (J + 3) / 4) * 2;   // of a wave, at a tile's end
  unsigned char* rows = lds + 2 * S::kBuffer + wave * S::kRowRegion;
  uint32_t now = 0;   // the buffer of this step
  Unit u;
  for (int round = 0; unit_at<TM, TN>(p, round, u); ++round) {
#pragma unroll
    for (int i = 0; i < I; ++i)
#pragma unroll
      for (int j = 0; j < J; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int t = 0; t < u.steps; ++t) {
      const uint32_t then = S::kBuffer - now;
      arrivals += 8;
      __builtin_amdgcn_s_setprio(0);
      half_step(std::integral_constant<int, 0>(), lds + now, 0);
      // `then` is there: everything requested but the stores of the tile before, which were issued behind its requests
      if (t == 0 && round > 0) wait_requests<kStores>();
      else wait_requests<0>();
      arrive(kThere);
      wait_for(kFree, arrivals);
      __builtin_amdgcn_s_setprio(1);   // (1 - 2 %)
      half_step(std::integral_constant<int, 1>(), lds + then, now);   // (requests the step after the next into `now`)
      now = then;
    }
    // ---- the tile leaves, 16 rows and 128 bytes of columns at a time through LDS, as whole lines; what lies past the matrix is
    // dropped by the window.  No wave waits for another here, and the next tile's first steps are on their way.
    using Out = std::conditional_t<kParts, float, __bf16>;
    constexpr int kBlocks = kParts ? 2 : 4;   // of 16 columns in 128 bytes
    const int row0 = u.m0 + wm, col0 = u.n0 + wn, cols = p.N - col0, n = lane % 16, h = lane / 16;
    Out* base = static_cast<Out*>(p.c) + (static_cast<int64_t>(u.part) * p.M + row0) * p.N + col0;
    const uint32_t pitch = static_cast<uint32_t>(p.N) * sizeof(Out), back = lane / 8 * pitch + lane % 8 * 16;
#pragma unroll
    for (int i = 0; i < I; ++i) {
      const int live = min(16, p.M - row0 - 16 * i);
      const u32x4 r = resource({reinterpret_cast<uint64_t>(base + static_cast<int64_t>(16 * i) * p.N),
                                live > 0 && cols > 0 ? static_cast<uint32_t>(((live - 1) * static_cast<int64_t>(p.N) + cols) * sizeof(Out)) : 0u});
      const buffer_rsrc window = __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(r[0] | static_cast<uint64_t>(r[1]) << 32), 0, static_cast<int>(r[2]), static_cast<int>(r[3]));
#pragma unroll
      for (int j0 = 0; j0 < J; j0 += kBlocks) {
#pragma unroll
        for (int j = 0; j < J; ++j) {
          if (j < j0 || j >= j0 + kBlocks) continue;
          unsigned char* to = rows + n * 128;
          if constexpr (kParts) {
            *reinterpret_cast<f32x4*>(to + (((j - j0) * 4 + h) ^ (n / 2)) * 16) = acc[i][j];
          } else {
            bf16x4 v;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = static_cast<__bf16>(acc[i][j][e]);
            *reinterpret_cast<bf16x4*>(to + (((j - j0) * 2 + h / 2) ^ (n / 2)) * 16 + h % 2 * 8) = v;
          }
        }
        const int here = min(kBlocks, J - j0) * 16, col = lane % 8 * (16 / static_cast<int>(sizeof(Out)));
        const bool in = col < here && 16 * j0 + col < cols;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const int row = 8 * q + lane / 8;
          const u32x4 v = *reinterpret_cast<const u32x4*>(rows + row * 128 + ((lane % 8) ^ (row / 2)) * 16);
          const int to = in ? static_cast<int>(back + 8 * q * pitch + 16 * j0 * sizeof(Out)) : static_cast<int>(0xfffffff0u);
          constexpr int kStreaming = 2;
          if (p.streaming) __builtin_amdgcn_raw_buffer_store_b128(v, window, to, 0, kStreaming);
          else __builtin_amdgcn_raw_buffer_store_b128(v, window, to, 0, 0);
        }
      }
    }
  }
  wait_requests<0>();   // (requests past the work's end still write zeros to LDS)
}

template <bool kSlowA, bool kSlowB, int I, int J, bool kParts>
int launch(LargeParams p, hipStream_t s) {
  using S = Shape<kSlowA, kSlowB, I, J>;
  static LdsOnce reserved;
  if (!reserve_lds_once(reserved, reinterpret_cast<const void*>(&product_large_kernel<kSlowA, kSlowB, I, J, kParts>), S::kLds))
    return fail(PICO_ERR_LAUNCH, "pico_product_large: cannot reserve %d bytes of LDS", S::kLds);
  p.tiles_m = (p.M + S::TM - 1) / S::TM;
  p.tiles_n = (p.N + S::TN - 1) / S::TN;
  const int64_t units = static_cast<int64_t>(p.tiles_m) * p.tiles_n * p.parts;
  // An output larger than the workgroups' one round of tiles would push the operands out of the caches as it is written: [4096 x
  // 2048] @ [49152 x 2048]^T 638 -> 570 us, [4096 x 1024] @ [49152 x 1024]^T 358 -> 304.
  p.streaming = !kParts && units > 256;
  hipLaunchKernelGGL((product_large_kernel<kSlowA, kSlowB, I, J, kParts>), dim3(static_cast<unsigned>(std::min<int64_t>(units, 256))), dim3(S::kThreads), S::kLds, s, p);
  return check_launch("pico_product_large");
}
template <bool kSlowA, bool kSlowB, bool kParts>
int launch_shape(const LargeParams& p, int tile_m, int tile_n, hipStream_t s) {
  if (tile_m == 256 && tile_n == 256) return launch<kSlowA, kSlowB, 8, 4, kParts>(p, s);
  if (tile_m == 256 && tile_n == 192) return launch<kSlowA, kSlowB, 8, 3, kParts>(p, s);
  if (tile_m == 192 && tile_n == 256) return launch<kSlowA, kSlowB, 6, 4, kParts>(p, s);
  if (tile_m == 256 && tile_n == 128) return launch<kSlowA, kSlowB, 8, 2, kParts>(p, s);
  if (tile_m == 128 && tile_n == 256) return launch<kSlowA, kSlowB, 4, 4, kParts>(p, s);
  return fail(PICO_ERR_SHAPE, "pico_product_large: tiles of %d x %d (256 x 256, or one side 192 or 128)", tile_m, tile_n);
}

}  // namespace
}  // namespace pico

using namespace pico;

extern "C" int pico_product_large_takes(int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int a_slow, int b_slow, int parts) {
  constexpr int64_t kMost = 0x7fffffff;
  // (two steps per piece at least: the kernel requests one step ahead of the tile it works on)
  if (M < 1 || N < 1 || M > kMost / 2 || N > kMost / 256 || K > kMost - 4096 || N % 8 != 0 || (a_slow ? M : K) % 8 != 0 || (b_slow ? N : K) % 8 != 0 ||
      lda % 8 != 0 || ldb % 8 != 0 || lda < (a_slow ? M : K) || ldb < (b_slow ? N : K) || (a_slow && !b_slow) || parts < 1 || parts > 64 ||
      (K + kStep - 1) / kStep < 2 * parts)
    return 0;
  // the windows of the buffer loads: a tile's rows, or the whole contraction where that is the slow axis
  if (lda > kMost / 2 || ldb > kMost / 2 || ((a_slow ? K + kStep : 256) * lda + K) * 2 > kMost || ((b_slow ? K + kStep : 256) * ldb + K) * 2 > kMost)
    return 0;
  return ((M + 127) / 128) * ((N + 127) / 128) * parts <= kMost / 256;
}

extern "C" int pico_product_large(const void* a, const void* b, void* c, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int a_slow,
                                  int b_slow, int tile_m, int tile_n, int parts, void* stream) {
  if (!pico_product_large_takes(M, N, K, lda, ldb, a_slow, b_slow, parts))
    return fail(PICO_ERR_SHAPE, "pico_product_large: M=%lld N=%lld K=%lld row pitches %lld, %lld, %d pieces (rows of a, b and c and the pitches must be multiples of 8 elements, two steps of 64 per piece, a tile's rows span less than 2 GiB, no a^T b^T)",
                (long long)M, (long long)N, (long long)K, (long long)lda, (long long)ldb, parts);
  if (!a || !b || !c) return fail(PICO_ERR_NULL, "pico_product_large: a, b and c are required");
  if (!aligned16(a) || !aligned16(b) || !aligned16(c)) return fail(PICO_ERR_ALIGN, "pico_product_large: pointers must be 16-byte aligned");
  const LargeParams p = {static_cast<const __bf16*>(a), static_cast<const __bf16*>(b), c, (int)M, (int)N, (int)K, lda, ldb, 0, 0, parts, false};
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (a_slow) return parts > 1 ? launch_shape<true, true, true>(p, tile_m, tile_n, s) : launch_shape<true, true, false>(p, tile_m, tile_n, s);
  if (b_slow) return parts > 1 ? launch_shape<false, true, true>(p, tile_m, tile_n, s) : launch_shape<false, true, false>(p, tile_m, tile_n, s);
  return parts > 1 ? launch_shape<false, false, true>(p, tile_m, tile_n, s) : launch_shape<false, false, false>(p, tile_m, tile_n, s);
}
