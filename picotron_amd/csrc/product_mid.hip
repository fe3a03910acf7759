// Matrix products between the smallest ones and those that fill the GPU many times over: C = op(A) op(B) in bf16 with fp32
// accumulation, in any of the three layouts of a linear layer, one tile of the output per workgroup.
//
// What bounds them is what one CU moves: a tile's operands come from L2 at 64 bytes a clock, and LDS takes them and gives
// them out again.  So the tile is chosen for each product such that one round of workgroups fills the GPU (32 x 32 .. 128 x 256);
// operands go to LDS without passing the registers, as many steps ahead as LDS holds; and the steps of the contraction are dealt to
// groups of waves inside the workgroup, 2 x 2 waves each (or two), because every wave of a group's row or column reads the same
// fragments: the reads are twice what the requests write then, three times with 2 x 4 waves.  Bytes a nanosecond and CU,
// by tiles at 72 .. 222 workgroups: 72 .. 97; 110 .. 135 with the requests alone.
//   [512 x 3072] @ [3072 x 576]: 12.9 us in tiles of 64 through registers, 12.0 in tiles of 64 here, 8.7 in 144 tiles of 32 x 64;
//   [2331 x 1536] @ [576 x 1536]^T: 12.0 in the GEMM library, 9.5 in 222 tiles of 64 x 96; [2331 x 3072] @ [3072 x 576] 27.7, 15.4;
//   [2331 x 3072]^T [2331 x 576]: 23.7 in tiles of 128, 15.3 in 240 tiles of 64 x 128.
// Fragments read a trip ahead into a second set of registers change nothing (9.8 and 10.0 us at the second size).  Two waves per
// group and four groups: 32 x 64 10.0 -> 8.7 at the first size, larger tiles lose (the ring holds two steps).
#include "product_tile.h"

namespace pico {
namespace {

struct MidParams {
  const __bf16 *a, *b;
  void* c;            // bf16 [M, N], or fp32 [parts, M, N]
  int M, N, K;
  int64_t lda, ldb;   // elements between the rows of a and b as they lie in memory
  int tiles_m, tiles_n, parts;
};

// Eight waves: KS groups deal the steps of the contraction between them, and the WM x WN waves of a group take 16 I x 16 J of the
// tile each.
template <bool kSlowA, bool kSlowB, int I, int J, int WM, int WN>
struct Form {
  static constexpr int KS = 8 / (WM * WN), kGroup = 64 * WM * WN, TM = 16 * I * WM, TN = 16 * J * WN;
  using A = Tile<kSlowA, TM, kGroup>;
  using B = Tile<kSlowB, TN, kGroup>;
  static constexpr int kStage = A::kBytes + B::kBytes;   // a group's step
  static constexpr int kFit = 156 * 1024 / (KS * kStage), kRing = kFit > 6 ? 6 : kFit;
  static_assert(kRing >= 2);
  static constexpr int kOutPitch = TN + 8, kSums = (KS - 1) * I * J * 1024 * WM * WN, kEnd = kSums + TM * kOutPitch * 2;
  static constexpr int kLds = kRing * KS * kStage > kEnd ? kRing * KS * kStage : kEnd;
  static_assert(kLds <= 160 * 1024);
};

template <bool kSlowA, bool kSlowB, int I, int J, int WM, int WN, bool kParts = false>
__device__ __forceinline__ void mid_tile(const MidParams& p, int block) {
  using F = Form<kSlowA, kSlowB, I, J, WM, WN>;
  using A = typename F::A;
  using B = typename F::B;
  constexpr int TM = F::TM, TN = F::TN, KS = F::KS, kPA = A::kPieces, kPB = B::kPieces, kPieces = kPA + kPB, kRing = F::kRing;
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
  const int tid = threadIdx.x, lane = tid % kWave, wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int group = wave / (WM * WN), in_group = wave % (WM * WN), gtid = in_group * kWave + lane;
  const int wm = in_group / WN * 16 * I, wn = in_group % WN * 16 * J;
  // workgroups go round the eight XCDs: each takes a run of neighbouring tiles, along the shorter side of the output
  const int tiles = p.tiles_m * p.tiles_n, units = kParts ? tiles * p.parts : tiles, xcd = block % 8;
  const int unit = xcd * (units / 8) + min(xcd, units % 8) + block / 8, part = kParts ? unit / tiles : 0, id = kParts ? unit % tiles : unit;
  const bool down = p.tiles_m < p.tiles_n;
  const int m0 = (down ? id % p.tiles_m : id / p.tiles_n) * TM, n0 = (down ? id / p.tiles_m : id % p.tiles_n) * TN;

  // ---- requests: the group's steps are group, group + KS, ...
  const int all = (p.K + kStep - 1) / kStep, from = kParts ? static_cast<int>(static_cast<int64_t>(part) * all / p.parts) : 0;
  const int steps = kParts ? static_cast<int>(static_cast<int64_t>(part + 1) * all / p.parts) - from : all, trips = (steps + KS - 1) / KS;   // (one at least)
  uint32_t oa[kPA], ob[kPB];
#pragma unroll
  for (int i = 0; i < kPA; ++i) oa[i] = A::offset(p.lda, gtid, i);
#pragma unroll
  for (int i = 0; i < kPB; ++i) ob[i] = B::offset(p.ldb, gtid, i);
  const uint32_t step_a = static_cast<uint32_t>(KS * (kSlowA ? kStep * p.lda * 2 : kStep * 2)), step_b = static_cast<uint32_t>(KS * (kSlowB ? kStep * p.ldb * 2 : kStep * 2));
  const int first = min(group, steps - 1);   // (a group without steps requests nothing)
  Window wa = open_window<kSlowA>(p.a, p.lda, m0, TM, p.M, (from + first) * kStep, p.K);
  Window wb = open_window<kSlowB>(p.b, p.ldb, n0, TN, p.N, (from + first) * kStep, p.K);
  int load = group;   // the step that is requested next
  const int k_piece = (gtid % 8 ^ (gtid / 16 & 7)) * 8, k_last = p.K - (from + steps - 1) * kStep;   // (a part that ends before the contraction does has whole steps)
  auto request_step = [&](uint32_t to) __attribute__((always_inline)) {
    if (load >= steps) wa.bytes = wb.bytes = 0;   // requests past the contraction's end read no memory
    if constexpr (!(kSlowA && kSlowB)) {
      if (load == steps - 1 && k_last < kStep) {   // pieces past the contraction's end read as zeros
        const bool in = k_piece < k_last;
#pragma unroll
        for (int i = 0; i < kPA; ++i) oa[i] = kSlowA || in ? oa[i] : 0xfffffff0u;
#pragma unroll
        for (int i = 0; i < kPB; ++i) ob[i] = kSlowB || in ? ob[i] : 0xfffffff0u;
      }
    }
    const u32x4 ra = resource(wa), rb = resource(wb);
    const uint32_t at = to + in_group * 1024;   // (dynamic LDS starts at 0: the build looks)
    each_load<kPA>([&](auto piece) {
      constexpr int i = decltype(piece)::value;
      request16_to<i * F::kGroup * 16>(at, ra, oa[i]);
    });
    each_load<kPB>([&](auto piece) {
      constexpr int i = decltype(piece)::value;
      request16_to<A::kBytes + i * F::kGroup * 16>(at, rb, ob[i]);
    });
    load += KS;
    advance(wa, step_a);
    advance(wb, step_b);
  };
  const uint32_t mine = group * F::kStage;
#pragma unroll
  for (int t = 0; t < kRing - 1; ++t) request_step(t * KS * F::kStage + mine);

  f32x4 acc[I][J];
#pragma unroll
  for (int i = 0; i < I; ++i)
#pragma unroll
    for (int j = 0; j < J; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  uint32_t now = mine, free = (kRing - 1) * KS * F::kStage + mine;
  for (int t = 0; t < trips; ++t) {
    wait_requests<(kRing - 2) * kPieces>();   // this trip's step is there
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();             // ... everybody's, and nobody reads the step before any more
    asm volatile("" ::: "memory");
    request_step(free);
    free = now;
    const unsigned char* ta = lds + now;
    const unsigned char* tb = ta + A::kBytes;
    bf16x8 fa[2][I], fb[2][J];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
#pragma unroll
      for (int j = 0; j < J; ++j) fb[s][j] = B::fragment(tb, wn + 16 * j, s, lane);
#pragma unroll
      for (int i = 0; i < I; ++i) fa[s][i] = A::fragment(ta, wm + 16 * i, s, lane);
    }
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int i = 0; i < I; ++i)
#pragma unroll
        for (int j = 0; j < J; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[s][j], fa[s][i], acc[i][j], 0, 0, 0);   // C^T: a lane holds four columns of a row of C
    now += KS * F::kStage;
    if (now >= kRing * KS * F::kStage) now -= kRing * KS * F::kStage;
  }
  wait_requests<0>();   // (also those past the end write LDS)
  __syncthreads();

  // ---- the groups' sums, in the order of the groups
  if constexpr (KS > 1) {
    auto place = [&](int g, int i, int j) { return reinterpret_cast<f32x4*>(lds) + (((g - 1) * WM * WN + in_group) * I * J + i * J + j) * kWave + lane; };
    if (group > 0) {
#pragma unroll
      for (int i = 0; i < I; ++i)
#pragma unroll
        for (int j = 0; j < J; ++j) *place(group, i, j) = acc[i][j];
    }
    __syncthreads();
    if (group == 0) {
#pragma unroll
      for (int g = 1; g < KS; ++g)
#pragma unroll
        for (int i = 0; i < I; ++i)
#pragma unroll
          for (int j = 0; j < J; ++j) acc[i][j] += *place(g, i, j);
    }
  }
  if constexpr (kParts) {   // a lane's four columns at a time
    if (group == 0) {
      float* c = static_cast<float*>(p.c) + static_cast<int64_t>(part) * p.M * p.N;
#pragma unroll
      for (int i = 0; i < I; ++i) {
        const int row = m0 + wm + 16 * i + lane % 16;
#pragma unroll
        for (int j = 0; j < J; ++j) {
          const int col = n0 + wn + 16 * j + 4 * (lane / 16);
          if (row < p.M && col < p.N) *reinterpret_cast<f32x4*>(c + static_cast<int64_t>(row) * p.N + col) = acc[i][j];
        }
      }
    }
    return;
  }
  // ---- the tile leaves through LDS as whole lines (behind the groups' sums, which may still be read)
  unsigned char* out = lds + F::kSums;
  if (group == 0) {
    const int n = lane % 16, h = lane / 16;
#pragma unroll
    for (int i = 0; i < I; ++i)
#pragma unroll
      for (int j = 0; j < J; ++j) {
        bf16x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = static_cast<__bf16>(acc[i][j][e]);
        *reinterpret_cast<bf16x4*>(out + ((wm + 16 * i + n) * F::kOutPitch + wn + 16 * j + 4 * h) * 2) = v;
      }
  }
  __syncthreads();
  for (int idx = tid; idx < TM * TN / 8; idx += 512) {
    const int r = idx / (TN / 8), cv = idx % (TN / 8);
    if (m0 + r < p.M && n0 + cv * 8 < p.N)
      *reinterpret_cast<u32x4*>(static_cast<__bf16*>(p.c) + static_cast<int64_t>(m0 + r) * p.N + n0 + cv * 8) = *reinterpret_cast<const u32x4*>(out + r * F::kOutPitch * 2 + cv * 16);
  }
}

template <bool kSlowA, bool kSlowB, int I, int J, int WM, int WN, bool kParts>
__global__ __launch_bounds__(512, 2) void product_mid_kernel(const MidParams p) {
  mid_tile<kSlowA, kSlowB, I, J, WM, WN, kParts>(p, blockIdx.x);
}

template <bool kSlowA, bool kSlowB, int I, int J, int WM, int WN, bool kParts = false>
int launch(MidParams p, hipStream_t s) {
  using F = Form<kSlowA, kSlowB, I, J, WM, WN>;
  p.tiles_m = (p.M + F::TM - 1) / F::TM;
  p.tiles_n = (p.N + F::TN - 1) / F::TN;
  static LdsOnce reserved;
  if (!reserve_lds_once(reserved, reinterpret_cast<const void*>(&product_mid_kernel<kSlowA, kSlowB, I, J, WM, WN, kParts>), F::kLds))
    return fail(PICO_ERR_LAUNCH, "pico_product_mid: cannot reserve %d bytes of LDS", F::kLds);
  hipLaunchKernelGGL((product_mid_kernel<kSlowA, kSlowB, I, J, WM, WN, kParts>), dim3(static_cast<unsigned>(p.tiles_m) * p.tiles_n * (kParts ? p.parts : 1)), dim3(512), F::kLds, s, p);
  return check_launch("pico_product_mid");
}
template <bool kSlowA, bool kSlowB>
int launch_form(const MidParams& p, int tm, int tn, hipStream_t s) {
  switch (tm << 16 | tn) {
    case 32 << 16 | 32: return launch<kSlowA, kSlowB, 2, 1, 1, 2>(p, s);
    case 32 << 16 | 64: return launch<kSlowA, kSlowB, 2, 2, 1, 2>(p, s);
    case 64 << 16 | 32: return launch<kSlowA, kSlowB, 2, 2, 2, 1>(p, s);
    case 64 << 16 | 64: return launch<kSlowA, kSlowB, 2, 2, 2, 2>(p, s);
    case 64 << 16 | 96: return launch<kSlowA, kSlowB, 2, 3, 2, 2>(p, s);
    case 96 << 16 | 64: return launch<kSlowA, kSlowB, 3, 2, 2, 2>(p, s);
    case 96 << 16 | 96: return launch<kSlowA, kSlowB, 3, 3, 2, 2>(p, s);
    case 64 << 16 | 128: return launch<kSlowA, kSlowB, 2, 4, 2, 2>(p, s);
    case 128 << 16 | 64: return launch<kSlowA, kSlowB, 4, 2, 2, 2>(p, s);
    case 128 << 16 | 96: return launch<kSlowA, kSlowB, 4, 3, 2, 2>(p, s);
    case 128 << 16 | 128: return launch<kSlowA, kSlowB, 4, 4, 2, 2>(p, s);
    case 128 << 16 | 192: return launch<kSlowA, kSlowB, 4, 3, 2, 4>(p, s);
    case 192 << 16 | 128: return launch<kSlowA, kSlowB, 6, 2, 2, 4>(p, s);
    case 128 << 16 | 256: return launch<kSlowA, kSlowB, 4, 4, 2, 4>(p, s);
    default: return fail(PICO_ERR_SHAPE, "pico_product_mid: no tiles of %d x %d", tm, tn);
  }
}

// The contraction in parts, as fp32 pieces: few tiles and a long contraction, where one round of workgroups takes
// pieces of tiles ([1063 x 8192] @ [8192 x 192] 20.7 -> 14.3 us, [726 x 8192] @ [8192 x 1024] 29.8 -> 24.8).
template <bool kSlowA, bool kSlowB>
int launch_parts(const MidParams& p, int tm, int tn, hipStream_t s) {
  switch (tm << 16 | tn) {
    case 64 << 16 | 96: return launch<kSlowA, kSlowB, 2, 3, 2, 2, true>(p, s);
    case 64 << 16 | 128: return launch<kSlowA, kSlowB, 2, 4, 2, 2, true>(p, s);
    case 96 << 16 | 96: return launch<kSlowA, kSlowB, 3, 3, 2, 2, true>(p, s);
    case 128 << 16 | 128: return launch<kSlowA, kSlowB, 4, 4, 2, 2, true>(p, s);
    case 128 << 16 | 192: return launch<kSlowA, kSlowB, 4, 3, 2, 4, true>(p, s);
    case 192 << 16 | 128: return launch<kSlowA, kSlowB, 6, 2, 2, 4, true>(p, s);
    case 128 << 16 | 256: return launch<kSlowA, kSlowB, 4, 4, 2, 4, true>(p, s);
    default: return fail(PICO_ERR_SHAPE, "pico_product_mid: no tiles of %d x %d in parts", tm, tn);
  }
}

// Both gradients of a linear layer in one launch, dX = dY W and dW = dY^T X.  Each alone leaves CUs idle and pays a launch of its own:
// [512 x 576] and [576 x 576] take 4.3 and 4.2 us alone, 5.2 together; [2331 x 576] and [576 x 576] 15.5, 11.2.  The tiles of both
// are chosen together, one workgroup per CU at a time, the longer walks first.
struct MidPairParams {
  MidParams dx, dw;
  int blocks_first;   // of the product that comes first, rounded up to whole rounds of the XCDs
  bool dw_first;
};
struct Tiles32x64 {
  static constexpr int TM = 32, TN = 64, I = 2, J = 2, WM = 1, WN = 2;
};
struct Tiles64x64 {
  static constexpr int TM = 64, TN = 64, I = 2, J = 2, WM = 2, WN = 2;
};
struct Tiles64x96 {
  static constexpr int TM = 64, TN = 96, I = 2, J = 3, WM = 2, WN = 2;
};
struct Tiles64x128 {
  static constexpr int TM = 64, TN = 128, I = 2, J = 4, WM = 2, WN = 2;
};
template <typename X, typename W>
__global__ __launch_bounds__(512, 2) void product_pair_kernel(const MidPairParams p) {
  const int block = blockIdx.x, rest = block - p.blocks_first, at = rest < 0 ? block : rest;
  if ((rest < 0) == p.dw_first) {
    if (at < p.dw.tiles_m * p.dw.tiles_n) mid_tile<true, true, W::I, W::J, W::WM, W::WN>(p.dw, at);
  } else {
    if (at < p.dx.tiles_m * p.dx.tiles_n) mid_tile<false, true, X::I, X::J, X::WM, X::WN>(p.dx, at);
  }
}
template <typename X, typename W>
int launch_pair(MidPairParams p, hipStream_t s) {
  constexpr int kDx = Form<false, true, X::I, X::J, X::WM, X::WN>::kLds, kDw = Form<true, true, W::I, W::J, W::WM, W::WN>::kLds, kLds = kDx > kDw ? kDx : kDw;
  p.dx.tiles_m = (p.dx.M + X::TM - 1) / X::TM;
  p.dx.tiles_n = (p.dx.N + X::TN - 1) / X::TN;
  p.dw.tiles_m = (p.dw.M + W::TM - 1) / W::TM;
  p.dw.tiles_n = (p.dw.N + W::TN - 1) / W::TN;
  const int dx = p.dx.tiles_m * p.dx.tiles_n, dw = p.dw.tiles_m * p.dw.tiles_n;
  p.blocks_first = ((p.dw_first ? dw : dx) + 7) / 8 * 8;
  static LdsOnce reserved;
  if (!reserve_lds_once(reserved, reinterpret_cast<const void*>(&product_pair_kernel<X, W>), kLds))
    return fail(PICO_ERR_LAUNCH, "pico_product_pair: cannot reserve %d bytes of LDS", kLds);
  hipLaunchKernelGGL((product_pair_kernel<X, W>), dim3(static_cast<unsigned>(p.blocks_first + (p.dw_first ? dx : dw))), dim3(512), kLds, s, p);
  return check_launch("pico_product_pair");
}
template <typename X>
int launch_pair_w(const MidPairParams& p, int tm, int tn, hipStream_t s) {
  switch (tm << 16 | tn) {
    case 32 << 16 | 64: return launch_pair<X, Tiles32x64>(p, s);
    case 64 << 16 | 64: return launch_pair<X, Tiles64x64>(p, s);
    case 64 << 16 | 96: return launch_pair<X, Tiles64x96>(p, s);
    case 64 << 16 | 128: return launch_pair<X, Tiles64x128>(p, s);
    default: return fail(PICO_ERR_SHAPE, "pico_product_pair: no tiles of %d x %d for dw", tm, tn);
  }
}

}  // namespace
}  // namespace pico

using namespace pico;

extern "C" int pico_product_mid_takes(int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int a_slow, int b_slow) {
  constexpr int64_t kMost = 0x7fffffff;
  if (M < 1 || N < 1 || K < 1 || M > kMost / 2 || N > kMost / 256 || K > kMost - 4096 || N % 8 != 0 || (a_slow ? M : K) % 8 != 0 || (b_slow ? N : K) % 8 != 0 ||
      lda % 8 != 0 || ldb % 8 != 0 || lda < (a_slow ? M : K) || ldb < (b_slow ? N : K) || (a_slow && !b_slow))
    return 0;
  // the windows of the buffer loads: a tile's rows, or the whole contraction where that is the slow axis
  if (lda > kMost / 2 || ldb > kMost / 2 || ((a_slow ? K + kStep : 256) * lda + K) * 2 > kMost || ((b_slow ? K + kStep : 256) * ldb + K) * 2 > kMost)
    return 0;
  return ((M + 31) / 32) * ((N + 31) / 32) <= kMost / 256;
}

extern "C" int pico_product_mid(const void* a, const void* b, void* c, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int a_slow,
                                int b_slow, int tile_m, int tile_n, int parts, void* stream) {
  if (!pico_product_mid_takes(M, N, K, lda, ldb, a_slow, b_slow))
    return fail(PICO_ERR_SHAPE, "pico_product_mid: M=%lld N=%lld K=%lld row pitches %lld, %lld (rows of a, b and c and the pitches must be multiples of 8 elements, a tile's rows span less than 2 GiB, no a^T b^T)",
                (long long)M, (long long)N, (long long)K, (long long)lda, (long long)ldb);
  if (!a || !b || !c) return fail(PICO_ERR_NULL, "pico_product_mid: a, b and c are required");
  if (!aligned16(a) || !aligned16(b) || !aligned16(c)) return fail(PICO_ERR_ALIGN, "pico_product_mid: pointers must be 16-byte aligned");
  const MidParams p = {static_cast<const __bf16*>(a), static_cast<const __bf16*>(b), c, (int)M, (int)N, (int)K, lda, ldb, 0, 0, parts};
  if (parts < 1 || parts > 64 || (K + kStep - 1) / kStep < parts)
    return fail(PICO_ERR_SHAPE, "pico_product_mid: %d parts (1 .. 64, a step of 64 each)", parts);
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (parts > 1)
    return a_slow ? launch_parts<true, true>(p, tile_m, tile_n, s) : b_slow ? launch_parts<false, true>(p, tile_m, tile_n, s) : launch_parts<false, false>(p, tile_m, tile_n, s);
  if (a_slow) return launch_form<true, true>(p, tile_m, tile_n, s);
  return b_slow ? launch_form<false, true>(p, tile_m, tile_n, s) : launch_form<false, false>(p, tile_m, tile_n, s);
}

extern "C" int pico_product_pair(const void* dy, const void* w, const void* x, void* dx, void* dw, int64_t rows, int64_t out, int64_t in,
                                 int64_t ld_dy, int64_t ld_w, int64_t ld_x, int dx_tile_m, int dx_tile_n, int dw_tile_m, int dw_tile_n, void* stream) {
  if (!pico_product_mid_takes(rows, in, out, ld_dy, ld_w, 0, 1) || !pico_product_mid_takes(out, in, rows, ld_dy, ld_x, 1, 1))
    return fail(PICO_ERR_SHAPE, "pico_product_pair: rows=%lld out=%lld in=%lld row pitches %lld, %lld, %lld (out, in and the pitches must be multiples of 8 elements, a tile's rows span less than 2 GiB)",
                (long long)rows, (long long)out, (long long)in, (long long)ld_dy, (long long)ld_w, (long long)ld_x);
  if (!dy || !w || !x || !dx || !dw) return fail(PICO_ERR_NULL, "pico_product_pair: dy, w, x, dx and dw are required");
  if (!aligned16(dy) || !aligned16(w) || !aligned16(x) || !aligned16(dx) || !aligned16(dw)) return fail(PICO_ERR_ALIGN, "pico_product_pair: pointers must be 16-byte aligned");
  MidPairParams p;
  p.dx = {static_cast<const __bf16*>(dy), static_cast<const __bf16*>(w), dx, (int)rows, (int)in, (int)out, ld_dy, ld_w, 0, 0, 1};
  p.dw = {static_cast<const __bf16*>(dy), static_cast<const __bf16*>(x), dw, (int)out, (int)in, (int)rows, ld_dy, ld_x, 0, 0, 1};
  p.dw_first = rows > out;   // the longer walks start first
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (dx_tile_m << 16 | dx_tile_n) {
    case 32 << 16 | 64: return launch_pair_w<Tiles32x64>(p, dw_tile_m, dw_tile_n, s);
    case 64 << 16 | 64: return launch_pair_w<Tiles64x64>(p, dw_tile_m, dw_tile_n, s);
    case 64 << 16 | 96: return launch_pair_w<Tiles64x96>(p, dw_tile_m, dw_tile_n, s);
    case 64 << 16 | 128: return launch_pair_w<Tiles64x128>(p, dw_tile_m, dw_tile_n, s);
    default: return fail(PICO_ERR_SHAPE, "pico_product_pair: no tiles of %d x %d for dx", dx_tile_m, dx_tile_n);
  }
}
