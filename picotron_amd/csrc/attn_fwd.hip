// Flash-style attention forward for gfx950: S^T = K Q^T and O^T = V^T P^T on MFMA 32x32x16 bf16.
//
// Computing the TRANSPOSED score tile puts one query in each lane (column n of the C tile) and
// the keys in its registers, so the online-softmax max/sum are in-register reductions plus one
// exchange between the two wave halves, the per-query rescale factor is a per-lane scalar for the
// O^T accumulator, and the probabilities can be fed to the second MFMA as its B operand without
// leaving registers.  K and V tiles are staged row-major in LDS once per workgroup; K is read with
// 16-byte loads, V with transposing LDS reads (the contraction index of P V is V's row).
//
// The loop is bound by issue slots: per 32 x 64 tile of scores the softmax's vector instructions take about as long as the
// products.  The tiles are therefore loaded by requests that write LDS themselves: through registers they cost
// 2 x KT D / 8 / threads LDS writes with their waits at the end of every trip, and as many registers of 16 bytes (B1 H32 S4096
// D128 147 -> 142 us, H32/8 S8192 524 -> 507; level at head_dim 64, where one register per tensor and trip was enough).
#include "attn_common.h"

namespace pico {
namespace {

struct FwdParams {
  AttnParams a;
  void* out;
  float* lse;
  int out_f32;
  int merge;
  int pair_order;  // dispatch order of the query tiles, see the kernel
  RopeArgs rope;   // rope.cos != nullptr: q arrives un-rotated and is rotated in the prologue (k is rotated already)
  __bf16* q_rot;   // ... and, if given, the rotated q is written here for the backward
  int64_t qrs[3];  // element strides (b, h, s) of q_rot
};

// KS > 1 splits the keys of a staged tile over KS waves that share the same queries (NW / KS waves cover the queries):
// for launches with about one wave per SIMD, where a wave's S -> softmax -> PV chain per key tile is not hidden by
// anything, this multiplies the waves in flight and divides each chain's length by KS.  The KS partial (m, l, O)
// states of a query meet in LDS at the end.
template <int D, int QB, int NW, int KT, int KS = 1>
struct FwdCfg {
  static constexpr int kThreads = 64 * NW;
  static constexpr int kQWaves = NW / KS;        // waves that cover different queries
  static constexpr int BM = 32 * QB * kQWaves;   // queries per workgroup
  static_assert(NW % KS == 0 && (KS == 1 || KT == 64 * KS), "one 64-key step of every staged tile per key-split wave");
  static_assert(KS == 1 || QB == 1, "key split is built for one query block per wave");
  static constexpr int BN = 64;            // keys per compute step
  static constexpr int kKT = KT;           // keys per staged LDS tile (a multiple of BN), double-buffered
  static constexpr int kKDepth = D >= 128 ? 2 : 0;  // K fragments in flight from LDS ahead of the MFMA that uses them (0: compiler's order)
  static constexpr int kVecPerRow = D / 8;
  static constexpr int kLoads = KT * kVecPerRow / kThreads;  // 16-byte loads per thread per tensor
  static constexpr int kSideBytes = TileLayout<D>::bytes(KT);   // a tile's K, or V; two of K, then two of V
  // workgroups that share a CU: eight waves at head_dim 128 and with split keys have it to themselves.  The kernel's register
  // budget is this number's, and the plan counts on it.  (Left to the whole file, four waves at head_dim 128 took 290 and one
  // workgroup fitted: B1 H20 S3000 100 -> 68 us with the budget, 0.84 in the geometric mean of 93 drawn launches; at head_dim
  // 64 accumulators no longer move between the two halves of the file, 0.88 of 107.)
  static constexpr int kPerCu = NW == 8 && (D >= 128 || KS > 1) ? 1 : 2;
  // the Q fragments pass through LDS behind the tile buffers where there is room, so that the first tile is requested at once, and
  // through the tile buffers otherwise
  static constexpr size_t kTiles = 4 * kSideBytes, kFragmentBytes = NW * QB * WaveTile<D>::kRegionBytes;
  static constexpr bool kBehind = kPerCu * (kTiles + kFragmentBytes) <= 160 * 1024;
  static constexpr size_t kFragments = kBehind ? kTiles : 0, kLdsBytes = kTiles + (kBehind ? kFragmentBytes : 0);
  static_assert(NW * QB * kRowRegionBytes <= kLdsBytes, "the epilogue reuses the tile buffers");
  static_assert(kFragmentBytes <= kLdsBytes);
  static_assert(kPerCu * kLdsBytes <= 160 * 1024, "the workgroups of a CU share its LDS");
  // exchange of partial states between key-split waves: per wave O^T accumulators (D/32 x 16 registers x 64 lanes) + m + l
  static constexpr size_t kExchangeBytes = (D / 32) * 16 * 64 * 4 + 2 * 64 * 4;
  static_assert(KS == 1 || NW * kExchangeBytes <= kLdsBytes, "the exchange reuses the tile buffers");
  static_assert(kFragments + NW * QB * WaveTile<D>::kRegionBytes <= kLdsBytes, "the Q fragments pass through LDS");
  static_assert(KT % BN == 0 && (KT * kVecPerRow) % kThreads == 0, "tile must split evenly over the threads");
};

// what a wave of a piece leaves: O^T accumulators, m and l per lane
constexpr int fwd_piece_floats(int D) { return (D / 32) * 16 * kWave + 2 * kWave; }

// lse per query (the head's rows start at lse_row0); the wave's 32 output rows leave through its piece of LDS as whole lines
template <int D>
__device__ __forceinline__ void fwd_epilogue(const FwdParams& p, unsigned char* region, f32x16 (&o)[D / 32], float m_run, float l_run,
                                             int b, int hq, int64_t lse_row0, int row0, int lane) {
  const AttnParams& a = p.a;
  const int row = row0 + lane % 32;
  const float l_tot = half_sum(l_run);
  const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
  if (row < a.Sq && lane < 32)
    p.lse[lse_row0 + row] = l_tot > 0.f ? (m_run + fast_log2(l_tot)) * kLn2 : -INFINITY;
  // normalise in place: 1 / l differs per lane (row), the store helper applies one scale to all
#pragma unroll
  for (int db = 0; db < D / 32; ++db)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[db][i] *= inv;
  const int64_t off = b * a.os[0] + hq * a.os[1] + static_cast<int64_t>(row0) * a.os[2];
  if (p.out_f32)
    wave_store_rows<D, true>(region, o, 1.f, static_cast<float*>(p.out) + off, a.os[2], a.Sq - row0, lane, false, false);
  else
    wave_store_rows<D, false>(region, o, 1.f, static_cast<__bf16*>(p.out) + off, a.os[2], a.Sq - row0, lane, false, false);
}

// kCut: tiles may be cut into pieces (see Pieces) and chunks may end inside a key tile; a kernel of its own, because the loop
// of the plain one loses up to 10 % to that bookkeeping (B4 H32 S1024 D64 29.9 -> 33.0 us, B1 H32 S4096 D128 137 -> 144).
template <int D, int QB, int NW, int KT, int KS, bool kCut>
__global__ __launch_bounds__(64 * NW, (FwdCfg<D, QB, NW, KT, KS>::kPerCu * NW / 4)) void attn_fwd_kernel(const FwdParams p) {
  using C = FwdCfg<D, QB, NW, KT, KS>;
  using L = TileLayout<D>;
  constexpr int BM = C::BM, BN = C::BN;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];

  // (whole tiles at head_dim 64 leave the rotation's line out: us of launches behind each other, with it and without, B2 H9/3 S256 6.08, 6.02, rotated 7.07,
  // 7.00, B8 H3 S1314 15.47, 15.33; replayed from a graph, whose arguments stay in the caches, 5.50, 5.45, and 5.45 without any of this.  The others gain by it:
  // head_dim 128 B4 H1 S153 7.22, 7.17, B8 H2 S182 7.40, 7.34; cut at head_dim 64 B2 H1 S5778 29.83, 29.72)
  if constexpr (D == 128 || kCut) {
    const Arguments<sizeof(FwdParams) - 4> rope;
    AttnArguments().arrive();
    rope.arrive();
  } else {
    AttnArguments().arrive();
  }
  const AttnParams& a = p.a;
  const int n_qtiles = (a.Sq + BM - 1) / BM;
  // key tiles that the queries of a tile see (the last of a head's query tiles comes first in the order below)
  auto trips_of = [&](int i) { return query_tile_trips(a, n_qtiles - 1 - i, BM, KT); };
  // grid = (Hq * B, query tiles): x runs fastest in dispatch order, so every head's last query tile (the
  // longest under a causal mask) starts first and the short tiles fill in behind.  When the whole launch is
  // resident at once (pair_order), workgroups j and j + (half the grid) share a CU, so the second half runs
  // the short tiles in ASCENDING order: every CU then holds a long and a short tile of equal total length.
  const int y = static_cast<int>(blockIdx.y), half = (n_qtiles + 1) / 2;
  Piece piece = {y, 0, 1};
  if (kCut && a.pieces.len > 0) piece = find_piece(y, n_qtiles, a.pieces.len, trips_of);
  const int qtile = (!kCut && p.pair_order && y >= half) ? y - half : n_qtiles - 1 - piece.tile;
  const int hq = blockIdx.x % a.Hq, b = blockIdx.x / a.Hq;
  const int hkv = hq / (a.Hq / a.Hkv);
  const int q0 = qtile * BM;
  const int tid = threadIdx.x, lane = tid % 64;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);   // uniform over the wave: lets wave-dependent tests be scalar branches
  const int n = lane % 32, h = lane / 32;
  const int qw = wave % C::kQWaves, ks = wave / C::kQWaves;   // which queries, which 64-key step of a staged tile

  const __bf16* qbase = a.q + b * a.qs[0] + hq * a.qs[1];

  // ---- key range of this query tile
  const int q_hi = (q0 + BM < a.Sq ? q0 + BM : a.Sq);           // one past the last live query
  int kv_end = a.Sk;
  if (a.causal) {
    const int vis = a.q_offset + q_hi;                            // keys < vis can be seen by some query
    kv_end = vis < a.Sk ? vis : a.Sk;
    if (kv_end < 0) kv_end = 0;
  }
  int t_first = 0, ntiles = kCut ? tiles_before(a.kv, kv_end, KT) : (kv_end + KT - 1) / KT;
  if (kCut && piece.parts > 1) {
    t_first = ntiles * piece.part / piece.parts;
    ntiles = ntiles * (piece.part + 1) / piece.parts - t_first;
  }

  // ---- staging of one K/V tile of KT keys: a wave-uniform window per tile (first key row, bytes left in the
  //      sequence) plus per-lane byte offsets that are computed once; rows past Sk read as zeros.  A lane asks for the
  //      piece that belongs at its place of LDS (TileLayout).  The loop body holds no wait for memory other than the
  //      one in front of the barrier that ends a trip, a whole tile after the requests.
  uint32_t k_off[C::kLoads], v_off[C::kLoads];
#pragma unroll
  for (int i = 0; i < C::kLoads; ++i) {
    const int r = L::row(wave + NW * i, lane), cv = L::column(lane);
    k_off[i] = static_cast<uint32_t>((static_cast<int64_t>(r) * a.ks[2] + cv) * 2);
    v_off[i] = static_cast<uint32_t>((static_cast<int64_t>(r) * a.vs[2] + cv) * 2);
  }
  // a cursor walks the key tiles in order (and from chunk to chunk): stepping it is a few scalar adds
  KvCursor<D> cur;
  cur.open(a, t_first, b, hkv, KT);
  KvPosition pos;
  pos.open(a.kv, t_first, KT);
  // the next tile goes to LDS buffer `buf`
  auto request_tile = [&](int buf) {
    const u32x4 kb = request_window(reinterpret_cast<uint64_t>(cur.k), cur.k_left), vb = request_window(reinterpret_cast<uint64_t>(cur.v), cur.v_left);
    const uint32_t to = static_cast<uint32_t>(buf) * C::kSideBytes + wave * L::kPitch;
    each_load<C::kLoads>([&](auto load) {
      constexpr int i = decltype(load)::value;
      request16_to<i * NW * L::kPitch>(to, kb, k_off[i]);
      request16_to<2 * C::kSideBytes + i * NW * L::kPitch>(to, vb, v_off[i]);
    });
    cur.next(a);
  };

  if constexpr (C::kBehind) {
    if (ntiles > 0) request_tile(0);
  }

  // ---- Q fragments (B operand of S^T): lane = query, 8 consecutive d per 16-wide k step; fetched row-major and
  //      turned into fragments through the wave's piece of LDS (the tile buffers are filled only after the
  //      barrier below)
  bf16x8 qf[QB][D / 16];
  int qrow[QB];
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    const int row0 = q0 + (qw * QB + qb) * 32;
    qrow[qb] = row0 + n;
    WaveTile<D> qt;
    qt.issue(make_buffer(qbase + static_cast<int64_t>(row0) * a.qs[2], span_bytes(a.Sq - row0, a.qs[2], D)), a.qs[2], lane);
    qt.fragments(smem_raw + C::kFragments + (wave * QB + qb) * WaveTile<D>::kRegionBytes, lane, qf[qb]);
    if (p.rope.cos != nullptr) {
      // RoPE on the wave's own queries, once per query in the whole launch (every query belongs to one wave)
      const bool qlive = qrow[qb] < a.Sq;
      rope_rotate_fragments<D>(qf[qb], p.rope, qlive ? p.rope.q_pos0 + qrow[qb] : 0, h);
      if (p.q_rot != nullptr && qlive && (KS == 1 || ks == 0) && piece.part == 0) {
        __bf16* dst = p.q_rot + b * p.qrs[0] + hq * p.qrs[1] + static_cast<int64_t>(qrow[qb]) * p.qrs[2];
#pragma unroll
        for (int s = 0; s < D / 16; ++s) *reinterpret_cast<bf16x8*>(dst + 16 * s + 8 * h) = qf[qb][s];
      }
    }
  }

  // ---- running state: m in the log2 domain (scores scaled by sm_scale*log2e), l split over the halves
  const float c = a.sm_scale * kLog2e;
  float m_run[QB], l_run[QB];
  f32x16 o[QB][D / 32];
  const int64_t lse_row0 = (static_cast<int64_t>(b) * a.Hq + hq) * a.Sq;
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    m_run[qb] = -INFINITY;
    l_run[qb] = 0.f;
#pragma unroll
    for (int db = 0; db < D / 32; ++db)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[qb][db][i] = 0.f;
    if (p.merge && ks == 0 && piece.part == 0 && qrow[qb] < a.Sq) {
      // continue from (out, lse) of the earlier blocks: m = lse, l = 1, acc = out
      const float prev = p.lse[lse_row0 + qrow[qb]];
      if (prev != -INFINITY) {
        m_run[qb] = prev * kLog2e;
        l_run[qb] = (h == 0) ? 1.f : 0.f;
        const float* po = static_cast<const float*>(p.out) + b * a.os[0] + hq * a.os[1] +
                          static_cast<int64_t>(qrow[qb]) * a.os[2];
#pragma unroll
        for (int db = 0; db < D / 32; ++db)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const f32x4 v4 = *reinterpret_cast<const f32x4*>(po + 32 * db + 8 * j + 4 * h);
#pragma unroll
            for (int t = 0; t < 4; ++t) o[qb][db][4 * j + t] = v4[t];
          }
      }
    }
  }

  if constexpr (!C::kBehind) {
    __syncthreads();  // every wave has its Q fragments: the tile buffers may be filled
    if (ntiles > 0) request_tile(0);
  }
  // While tile 0 is on its way: the lane's places in the K and V tiles, and how many tiles the wave's queries see.  Those come first in
  // its loop; with the others it only helps.  (A test inside the trip made the accumulators' registers depend on it, and the compiler
  // copied all of them in some orders of the trip.  Counted behind the barrier, with a division for chunks that only kCut has inside tiles,
  // a launch of one key tile paid 0.2 us for it: B8 H16/4 S17 D128 5.44 -> 5.78, this way 5.5.)
  static_assert(QB == 1);
  uint32_t row_at = L::row_place(lane), tr_at = 2 * C::kSideBytes + L::column_place(lane);
  const int see = max(min(a.causal ? a.q_offset + q0 + 32 * qw + 32 : kv_end, kv_end) - BN * ks, 0);
  int mine = min(max((kCut ? tiles_before(a.kv, see, KT) : (see + KT - 1) / KT) - t_first, 0), ntiles);
  asm volatile("" : "+v"(row_at), "+v"(tr_at), "+s"(mine));   // (kept, not computed again in front of the reads)
  // Every load issued so far (Q fragments, the merge state, tile 0) is complete from here on.  Without this the
  // barrier would publish a tile that is still on its way, and the compiler would put a vmcnt(0) wait in front of the
  // loop's first MFMAs, where it would wait for the NEXT tile on every trip.
  __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);
  __syncthreads();

  // a trip on the LDS buffer `parity`, a constant, so that a lane's addresses are the same in every trip
  auto trip = [&](auto parity, int t) __attribute__((always_inline)) {
    constexpr uint32_t kAt = decltype(parity)::value * C::kSideBytes;
    static_assert(kAt + L::rows(KT - 32) + L::kRows16 + L::kRows8 + 2 * D <= 65535, "offsets of LDS reads");
    const int tile_key0 = kCut ? pos.key0 : t * KT, keys_end = kCut ? pos.end : a.Sk;
    if constexpr (kCut) pos.next(a.kv, KT);
    // tile t+1 goes into the other buffer (its readers finished before the barrier that ended trip t-1)
    if (t + 1 < ntiles) request_tile(1 - decltype(parity)::value);

#pragma unroll
    for (int sub = 0; sub < KT / BN; ++sub) {
      if (KS > 1 && sub != ks) continue;
      const int k0 = tile_key0 + sub * BN;
      if (kCut && KT > BN && k0 >= keys_end) break;
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) {
        const int blk_q_lo = a.q_offset + q0 + (qw * QB + qb) * 32;  // position of the block's first query
        // ---- S^T[key][query] for 64 keys x 32 queries
        f32x16 s_acc[BN / 32];
        // Where no order is pinned by hand (head_dim 64), the compiler's scheduler is asked for its MFMA / LDS-read
        // interleaving of this block (-1 % with 8 waves, -5 % with 4; the key-split variant is better off without)
        if constexpr (C::kKDepth == 0 && KS == 1) __builtin_amdgcn_iglp_opt(0);
        // D = 128: the K fragments are fetched from LDS a fixed number of MFMAs ahead of their use.  An LDS read
        // takes several MFMA times to come back, so a read issued right before its MFMA leaves the matrix pipe
        // waiting for it (measured: +5 %).  At D = 64 the softmax arithmetic, not this wait, paces the loop, and the
        // compiler's own order is 2 % faster.
        if constexpr (C::kKDepth > 0) {
          constexpr int kSteps = (BN / 32) * (D / 16), kDepth = C::kKDepth < kSteps ? C::kKDepth : kSteps;
          bf16x8 kf[kSteps];
#pragma unroll
          for (int j = 0; j < kSteps; ++j)
            kf[j] = lds_at<bf16x8>(row_at + (kAt + L::rows(sub * BN + 32 * (j / (D / 16))) + j % (D / 16) * 32));
#pragma unroll
          for (int mb = 0; mb < BN / 32; ++mb) {
#pragma unroll
            for (int i = 0; i < 16; ++i) s_acc[mb][i] = 0.f;
#pragma unroll
            for (int s = 0; s < D / 16; ++s) s_acc[mb] = mfma32(kf[mb * (D / 16) + s], qf[qb][s], s_acc[mb]);
          }
          // scheduling groups: kDepth LDS reads, then one MFMA and one read in turn, then the last kDepth MFMAs
          __builtin_amdgcn_sched_group_barrier(0x100, kDepth, 0);
#pragma unroll
          for (int j = 0; j < kSteps - kDepth; ++j) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
          }
          __builtin_amdgcn_sched_group_barrier(0x008, kDepth, 0);
        } else {
#pragma unroll
          for (int mb = 0; mb < BN / 32; ++mb) {
#pragma unroll
            for (int i = 0; i < 16; ++i) s_acc[mb][i] = 0.f;
#pragma unroll
            for (int s = 0; s < D / 16; ++s) {
              const bf16x8 kf = lds_at<bf16x8>(row_at + (kAt + L::rows(sub * BN + 32 * mb) + s * 32));
              s_acc[mb] = mfma32(kf, qf[qb][s], s_acc[mb]);
            }
          }
        }
        // ---- mask (only for tiles that straddle the diagonal or the end of their chunk)
        const bool need_mask = (a.causal && k0 + BN - 1 > blk_q_lo) || (k0 + BN > keys_end);
        if (need_mask) {
          // the asm statement keeps this a real (wave-uniform) branch: without it the compiler turns the
          // block into per-element selects that every tile pays for
          asm volatile("; masked tile" ::: "memory");
          const int qpos = a.causal ? a.q_offset + qrow[qb] : 0x7fffffff;
          const int last = (qpos < keys_end ? qpos : keys_end - 1) - k0 - 4 * h;   // (one compare with a constant per element)
#pragma unroll
          for (int mb = 0; mb < BN / 32; ++mb)
#pragma unroll
            for (int i = 0; i < 16; ++i)
              if (32 * mb + 8 * (i / 4) + i % 4 > last) s_acc[mb][i] = -INFINITY;
        }
        // ---- online softmax.  The running maximum is only raised (and O, l rescaled) when some query of
        //      the wave saw its maximum grow by more than 2^kTau; until then exp2(s - m) may exceed 1 by at
        //      most that factor, which fp32 accumulators and bf16 probabilities hold without loss.
        constexpr float kTau = 8.f;
        float mx = s_acc[0][0];
#pragma unroll
        for (int mb = 0; mb < BN / 32; ++mb)
#pragma unroll
          for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s_acc[mb][i]);
        mx = half_max(mx) * c;
        if (__any(mx > m_run[qb] + kTau)) {
          const float m_new = fmaxf(m_run[qb], mx);
          const float alpha = (m_new == -INFINITY) ? 1.f : fast_exp2(m_run[qb] - m_new);
          m_run[qb] = m_new;
#pragma unroll
          for (int db = 0; db < D / 32; ++db)
#pragma unroll
            for (int i = 0; i < 16; ++i) o[qb][db][i] *= alpha;
          l_run[qb] *= alpha;
        }
        const float m_use = (m_run[qb] == -INFINITY) ? 0.f : m_run[qb];
        float psum = 0.f;
        if constexpr (D == 128 && NW == 4) {
          // O^T += V^T P^T, eight keys of a lane at a time, exp2 of the next eight dealt out between the MFMAs: a wave issues in order, and
          // vector work that stands in front of a product leaves the matrix pipe idle.  B1 H20 S1500 37.8 -> 32.5 us, B4 H8 S900 25.2 -> 21.9, B1 H8
          // S700 18.1 -> 15.7.  (Eight waves lose by it, B1 H32 S4096 150 -> 152 right after a pause: their launches draw the power that the clock has
          // to fall for.  At head_dim 64 a product is too short to cover the exponentials: B4 H32 S1024 28.5 -> 29.2.)
          constexpr int kDb = D / 32, kAll = 4 * kDb, kPer = 8 / kDb, kAhead = 2;
          auto probability = [&](int e) {
            const float pv = fast_exp2(s_acc[e / 16][e % 16] * c - m_use);
            s_acc[e / 16][e % 16] = pv;
            psum += pv;
          };
          bf16x8 vf[kAll], pf[4];
          auto fetch = [&](int i) { vf[i] = lds_tr_at<D>(tr_at + (kAt + L::rows(sub * BN + 32 * (i / (2 * kDb))) + i / kDb % 2 * L::kRows16 + i % kDb * 64)); };
#pragma unroll
          for (int i = 0; i < kAhead; ++i) fetch(i);
#pragma unroll
          for (int e = 0; e < 8; ++e) probability(e);
          pf[0] = pack8(s_acc[0], 0);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int i = 0; i < kAll; ++i) {
            const int step = i / kDb, db = i % kDb;
            if (i + kAhead < kAll) fetch(i + kAhead);
            o[qb][db] = mfma32(vf[i], pf[step], o[qb][db]);
            if (step < 3) {
#pragma unroll
              for (int e = 0; e < kPer; ++e) probability(8 * (step + 1) + kPer * db + e);
              if (db + 1 == kDb) pf[step + 1] = pack8(s_acc[(step + 1) / 2], (step + 1) % 2 * 8);
            }
            __builtin_amdgcn_sched_barrier(0);
          }
          l_run[qb] += psum;
        } else {
#pragma unroll
          for (int mb = 0; mb < BN / 32; ++mb)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
              const float pv = fast_exp2(s_acc[mb][i] * c - m_use);
              s_acc[mb][i] = pv;
              psum += pv;
            }
          l_run[qb] += psum;
          // ---- O^T[d][query] += V^T[d][key] P^T[key][query]
#pragma unroll
          for (int mb = 0; mb < BN / 32; ++mb)
#pragma unroll
            for (int cc = 0; cc < 2; ++cc) {
              const bf16x8 pf = pack8(s_acc[mb], 8 * cc);
#pragma unroll
              for (int db = 0; db < D / 32; ++db) {
                const bf16x8 vf = lds_tr_at<D>(tr_at + (kAt + L::rows(sub * BN + 32 * mb) + cc * L::kRows16 + db * 64));
                o[qb][db] = mfma32(vf, pf, o[qb][db]);
              }
            }
        }
      }
    }
    wait_requests<0>();
    __syncthreads();  // all waves are done with buffer t&1 (it is refilled in trip t+1) and tile t+1 is visible
  };
  int t = 0;
  while (t < mine) {
    trip(std::integral_constant<int, 0>(), t++);
    if (t >= mine) break;
    trip(std::integral_constant<int, 1>(), t++);
  }
  for (; t < ntiles; ++t) {
    if (t + 1 < ntiles) request_tile((t + 1) % 2);
    wait_requests<0>();
    __syncthreads();
  }

  // ---- key split: the waves ks > 0 hand their partial state to the wave ks == 0 of the same queries through LDS
  //      (the loop ended on a barrier, so the tile buffers are free).  States with different reference maxima m
  //      combine as O = sum_i 2^(m_i - m) O_i, l = sum_i 2^(m_i - m) l_i with m = max_i m_i.
  if constexpr (KS > 1) {
    float* xo = reinterpret_cast<float*>(smem_raw + wave * C::kExchangeBytes);
    float* xm = xo + (D / 32) * 16 * 64;
    if (ks > 0) {
#pragma unroll
      for (int db = 0; db < D / 32; ++db)
#pragma unroll
        for (int i = 0; i < 16; ++i) xo[(db * 16 + i) * 64 + lane] = o[0][db][i];
      xm[lane] = m_run[0];
      xm[64 + lane] = l_run[0];
    }
    __syncthreads();
    if (ks > 0) return;
    float m_all = m_run[0];
#pragma unroll
    for (int j = 1; j < KS; ++j) {
      const float* om = reinterpret_cast<const float*>(smem_raw + (qw + j * C::kQWaves) * C::kExchangeBytes) + (D / 32) * 16 * 64;
      m_all = fmaxf(m_all, om[lane]);
    }
    const float a0 = (m_run[0] == -INFINITY) ? 0.f : fast_exp2(m_run[0] - m_all);
#pragma unroll
    for (int db = 0; db < D / 32; ++db)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[0][db][i] *= a0;
    l_run[0] *= a0;
#pragma unroll
    for (int j = 1; j < KS; ++j) {
      const float* oo = reinterpret_cast<const float*>(smem_raw + (qw + j * C::kQWaves) * C::kExchangeBytes);
      const float* om = oo + (D / 32) * 16 * 64;
      const float mj = om[lane];
      const float aj = (mj == -INFINITY) ? 0.f : fast_exp2(mj - m_all);
#pragma unroll
      for (int db = 0; db < D / 32; ++db)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[0][db][i] += aj * oo[(db * 16 + i) * 64 + lane];
      l_run[0] += aj * om[64 + lane];
    }
    m_run[0] = m_all;
    // (the rows below leave through the first kQWaves * kRowRegionBytes of LDS, which no exchange area of a ks > 0 wave
    // overlaps)
    static_assert(C::kQWaves * kRowRegionBytes <= C::kQWaves * C::kExchangeBytes, "store pieces lie below the exchange areas read above");
  }

  if constexpr (QB == 1 && kCut) {
    if (piece.parts > 1) {   // one piece of several: the state leaves as it is (l per wave half)
      float* dst = a.pieces.ws + ((static_cast<int64_t>(blockIdx.x) * gridDim.y + blockIdx.y) * C::kQWaves + qw) * fwd_piece_floats(D);
      put_acc<D / 32>(dst, o[0], lane);
      dst[(D / 32) * 16 * kWave + lane] = m_run[0];
      dst[(D / 32) * 16 * kWave + kWave + lane] = l_run[0];
      return;
    }
  }
#pragma unroll
  for (int qb = 0; qb < QB; ++qb)
    fwd_epilogue<D>(p, smem_raw + (wave * QB + qb) * kRowRegionBytes, o[qb], m_run[qb], l_run[qb], b, hq, lse_row0,
                    q0 + (qw * QB + qb) * 32, lane);
}

// The pieces of every cut query tile put together: a wave per 32 queries merges the pieces' states, which lie as the pieces'
// registers held them, and ends as the kernel above does.
template <int D, int QW, int KT>
__global__ __launch_bounds__(64 * QW) void attn_fwd_join_kernel(const FwdParams p, const int pieces_per_head) {
  __shared__ __attribute__((aligned(16))) unsigned char smem_raw[QW * kRowRegionBytes];
  const AttnParams& a = p.a;
  constexpr int BM = 32 * QW;
  const int n_qtiles = (a.Sq + BM - 1) / BM, tile = static_cast<int>(blockIdx.y);
  auto trips_of = [&](int i) { return query_tile_trips(a, n_qtiles - 1 - i, BM, KT); };
  const int parts = pieces_of(trips_of(tile), a.pieces.len);
  if (parts == 1) return;   // (its workgroup has written the tile)
  const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int hq = blockIdx.x % a.Hq, b = blockIdx.x / a.Hq;
  const int row0 = (n_qtiles - 1 - tile) * BM + wave * 32;
  const int64_t first = static_cast<int64_t>(blockIdx.x) * pieces_per_head + first_piece(tile, a.pieces.len, trips_of);
  constexpr int kAcc = (D / 32) * 16 * kWave;
  const float* src = a.pieces.ws + (first * QW + wave) * fwd_piece_floats(D);
  constexpr int64_t kStep = static_cast<int64_t>(QW) * fwd_piece_floats(D);
  float m = -INFINITY, l = 0.f;
  for (int j = 0; j < parts; ++j) m = fmaxf(m, src[j * kStep + kAcc + lane]);
  f32x16 o[D / 32];
#pragma unroll
  for (int db = 0; db < D / 32; ++db)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[db][i] = 0.f;
  for (int j = 0; j < parts; ++j) {
    const float* sj = src + j * kStep;
    const float mj = sj[kAcc + lane], lj = sj[kAcc + kWave + lane];
    f32x4 raw[D / 32][4];
    get_acc<D / 32>(sj, raw, lane);
    const float aj = mj == -INFINITY ? 0.f : fast_exp2(mj - m);
    l += aj * lj;
#pragma unroll
    for (int db = 0; db < D / 32; ++db)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[db][i] += aj * raw[db][i / 4][i % 4];
  }
  fwd_epilogue<D>(p, smem_raw + wave * kRowRegionBytes, o, m, l, b, hq, (static_cast<int64_t>(b) * a.Hq + hq) * a.Sq, row0, lane);
}

template <int D, int QB, int NW, int KT, int KS, bool kCut>
int launch_impl(const FwdParams& p, hipStream_t s) {
  using C = FwdCfg<D, QB, NW, KT, KS>;
  static LdsOnce lds_reserved;
  if (!reserve_lds_once(lds_reserved, reinterpret_cast<const void*>(&attn_fwd_kernel<D, QB, NW, KT, KS, kCut>), C::kLdsBytes))
    return fail(PICO_ERR_LAUNCH, "pico_attn_fwd: cannot reserve %zu bytes of LDS", C::kLdsBytes);
  const int heads = p.a.Hq * p.a.B, n_qtiles = (p.a.Sq + C::BM - 1) / C::BM, len = p.a.pieces.len;
  FwdParams q = p;
  // (the pairing needs two workgroups per CU: at head_dim 128 the eight-wave kernel has one, the launch is two
  // generations of workgroups and longest-first is the better order -- 160 -> 137 us at B1 H32 S4096)
  constexpr bool kTwoPerCu = !(D >= 128 && NW == 8);
  q.pair_order = !kCut && kTwoPerCu && p.a.causal && n_qtiles >= 2 && static_cast<int64_t>(heads) * n_qtiles <= 512;
  const int n = count_pieces(n_qtiles, len, [&](int i) { return query_tile_trips(p.a, n_qtiles - 1 - i, C::BM, KT); });
  hipLaunchKernelGGL((attn_fwd_kernel<D, QB, NW, KT, KS, kCut>), dim3(heads, n), dim3(C::kThreads), C::kLdsBytes, s, q);
  if (kCut && len > 0)
    hipLaunchKernelGGL((attn_fwd_join_kernel<D, C::kQWaves, KT>), dim3(heads, n_qtiles), dim3(64 * C::kQWaves), 0, s, q, n);
  return PICO_OK;
}
template <int D, int QB, int NW, int KT, int KS = 1>
int launch(const FwdParams& p, hipStream_t s) {
  return p.a.pieces.len > 0 || ends_inside_tile(p.a.kv, KT) ? launch_impl<D, QB, NW, KT, KS, true>(p, s) : launch_impl<D, QB, NW, KT, KS, false>(p, s);
}

}  // namespace

int check_attn_desc(const char* fn, const pico_attn_desc* d) {
  if (!d) return fail(PICO_ERR_NULL, "%s: descriptor is NULL", fn);
  if (d->D != 64 && d->D != 128) return fail(PICO_ERR_SHAPE, "%s: head_dim %d not supported (64 or 128)", fn, d->D);
  if (d->B < 0 || d->Hq <= 0 || d->Hkv <= 0 || d->Sq < 0 || d->Sk < 0)
    return fail(PICO_ERR_SHAPE, "%s: negative size (B=%d Hq=%d Hkv=%d Sq=%d Sk=%d)", fn, d->B, d->Hq, d->Hkv, d->Sq, d->Sk);
  if (d->Hq % d->Hkv != 0) return fail(PICO_ERR_SHAPE, "%s: Hq=%d is not a multiple of Hkv=%d", fn, d->Hq, d->Hkv);
  if (static_cast<int64_t>(d->B) * d->Hq > 0x7fffffffLL) return fail(PICO_ERR_SHAPE, "%s: B * Hq too large", fn);
  if (d->q_offset < 0) return fail(PICO_ERR_SHAPE, "%s: q_offset=%d must be >= 0", fn, d->q_offset);
  if (!(d->sm_scale > 0.f)) return fail(PICO_ERR_SHAPE, "%s: sm_scale must be positive", fn);
  const int64_t* all[4] = {d->q_stride, d->k_stride, d->v_stride, d->o_stride};
  for (const int64_t* st : all)
    for (int i = 0; i < 3; ++i)
      if (st[i] < 0 || st[i] % 8 != 0)
        return fail(PICO_ERR_STRIDE, "%s: strides must be non-negative multiples of 8 elements", fn);
  // the kernels address one head's rows through 32-bit byte offsets (the key side is checked per chunk, set_chunks)
  const int64_t spans[2] = {(d->Sq - 1) * d->q_stride[2], (d->Sq - 1) * d->o_stride[2]};
  for (int64_t span : spans)
    if ((span + d->D) * 2 >= (1LL << 32))
      return fail(PICO_ERR_STRIDE, "%s: the rows of one head must span less than 4 GiB", fn);
  return PICO_OK;
}

int check_rope_tables(const char* fn, const pico_rope_tables* t, int D, int64_t last_pos) {
  if (!t || !t->cos || !t->sin) return fail(PICO_ERR_NULL, "%s: cos / sin tables are required", fn);
  if (t->dtype != PICO_BF16 && t->dtype != PICO_F32) return fail(PICO_ERR_DTYPE, "%s: table dtype code %d not supported", fn, t->dtype);
  if (t->pitch < D / 2 || t->pitch % 4 != 0 || !aligned16(t->cos) || !aligned16(t->sin) ||
      (t->dtype == PICO_BF16 && t->pitch % 8 != 0))
    return fail(PICO_ERR_STRIDE, "%s: table rows must hold D/2 columns, start 16-byte aligned and lie a multiple of 16 bytes apart", fn);
  if (last_pos >= t->rows) return fail(PICO_ERR_SHAPE, "%s: positions up to %lld needed, the tables have %d rows", fn,
                                       static_cast<long long>(last_pos), t->rows);
  return PICO_OK;
}

AttnParams make_params(const pico_attn_desc* d, const void* q, const void* k, const void* v) {
  AttnParams a;
  a.q = static_cast<const __bf16*>(q);
  for (int c = 0; c < kMaxChunks; ++c) a.kv.k[c] = a.kv.v[c] = nullptr;
  a.kv.k[0] = static_cast<const __bf16*>(k);
  a.kv.v[0] = static_cast<const __bf16*>(v);
  a.kv.count = 1;
  a.kv.len = d->Sk;
  a.B = d->B; a.Hq = d->Hq; a.Hkv = d->Hkv; a.Sq = d->Sq; a.Sk = d->Sk;
  a.causal = d->causal != 0;
  a.q_offset = d->q_offset;
  a.sm_scale = d->sm_scale;
  a.pieces = Pieces{0, nullptr};
  for (int i = 0; i < 3; ++i) {
    a.qs[i] = d->q_stride[i]; a.ks[i] = d->k_stride[i]; a.vs[i] = d->v_stride[i]; a.os[i] = d->o_stride[i];
  }
  return a;
}

int set_chunks(const char* fn, const pico_attn_desc* d, const pico_kv_chunks* kv, AttnParams& a, bool need_kv) {
  if (!kv) return fail(PICO_ERR_NULL, "%s: the chunk list is NULL", fn);
  if (kv->count < 1 || kv->count > kMaxChunks)
    return fail(PICO_ERR_SHAPE, "%s: %d chunks (1 to %d supported)", fn, kv->count, kMaxChunks);
  if (kv->chunk_len < 0 || static_cast<int64_t>(kv->count) * kv->chunk_len != d->Sk)
    return fail(PICO_ERR_SHAPE, "%s: %d chunks of %d keys do not make Sk=%d", fn, kv->count, kv->chunk_len, d->Sk);
  // a tile belongs to one chunk: chunks of one 64-key step or less would leave most of every tile empty
  if (kv->count > 1 && kv->chunk_len <= 64)
    return fail(PICO_ERR_SHAPE, "%s: with several chunks the chunk length (%d) must be over 64 (best a multiple of 128)", fn, kv->chunk_len);
  // a chunk is addressed through the same 32-bit window as a whole tensor
  if (((kv->chunk_len - 1) * std::max(d->k_stride[2], d->v_stride[2]) + d->D) * 2 >= (1LL << 32))
    return fail(PICO_ERR_STRIDE, "%s: the rows of one head must span less than 4 GiB", fn);
  for (int c = 0; c < kv->count; ++c) {
    if (need_kv && (!kv->k[c] || !kv->v[c])) return fail(PICO_ERR_NULL, "%s: k / v of chunk %d are NULL", fn, c);
    if (!aligned16(kv->k[c]) || !aligned16(kv->v[c]) || !aligned16(kv->dk[c]) || !aligned16(kv->dv[c]))
      return fail(PICO_ERR_ALIGN, "%s: chunk %d: k, v, dk and dv must be 16-byte aligned", fn, c);
    a.kv.k[c] = static_cast<const __bf16*>(kv->k[c]);
    a.kv.v[c] = static_cast<const __bf16*>(kv->v[c]);
  }
  a.kv.count = kv->count;
  a.kv.len = kv->chunk_len;
  return PICO_OK;
}

}  // namespace pico

using namespace pico;

namespace {

// rows of [B, H, S, D] memory addressed by `st` must not overlap: every stride spans what lies inside it
bool rows_disjoint(const int64_t* st, int B, int H, int S, int D) {
  struct Dim { int64_t stride; int extent; } dims[3] = {{st[0], B}, {st[1], H}, {st[2], S}};
  std::sort(dims, dims + 3, [](const Dim& x, const Dim& y) { return x.stride < y.stride; });
  int64_t span = D;   // elements covered by the dimensions handled so far
  for (const Dim& d : dims) {
    if (d.extent <= 1) continue;
    if (d.stride < span) return false;
    span = d.stride * (d.extent - 1) + span;
  }
  return true;
}

// How a launch is run: which kernel, and whether its query tiles are cut into pieces (see Pieces).
struct FwdPlan {
  enum { kWaves4, kWaves8, kSplit4, kSplit8 } kernel;
  int len = 0;               // piece length in staged key tiles, 0: not cut
  int64_t ws_bytes = 0;      // what the pieces need
};

FwdPlan make_fwd_plan(const AttnParams& a, int D) {
  FwdPlan plan;
  const int64_t heads = static_cast<int64_t>(a.B) * a.Hq;
  auto groups = [&](int bm) { return heads * ((a.Sq + bm - 1) / bm); };
  TripCost cost;
  int bm = 128, kt = 64;
  auto use = [&](auto cfg, double alone_us, double full_us, double cut) {
    using C = decltype(cfg);
    bm = C::BM;
    kt = C::kKT;
    cost = {alone_us, full_us, ends_inside_tile(a.kv, kt) ? 1.0 : cut, C::kPerCu, 0.0};   // (such chunks run the cutting kernel in any case)
  };
  // Tile choice for D = 64: more waves per workgroup share each staged K/V tile (fewer barriers and
  // global loads per MFMA), but the launch still has to fill 256 CUs, so small problems get small tiles.
  if (D == 64) {
    const int64_t visible_keys = a.causal ? std::min<int64_t>(a.Sk, static_cast<int64_t>(a.q_offset) + a.Sq) : a.Sk;
    // a launch whose queries all see at least as many keys as they are themselves (a rank's share of a ring, a dense
    // block): the waves of a workgroup then do nearly equal work, and workgroups of eight waves, which share every
    // staged tile among twice as many waves, pay even where the launch has few of them
    const bool rectangular = !a.causal || a.q_offset >= a.Sq;
    if (groups(256) >= 512) plan.kernel = FwdPlan::kWaves8;
    // (measured at B8, 256 queries x 1024 keys of every head: 26.9 us with eight waves, 30.1 us with four)
    else if (groups(128) >= 512) plan.kernel = rectangular && groups(256) >= 256 ? FwdPlan::kWaves8 : FwdPlan::kWaves4;
    // few waves in all: two waves per 32 queries, 64 keys of every 128 each -- in workgroups of eight waves (128 queries)
    // when those still cover the CUs and the launch is rectangular (one rank's share of B4 H32 S1024 in a ring of four: 19.8 -> 16.9 us for
    // rank 3 of 4; on a whole causal sequence, or with 256 keys, the smaller workgroups are a few percent faster)
    else plan.kernel = groups(128) >= 256 && rectangular && visible_keys >= 512 ? FwdPlan::kSplit8 : FwdPlan::kSplit4;
    switch (plan.kernel) {
      case FwdPlan::kWaves8: use(FwdCfg<64, 1, 8, 64>(), 1.55, 0.84, 1.15); break;
      case FwdPlan::kWaves4: use(FwdCfg<64, 1, 4, 64>(), 0.8, 0.4, 1.09); break;
      case FwdPlan::kSplit8: use(FwdCfg<64, 1, 8, 128, 2>(), 1.5, 1.3, 1.0); break;
      case FwdPlan::kSplit4: use(FwdCfg<64, 1, 4, 128, 2>(), 1.6, 0.5, 1.19); break;
    }
  } else {
    // (64-key staged tiles: 0.5-4 % faster than 128-key ones at every size measured)
    // Eight waves share each staged tile among 256 queries and have a CU to themselves; four waves do 128, two workgroups to a CU, and lose
    // 3 to 8 % where both fill the GPU evenly (B1 H32 S4096 130 us in a long row of launches, four waves 142, 150 and 161 right after a pause; 256 equal workgroups 70.5, 76; 384 causal ones
    // 50.2, 52.7).  Four waves win where eight leave CUs idle: up to 352 workgroups of 256 queries, most of which run alone on the second
    // round (B1 H32 S2048 58.0, four waves 48.0; S2500 76.0, 65.5; B2 H16 S2100 60.6, 52.4; from 360 on 1.04 times at the worst); just over
    // two rounds of equal ones (540: 295, 268; 624: 423, 384); and where a tenth of the queries of 256 do not exist (B8 H32 S300 30.0,
    // 22.0; B4 H32 S777 46.8, 39.0), unless the launch has many workgroups and the tiles' traffic counts (2304: 570, 628).  It never does for up to
    // 128 queries, one workgroup to a head either way, where half of eight waves and more have no query at all: B64 H32 S128 67.5, 45.1;
    // B128 H32/8 S64 88.5, 48.3; B48 H32/8 128 x 4096 762, 461.
    // From somewhere past 8192 keys on a head's K and V leave an XCD's L2 no room, and twice the traffic costs what the CUs gain.  The line
    // is a cut through launches that go both ways (288 workgroups, eight and four: 9 heads of 8192 x 8192 179, 174, without a mask 344, 362; x 10240
    // 403, 389, shifted 256, 234; x 12288 473, 460, shifted 314, 339; x 16384 618, 600, shifted 450, 491); at 32768 four lose in most (1207,
    // 1382; 36 heads of 2048 1374, 1662; 312 of 52184 1952, 2076).  Under one round of workgroups of eight the line does not hold them back,
    // which loses where the workgroups are about equal and few more than half a round (12 heads of 4096 x 16384 340, 387, x 32768 693, 852; 9 of
    // 4096 x 8192 131, 143), is level at 128 and 240 (466, 487; 937, 950) and pays for whole causal sequences (10 heads of 4096 65, 68; 14 heads 89, 77).
    const bool rectangular = !a.causal || a.q_offset >= a.Sq;   // (workgroups of about equal length)
    const int64_t wide = groups(256), narrow = groups(128);
    const bool idle = wide <= 352 && !(rectangular && wide == 256), third = rectangular && wide > 512 && wide <= 640;
    const bool padded = narrow <= 1024 && 10 * narrow <= 18 * wide;
    plan.kernel = wide < 256 || narrow == wide || (a.Sk <= 8192 && (idle || third || padded)) ? FwdPlan::kWaves4 : FwdPlan::kWaves8;
    if (plan.kernel == FwdPlan::kWaves8) use(FwdCfg<128, 1, 8, 64>(), 1.6, 2.13, 1.0);
    else use(FwdCfg<128, 1, 4, 64>(), 1.66, 0.96, 1.19);
  }
  const int n_qtiles = (a.Sq + bm - 1) / bm;
  cost.piece_bytes = 4.0 * (bm / 32) * fwd_piece_floats(D);
  auto trips_of = [&](int i) { return query_tile_trips(a, n_qtiles - 1 - i, bm, kt); };
  plan.len = choose_pieces(heads, n_qtiles, cost, false, trips_of);
  if (plan.len > 0) plan.ws_bytes = static_cast<int64_t>(heads * count_pieces(n_qtiles, plan.len, trips_of) * cost.piece_bytes);
  return plan;
}
const FwdPlan& plan_fwd(const AttnParams& a, int D) {
  static thread_local PlanTable<FwdPlan> table;
  return table.get(a, D, [&] { return make_fwd_plan(a, D); });
}

int run_fwd(const char* fn, const pico_attn_desc* desc, const void* q, const pico_kv_chunks* kv, void* out, float* lse,
            int out_dtype, int merge, const pico_rope_tables* rope, int q_pos_offset, void* q_rot,
            const int64_t* q_rot_stride, void* stream, float* workspace = nullptr, int64_t ws_bytes = 0) {
  if (int rc = check_attn_desc(fn, desc)) return rc;
  if (out_dtype != PICO_BF16 && out_dtype != PICO_F32)
    return fail(PICO_ERR_DTYPE, "%s: out dtype code %d not supported", fn, out_dtype);
  if (merge && out_dtype != PICO_F32) return fail(PICO_ERR_DTYPE, "%s: merge needs an fp32 running out", fn);
  FwdParams p;
  p.a = make_params(desc, q, nullptr, nullptr);
  if (int rc = set_chunks(fn, desc, kv, p.a, desc->B > 0 && desc->Sq > 0 && desc->Sk > 0)) return rc;
  if (desc->B == 0 || desc->Sq == 0) return PICO_OK;
  if (!q || !out || !lse) return fail(PICO_ERR_NULL, "%s: q, out and lse are required", fn);
  if (!aligned16(q) || !aligned16(out) || !aligned16(q_rot))
    return fail(PICO_ERR_ALIGN, "%s: q, out and q_rot must be 16-byte aligned", fn);
  p.out = out;
  p.lse = lse;
  p.out_f32 = out_dtype == PICO_F32;
  p.merge = merge != 0;
  p.rope = RopeArgs{nullptr, nullptr, 0, 0, 0, 0};
  p.q_rot = nullptr;
  p.qrs[0] = p.qrs[1] = p.qrs[2] = 0;
  if (rope) {
    if (q_pos_offset < 0) return fail(PICO_ERR_SHAPE, "%s: q_pos_offset=%d must be >= 0", fn, q_pos_offset);
    if (int rc = check_rope_tables(fn, rope, desc->D, static_cast<int64_t>(q_pos_offset) + desc->Sq - 1)) return rc;
    p.rope = RopeArgs{rope->cos, rope->sin, rope->pitch, rope->dtype == PICO_F32, q_pos_offset, 0};
    if (q_rot) {
      if (!q_rot_stride) return fail(PICO_ERR_NULL, "%s: q_rot needs its strides", fn);
      for (int i = 0; i < 3; ++i) {
        if (q_rot_stride[i] < 0 || q_rot_stride[i] % 8 != 0)
          return fail(PICO_ERR_STRIDE, "%s: q_rot strides must be non-negative multiples of 8 elements", fn);
        p.qrs[i] = q_rot_stride[i];
      }
      if (!rows_disjoint(q_rot_stride, desc->B, desc->Hq, desc->Sq, desc->D))
        return fail(PICO_ERR_STRIDE, "%s: q_rot strides make rows overlap (every stride must span what lies inside it)", fn);
      p.q_rot = static_cast<__bf16*>(q_rot);
    }
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  const FwdPlan& plan = plan_fwd(p.a, desc->D);
  p.a.pieces = Pieces{workspace && ws_bytes >= plan.ws_bytes ? plan.len : 0, workspace};
  int rc;
  if (desc->D == 64) {
    if (plan.kernel == FwdPlan::kWaves8) rc = launch<64, 1, 8, 64>(p, s);
    else if (plan.kernel == FwdPlan::kWaves4) rc = launch<64, 1, 4, 64>(p, s);
    else if (plan.kernel == FwdPlan::kSplit8) rc = launch<64, 1, 8, 128, 2>(p, s);
    else rc = launch<64, 1, 4, 128, 2>(p, s);
  } else {
    rc = plan.kernel == FwdPlan::kWaves8 ? launch<128, 1, 8, 64>(p, s) : launch<128, 1, 4, 64>(p, s);
  }
  if (rc) return rc;
  return check_launch(fn);
}

pico_kv_chunks one_chunk(const pico_attn_desc* desc, const void* k, const void* v) {
  pico_kv_chunks kv = {};
  kv.count = 1;
  kv.chunk_len = desc ? desc->Sk : 0;
  kv.k[0] = k;
  kv.v[0] = v;
  return kv;
}

}  // namespace

extern "C" int pico_attn_fwd(const pico_attn_desc* desc, const void* q, const void* k, const void* v, void* out,
                             float* lse, int out_dtype, int merge, void* stream) {
  const pico_kv_chunks kv = one_chunk(desc, k, v);
  return run_fwd("pico_attn_fwd", desc, q, &kv, out, lse, out_dtype, merge, nullptr, 0, nullptr, nullptr, stream);
}

extern "C" int pico_attn_fwd_rope(const pico_attn_desc* desc, const void* q, const void* k_rot, const void* v, void* out,
                                  float* lse, int out_dtype, int merge, const pico_rope_tables* rope, int q_pos_offset,
                                  void* q_rot, const int64_t* q_rot_stride, void* stream) {
  if (!rope) return fail(PICO_ERR_NULL, "pico_attn_fwd_rope: the tables are required");
  const pico_kv_chunks kv = one_chunk(desc, k_rot, v);
  return run_fwd("pico_attn_fwd_rope", desc, q, &kv, out, lse, out_dtype, merge, rope, q_pos_offset, q_rot, q_rot_stride, stream);
}

namespace {

// the plan for a descriptor without its operands; nullptr: there is nothing to launch
const FwdPlan* plan_fwd(const pico_attn_desc* desc, int chunk_count) {
  if (!desc || chunk_count < 1 || (desc->D != 64 && desc->D != 128) || desc->B <= 0 || desc->Hq <= 0 || desc->Sq <= 0 || desc->Sk <= 0) return nullptr;
  AttnParams a = make_params(desc, nullptr, nullptr, nullptr);
  a.kv.count = chunk_count;
  a.kv.len = desc->Sk / chunk_count;
  return &plan_fwd(a, desc->D);
}

}  // namespace

extern "C" int64_t pico_attn_fwd_workspace_bytes(const pico_attn_desc* desc, int chunk_count) {
  const FwdPlan* plan = plan_fwd(desc, chunk_count);
  return plan ? plan->ws_bytes : 0;
}

extern "C" int pico_attn_fwd_plan(const pico_attn_desc* desc, int chunk_count, int32_t* out) {
  if (!out) return fail(PICO_ERR_NULL, "pico_attn_fwd_plan: the plan is NULL");
  const FwdPlan* plan = plan_fwd(desc, chunk_count);
  if (!plan) return fail(PICO_ERR_SHAPE, "pico_attn_fwd_plan: no launch for this descriptor");
  out[0] = plan->kernel == FwdPlan::kWaves8 || plan->kernel == FwdPlan::kSplit8 ? 8 : 4;
  out[1] = plan->kernel == FwdPlan::kSplit4 || plan->kernel == FwdPlan::kSplit8 ? 2 : 1;
  out[2] = plan->len;
  return PICO_OK;
}

extern "C" int pico_attn_fwd_chunks_ws(const pico_attn_desc* desc, const void* q, const pico_kv_chunks* kv, void* out,
                                       float* lse, int out_dtype, int merge, const pico_rope_tables* rope, int q_pos_offset,
                                       void* q_rot, const int64_t* q_rot_stride, void* workspace, int64_t workspace_bytes, void* stream) {
  if (!aligned16(workspace)) return fail(PICO_ERR_ALIGN, "pico_attn_fwd_chunks_ws: the workspace must be 16-byte aligned");
  return run_fwd("pico_attn_fwd_chunks_ws", desc, q, kv, out, lse, out_dtype, merge, rope, q_pos_offset, q_rot, q_rot_stride, stream,
                 static_cast<float*>(workspace), workspace_bytes);
}

extern "C" int pico_attn_fwd_chunks(const pico_attn_desc* desc, const void* q, const pico_kv_chunks* kv, void* out,
                                    float* lse, int out_dtype, int merge, const pico_rope_tables* rope, int q_pos_offset,
                                    void* q_rot, const int64_t* q_rot_stride, void* stream) {
  return run_fwd("pico_attn_fwd_chunks", desc, q, kv, out, lse, out_dtype, merge, rope, q_pos_offset, q_rot, q_rot_stride, stream);
}
