// Attention backward for gfx950 (MFMA bf16), split into two kernels so that no gradient needs atomics:
//
//  dK/dV kernel: one workgroup owns 128 keys of one kv head (32 per wave), keeps their K / V fragments and
//    the dK / dV accumulators in registers, and walks over the 64-query tiles (and the query heads of a
//    GQA group) that can see those keys:
//      S = Q K^T, dP = dO V^T   (C tile: lane = key, registers = queries)
//      P = exp2(S*c - lse*log2e),  dS = P * (dP - delta)
//      dV += P^T dO,  dK += dS^T Q   (P / dS feed the MFMA straight from registers as A operands; dO and Q
//                                     come from the row-major LDS tiles through transposing reads)
//  dQ kernel: one workgroup owns 32 queries per wave, keeps Q / dO fragments, lse and delta in registers and
//    walks over the K/V tiles like the forward kernel, in the transposed orientation (lane = query):
//      S^T = K Q^T, dP^T = V dO^T,  dS^T = P^T * (dP^T - delta)  (lse / delta are per-lane scalars)
//      dQ^T += K^T dS^T            (dS^T goes from the C registers into the B operand; K^T is read from the
//                                   row-major K tile through transposing LDS reads)
//
// Recomputing S and dP in the second kernel costs 2 of 7 MFMA products; a single-kernel version that
// accumulated dQ with fp32 atomics was bound by the atomic rate of the memory system (measured).
#include "attn_bwd.h"

#include <type_traits>

namespace pico {
namespace {

// =====================================================================================  dK / dV
// QS > 1: eight waves instead of four, QS of them own the same 32 keys and split every query tile between them, one
// 32-query sub-block each, with accumulators of their own that are added through LDS at the end of the key tile.
//   QS 2 (waves w and w + 4, which share a SIMD): a wave holds one sub-block's S / dP tiles instead of two, which is what
//     lets the head_dim 128 kernel fit 256 registers, i.e. two waves per SIMD.
//   QS 4: for launches that leave most CUs idle, whose time is that of one workgroup's chain of trips: twice the workgroups
//     (64 keys each), and a trip takes 128 queries in the time of 32.
// QS > 1: K fragments (of D / 16) that stay in registers; the others are read from LDS.  As many as fit (two of V beside them do not):
// 4 -> 7 with the registers that staging the tiles took, 3 % at B1 H32 S4096.
constexpr int kSplitKRegs = 7;

template <int D, int QS>
struct KvCfg {
  static constexpr bool kSplit = QS > 1;
  static constexpr int NW = kSplit ? 8 : 4;
  static constexpr int kKeyWaves = kSplit ? NW / QS : 4;   // waves that own different keys
  static constexpr int kThreads = 64 * NW;
  static constexpr int BN = 32 * kKeyWaves;  // keys per workgroup
  static constexpr int BM = QS > 2 ? 32 * QS : 64;   // queries per trip
  // Q and dO tiles are filled by loads that go to LDS directly and lie as TileLayout says.  (The loop is paced by LDS reads and their
  // latency, the matrix cores are busy for half of it: without the LDS writes and with more of K in registers B1 H32 S4096 D128
  // 281 -> 271 us, H32/8 S8192 1000 -> 950; at head_dim 64, which needs the constant distances of TileLayout for it, 244 -> 220 registers
  // and, with dQ, B1 H32 S4096 252 -> 248.5, B8 H32/8 S512 83.8 -> 81, B3 H9/3 S777 41.3 -> 40.2.)
  static constexpr int kTileElems = TileLayout<D>::bytes(BM) / 2;      // one tile
  static constexpr int kVecPerRow = D / 8;
  static constexpr int kQLoads = BM * kVecPerRow / kThreads;
  static constexpr int kBufElems = 2 * kTileElems;                     // Q + dO tile of one stage (bf16)
  static constexpr size_t kBufBytes = kBufElems * sizeof(__bf16) + 2 * BM * sizeof(float);
  static constexpr size_t kTileBytes = 2 * kBufBytes;  // the two Q / dO tile buffers
  // the K and V fragments of the key waves pass through LDS behind the tile buffers, one after the other; QS > 1: both stay there
  // instead of in registers
  static constexpr size_t kKvBytes = static_cast<size_t>(kKeyWaves) * (kSplit ? 2 : 1) * WaveTile<D>::kRegionBytes;
  static constexpr size_t kLdsBytes = kTileBytes + kKvBytes;
  static constexpr int kPerCu = kSplit ? 1 : 2;         // workgroups that share a CU
  static_assert(kPerCu * kLdsBytes <= 160 * 1024, "the workgroups of a CU share its LDS");
  static_assert(NW * kRowRegionBytes <= kTileBytes, "the epilogue reuses the tile buffers");
  // QS > 1: one accumulator set (D/32 x 16 registers x 64 lanes of fp32) of every wave but the key waves' first passes through LDS at a time
  static constexpr size_t kExchangeBytes = static_cast<size_t>(D / 32) * 16 * 64 * 4;
  static_assert(!kSplit || (QS - 1) * kKeyWaves * kExchangeBytes <= kTileBytes, "the exchange reuses the tile buffers");
};

// (per head_dim, where the launch is not tiny)
template <int D> constexpr int kUsualSplit = D == 128 ? 2 : 1;

// the rows of dK (kDk) and / or dV (kDv) that a wave's accumulators hold: 32 keys from row `row0` of their chunk, position
// `key0`, through the wave's piece of LDS.  bf16 gradients are written with streaming stores: nothing on this GPU reads them
// back soon, and lines left dirty in L2 are only written back when the kernel ends.
template <int D, bool kDk, bool kDv>
__device__ __forceinline__ void dkdv_store(const BwdParams& p, unsigned char* region, f32x16 (&dk_acc)[D / 32], f32x16 (&dv_acc)[D / 32],
                                           int chunk, int b, int hkv, int row0, int key0, int lane) {
  const AttnParams& a = p.a;
  const int n = lane % 32, h = lane / 32;
  const int rows_live = a.kv.len - row0;
  const int64_t off = b * p.dks[0] + hkv * p.dks[1] + static_cast<int64_t>(row0) * p.dks[2];
  // gradient w.r.t. the un-rotated k: rotate the lane's row of dK back (linear, so the scale and the sum can follow)
  if (kDk && p.rope.cos != nullptr) rope_unrotate_acc<D>(dk_acc, p.rope, n < rows_live ? p.rope.k_pos0 + key0 + n : 0, h);
  const bool accumulate = (p.dkv_accumulate >> chunk) & 1u;
  if (p.dk_final[chunk] != nullptr) {
    // the last block this chunk's gradient was waiting for: total = travelling sums + this block, rounded once
    const int64_t foff = b * p.dkfs[0] + hkv * p.dkfs[1] + static_cast<int64_t>(row0) * p.dkfs[2];
    if (kDk) wave_store_rows_total<D>(region, dk_acc, a.sm_scale, accumulate ? static_cast<const float*>(p.dk[chunk]) + off : nullptr,
                                      p.dks[2], p.dk_final[chunk] + foff, p.dkfs[2], rows_live, lane);
    if (kDv) wave_store_rows_total<D>(region, dv_acc, 1.f, accumulate ? static_cast<const float*>(p.dv[chunk]) + off : nullptr,
                                      p.dks[2], p.dv_final[chunk] + foff, p.dkfs[2], rows_live, lane);
  } else if (p.dkv_f32) {
    if (kDk) wave_store_rows<D, true>(region, dk_acc, a.sm_scale, static_cast<float*>(p.dk[chunk]) + off, p.dks[2], rows_live, lane, accumulate, false);
    if (kDv) wave_store_rows<D, true>(region, dv_acc, 1.f, static_cast<float*>(p.dv[chunk]) + off, p.dks[2], rows_live, lane, accumulate, false);
  } else {
    if (kDk) wave_store_rows<D, false>(region, dk_acc, a.sm_scale, static_cast<__bf16*>(p.dk[chunk]) + off, p.dks[2], rows_live, lane, false, kStreamGrads);
    if (kDv) wave_store_rows<D, false>(region, dv_acc, 1.f, static_cast<__bf16*>(p.dv[chunk]) + off, p.dks[2], rows_live, lane, false, kStreamGrads);
  }
}

// what a wave of a piece leaves: its dK and dV accumulators
__host__ __device__ constexpr int dkdv_piece_floats(int D) { return 2 * (D / 32) * 16 * kWave; }

template <int D, int QS, bool kCut>
__device__ __forceinline__ void attn_bwd_dkdv_tile(const BwdParams& p, const int ktile, const int part = 0, const int parts = 1) {
  using C = KvCfg<D, QS>;
  using L = TileLayout<D>;
  constexpr bool kSplit = C::kSplit;
  constexpr int BM = C::BM, BN = C::BN;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];

  const AttnParams& a = p.a;
  const int hkv = blockIdx.x % a.Hkv, b = blockIdx.x / a.Hkv;
  const int group = a.Hq / a.Hkv;
  const KeyTile kt_at = key_tile(a.kv, ktile, BN);
  const int key0 = kt_at.key0, chunk = kt_at.chunk, crow0 = kt_at.row0;
  if (p.dk[chunk] == nullptr && p.dk_final[chunk] == nullptr) return;   // this chunk's gradient is not wanted (uniform over the workgroup)
  const int tid = threadIdx.x, wave_id = tid / 64, lane = tid % 64;
  // wave: which 32 keys of the tile; query_sb (QS > 1 only): which 32-query sub-block of every query tile
  const int wave = __builtin_amdgcn_readfirstlane(wave_id % C::kKeyWaves);
  const int query_sb = kSplit ? __builtin_amdgcn_readfirstlane(wave_id / C::kKeyWaves) : 0;
  const int n = lane % 32, h = lane / 32;
  const float c = a.sm_scale * kLog2e;

  const __bf16* kbase = a.kv.k[chunk] + b * a.ks[0] + hkv * a.ks[1];
  const __bf16* vbase = a.kv.v[chunk] + b * a.vs[0] + hkv * a.vs[1];

  // ---- K, V fragments of this wave's 32 keys (B operand: lane = key, 8 consecutive d per k step), fetched
  //      row-major and turned into fragments through the wave's piece of LDS behind the tiles.  The loads are issued here; the first
  //      Q / dO tile's loads follow them further down before anything waits, so that the two latencies overlap.
  bf16x8 kf[D / 16], vf[D / 16];
  constexpr int kKRegs = kSplitKRegs < D / 16 ? kSplitKRegs : D / 16;
  constexpr int kFragPitch = (D + 8) * 2;   // WaveTile's row pitch in bytes
  unsigned char* const split_k = smem_raw + C::kTileBytes + wave * 2 * WaveTile<D>::kRegionBytes;   // (QS > 1 only)
  unsigned char* const split_v = split_k + WaveTile<D>::kRegionBytes;
  const bool loads_kv = !kSplit || query_sb == 0;
  WaveTile<D> kt, vt;
  if (loads_kv) {
    // (the wave index read as a scalar: the buffer windows below are then built in scalar registers; from the
    // per-lane value the compiler cannot tell that they are the same in all lanes and loops over the lanes' values)
    const int row0 = crow0 + 32 * __builtin_amdgcn_readfirstlane(wave);
    kt.issue(make_buffer(kbase + static_cast<int64_t>(row0) * a.ks[2], span_bytes(a.kv.len - row0, a.ks[2], D)), a.ks[2], lane);
    vt.issue(make_buffer(vbase + static_cast<int64_t>(row0) * a.vs[2], span_bytes(a.kv.len - row0, a.vs[2], D)), a.vs[2], lane);
  }

  f32x16 dk_acc[D / 32], dv_acc[D / 32];
#pragma unroll
  for (int db = 0; db < D / 32; ++db)
#pragma unroll
    for (int i = 0; i < 16; ++i) { dk_acc[db][i] = 0.f; dv_acc[db][i] = 0.f; }

  // ---- trip space: (query head of the group) x (query tiles that can see key0)
  const int n_qtiles = (a.Sq + BM - 1) / BM;
  const int qt_start = first_query_tile(a, key0, BM);
  const int tiles_per_head = n_qtiles > qt_start ? n_qtiles - qt_start : 0;
  int n_iter = tiles_per_head * group, head_first = hkv * group, tile_first = qt_start;
  if (kCut && parts > 1) {   // this workgroup's share of the trips
    const int t0 = n_iter * part / parts;
    n_iter = n_iter * (part + 1) / parts - t0;
    const int skip = t0 / tiles_per_head;
    head_first += skip;
    tile_first += t0 - skip * tiles_per_head;
  }

  // Loads of a Q / dO tile straight to LDS, of its lse and delta through registers.  A cursor (wave-uniform:
  // it lives in scalar registers) walks the trip space; stepping to the next tile of the same head is a few
  // scalar adds, only a change of head recomputes addresses.  The per-lane byte offsets are computed once,
  // and rows past Sq read as zeros because they lie past the end of the buffer window.  Every instruction
  // of a wave costs an issue slot, scalar ones included, so the per-trip bookkeeping is kept this small.
  float lreg = 0.f, dreg = 0.f;
  uint32_t q_off[C::kQLoads], do_off[C::kQLoads];
#pragma unroll
  for (int i = 0; i < C::kQLoads; ++i) {
    const int r = L::row(wave_id + C::NW * i, lane), cv = L::column(lane);
    q_off[i] = static_cast<uint32_t>((static_cast<int64_t>(r) * a.qs[2] + cv) * 2);
    do_off[i] = static_cast<uint32_t>((static_cast<int64_t>(r) * a.os[2] + cv) * 2);
  }
  const uint32_t row_off = static_cast<uint32_t>((tid % BM) * 4);
  const uint32_t q_step = static_cast<uint32_t>(BM * a.qs[2] * 2), do_step = static_cast<uint32_t>(BM * a.os[2] * 2);
  struct Cursor {
    int tile, head;                  // query tile within the head, query head
    const char *q, *dout;            // first row of the tile
    const float *lse, *delta;
    uint32_t q_left, do_left, rows_left;  // bytes from there to the end of the head's rows
  } cur;
  auto seek = [&](int head, int tile) {
    const int q0 = tile * BM;
    cur.tile = tile;
    cur.head = head;
    cur.q = reinterpret_cast<const char*>(a.q + b * a.qs[0] + head * a.qs[1] + static_cast<int64_t>(q0) * a.qs[2]);
    cur.dout = reinterpret_cast<const char*>(p.dout + b * a.os[0] + head * a.os[1] + static_cast<int64_t>(q0) * a.os[2]);
    const int64_t row0 = (static_cast<int64_t>(b) * a.Hq + head) * a.Sq + q0;
    cur.lse = p.lse + row0;
    cur.delta = p.delta + row0;
    cur.q_left = span_bytes(a.Sq - q0, a.qs[2], D);
    cur.do_left = span_bytes(a.Sq - q0, a.os[2], D);
    cur.rows_left = static_cast<uint32_t>(a.Sq - q0) * 4u;
  };
  auto advance = [&]() {
    if (cur.tile + 1 == n_qtiles) {
      seek(cur.head + 1, qt_start);
    } else {
      ++cur.tile;
      cur.q += q_step;  cur.q_left -= q_step;
      cur.dout += do_step;  cur.do_left -= do_step;
      cur.lse += BM;  cur.delta += BM;  cur.rows_left -= BM * 4;
    }
  };
  // the tile under the cursor goes to the LDS buffer at buf_off (its lse and delta rows through registers, see stage)
  auto request_tile = [&](uint32_t buf_off) {
    const u32x4 qb = request_window(reinterpret_cast<uint64_t>(cur.q), cur.q_left), dob = request_window(reinterpret_cast<uint64_t>(cur.dout), cur.do_left);
    const uint32_t to = buf_off + __builtin_amdgcn_readfirstlane(wave_id) * L::kPitch;
    each_load<C::kQLoads>([&](auto load) {
      constexpr int i = decltype(load)::value;
      request16_to<i * C::NW * L::kPitch>(to, qb, q_off[i]);
    });
    each_load<C::kQLoads>([&](auto load) {
      constexpr int i = decltype(load)::value;
      request16_to<C::kTileElems * 2 + i * C::NW * L::kPitch>(to, dob, do_off[i]);
    });
  };
  auto prefetch = [&]() {  // lse and delta of the tile under the cursor
    const buffer_rsrc lb = make_buffer(cur.lse, cur.rows_left), db = make_buffer(cur.delta, cur.rows_left);
    lreg = buffer_load_f32(lb, row_off);
    dreg = buffer_load_f32(db, row_off);
  };
  auto stage = [&](uint32_t buf_off) {  // ... (still under the cursor) go to the LDS buffer there
    float* sL = reinterpret_cast<float*>(smem_raw + buf_off + 2 * C::kTileElems * sizeof(__bf16));
    float* sDelta = sL + BM;
    if (tid < BM) {
      // rows past Sq, and rows whose lse is -inf (they saw no key), get lse = +inf so that P = 0
      const bool live = static_cast<uint32_t>(tid) * 4u < cur.rows_left && lreg != -INFINITY;
      sL[tid] = live ? lreg * kLog2e : INFINITY;
      sDelta[tid] = -dreg;   // stored negated: it is loaded straight into the dP accumulator (0 past Sq)
    }
  };

  if (n_iter > 0) {
    seek(head_first, tile_first);
    prefetch();
    request_tile(0);
  }
  if (loads_kv) {
    if constexpr (!kSplit) {
      unsigned char* region = smem_raw + C::kTileBytes + wave * WaveTile<D>::kRegionBytes;
      kt.fragments(region, lane, kf);
      vt.fragments(region, lane, vf);
    } else {
      // the first of the waves that share these keys leaves both tiles in their piece of LDS
      kt.fragments(split_k, lane, kf);
      vt.fragments(split_v, lane, vf);
    }
  }
  if constexpr (QS > 1) {
    __syncthreads();
    // the first few K fragments stay in registers (as many as fit beside the accumulators)
#pragma unroll
    for (int j = 0; j < kKRegs; ++j) kf[j] = *reinterpret_cast<const bf16x8*>(split_k + n * kFragPitch + (16 * j + 8 * h) * 2);
  }
  if (n_iter > 0) stage(0);
  // All loads above are complete from here on (also the first tile, which the barrier publishes).  Saying so
  // keeps the compiler from putting a vmcnt(0) wait in front of the loop's first MFMAs, where it would wait for the
  // NEXT tile on every trip.
  __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);
  __syncthreads();
  // the lane's places in a tile (QS > 1: in the wave's sub-block of it), in its rows' lse and -delta, and (QS > 1) in its keys' K and V
  const int sub_block = query_sb / 2 * L::kRows64 + query_sb % 2 * L::kRows32;
  uint32_t row_first = sub_block + L::row_place(lane), tr_first = sub_block + L::column_place(lane);
  uint32_t lse_first = 2 * C::kTileElems * 2 + (32 * query_sb + 4 * h) * 4, kv_at = C::kTileBytes + wave * 2 * WaveTile<D>::kRegionBytes + n * kFragPitch + 16 * h;
  asm volatile("" : "+v"(row_first), "+v"(tr_first), "+v"(lse_first), "+v"(kv_at));   // (kept, not computed again)
  const int kw0 = key0 + 32 * wave;
  int tile = tile_first;     // query tile (within its head) of the trip being computed
  uint32_t buf_off = 0;      // byte offset of the LDS buffer being read
  // a trip; kOff: every pair of it is visible to this wave
  auto trip = [&](auto off_c, const bool has_next) __attribute__((always_inline)) {
    constexpr bool kOff = decltype(off_c)::value;
    // the next tile travels to the other LDS buffer while this trip computes (that buffer's readers finished before the barrier that
    // ended the last trip)
    if (has_next) {
      advance();
      prefetch();
      request_tile(buf_off ^ static_cast<uint32_t>(C::kBufBytes));
    }
    const int q0 = tile * BM;
    // this lane's places in the tile of this trip and its rows' lse and -delta
    const uint32_t row_lane = buf_off + row_first, tr_lane = buf_off + tr_first, lse_lane = buf_off + lse_first;
    constexpr int kDo = C::kTileElems * 2;   // from Q's tile to dO's
    // 32-query sub-block sb of the wave's (QS > 1: it has one, where its places point)
    auto sub = [](int sb) { return kSplit ? 0 : sb * L::kRows32; };
    auto lse_row = [&](int sb, int j) { return lds_at<f32x4>(lse_lane + (kSplit ? 32 * j : 32 * (4 * sb + j))); };
    auto delta_row = [&](int sb, int j) { return lds_at<f32x4>(lse_lane + (BM * 4 + (kSplit ? 32 * j : 32 * (4 * sb + j)))); };

    // The three phases of a 32-query sub-block (and of the one that a wave with QS 4 has: S beside dP and dV beside dK are two chains at a time, which
    // its few trips wait for.  Product after product, as with QS 2 below, it lost 2 to 4 %: dK/dV of B2 H9/3 S256 11.6 us, 11.9 so;
    // B8 H9/3 S512 18.0, 18.8; B1 H8 S700 11.5, 12.0).
    // products(): S = Q K^T and dP = dO V^T (C tile: lane = key, registers = queries); the dP accumulator starts at
    // -delta of its row (sDelta holds the negated value), so dP - delta comes out of the MFMA.
    auto products = [&](int sb, f32x16& s_acc, f32x16& dp_acc) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const f32x4 d4 = delta_row(sb, j);
#pragma unroll
        for (int t = 0; t < 4; ++t) { s_acc[4 * j + t] = 0.f; dp_acc[4 * j + t] = d4[t]; }
      }
      if constexpr (kSplit) {
        // V comes from LDS as well: the operands are requested kAhead steps before the MFMAs that use them, and the scheduling barriers
        // keep that order (left alone, the compiler reuses one set of registers and every MFMA waits for an LDS round trip)
        constexpr int kSteps = D / 16, kAhead = 2;
        static_assert(QS == 2 || kKRegs == kSteps);
        bf16x8 qa[kSteps], da[kSteps], vb[kSteps];
        auto fetch = [&](int j) {
          qa[j] = lds_at<bf16x8>(row_lane + 32 * j);
          da[j] = lds_at<bf16x8>(row_lane + (kDo + 32 * j));
          vb[j] = lds_at<bf16x8>(kv_at + (WaveTile<D>::kRegionBytes + 32 * j));
        };
#pragma unroll
        for (int j = 0; j < kAhead; ++j) fetch(j);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < kSteps; ++j) {
          if (j + kAhead < kSteps) fetch(j + kAhead);
          s_acc = mfma32(qa[j], kf[j], s_acc);
          dp_acc = mfma32(da[j], vb[j], dp_acc);
          __builtin_amdgcn_sched_barrier(0);
        }
      } else {
#pragma unroll
        for (int s = 0; s < D / 16; ++s) {
          const bf16x8 qa = lds_at<bf16x8>(row_lane + (sub(sb) + 32 * s)), da = lds_at<bf16x8>(row_lane + (kDo + sub(sb) + 32 * s));
          s_acc = mfma32(qa, kf[s], s_acc);
          dp_acc = mfma32(da, vf[s], dp_acc);
        }
      }
    };
    // softmax_grad(): P = exp2(S*c - lse*log2e), dS = P * (dP - delta) [already in the accumulator]; the mask test
    // is compiled in only for sub-blocks on the diagonal.
    auto softmax_grad = [&](int sb, f32x16& s_acc, f32x16& dp_acc, auto mask_c) {
      constexpr bool kMask = decltype(mask_c)::value;
      const int qs_pos = a.q_offset + q0 + 32 * sb;
      const int key_rel = kw0 + n - qs_pos - 4 * h;  // key is masked for row (8j + 4h + t) iff key_rel > 8j + t
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const f32x4 l4 = lse_row(sb, j);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const int i = 4 * j + t;
          float pv = fast_exp2(s_acc[i] * c - l4[t]);
          if constexpr (kMask) {
            if (key_rel > 8 * j + t) pv = 0.f;
          }
          s_acc[i] = pv;
          dp_acc[i] = pv * dp_acc[i];
        }
      }
    };
    // accumulate(): the transposed products dV^T += dO^T P and dK^T += Q^T dS (lane = key, registers = 4 consecutive
    // d, which is what lets the epilogue write whole 16-byte pieces of a row); P / dS come from the registers,
    // dO^T / Q^T from the row-major LDS tiles through transposing reads.
    auto accumulate = [&](int sb, const f32x16& s_acc, const f32x16& dp_acc) {
      if constexpr (kSplit) {
        constexpr int kSlots = 2 * (D / 32), kAhead = 2;
        bf16x8 dof[kSlots], qf[kSlots];
        auto fetch = [&](int idx) {
          const int at = idx / (D / 32) * L::kRows16 + idx % (D / 32) * 64;
          dof[idx] = lds_tr_at<D>(tr_lane + (kDo + at));
          qf[idx] = lds_tr_at<D>(tr_lane + at);
        };
#pragma unroll
        for (int j = 0; j < kAhead; ++j) fetch(j);
        bf16x8 pf = pack8(s_acc, 0), dsf = pack8(dp_acc, 0);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int idx = 0; idx < kSlots; ++idx) {
          const int db = idx % (D / 32);
          if (idx + kAhead < kSlots) fetch(idx + kAhead);
          dv_acc[db] = mfma32(dof[idx], pf, dv_acc[db]);
          dk_acc[db] = mfma32(qf[idx], dsf, dk_acc[db]);
          if (idx + 1 == D / 32) { pf = pack8(s_acc, 8); dsf = pack8(dp_acc, 8); }
          __builtin_amdgcn_sched_barrier(0);
        }
        return;
      }
#pragma unroll
      for (int cc = 0; cc < 2; ++cc) {
        // registers 8cc+4jj+t hold queries 32sb + 16cc + 8jj + 4h + t: dO / Q rows are fetched in that order
        const bf16x8 pf = pack8(s_acc, 8 * cc);
        const bf16x8 dsf = pack8(dp_acc, 8 * cc);
#pragma unroll
        for (int db = 0; db < D / 32; ++db) {
          const uint32_t at = sub(sb) + cc * L::kRows16 + db * 64;
          const bf16x8 dof = lds_tr_at<D>(tr_lane + (kDo + at)), qf = lds_tr_at<D>(tr_lane + at);
          dv_acc[db] = mfma32(dof, pf, dv_acc[db]);
          dk_acc[db] = mfma32(qf, dsf, dk_acc[db]);
        }
      }
    };

    // The same for the one sub-block of a wave with QS 2, product after product: exp2 and P need S alone and are dealt out between
    // the MFMAs of dP, dS between those of dV, so that the vector pipe works in the shadow of every product but S and dK.  Both operands come from
    // LDS: they are requested kAhead MFMAs before the one that uses them, across the products, and the scheduling barriers keep
    // that order (left alone, the compiler reuses one set of registers and every MFMA waits for an LDS round trip).  Forward and backward of a
    // ring of 8 x 4096 rows, 32 / 8 heads of 128, 33.19 -> 32.89 ms, B1 H32 S2048 D128 125.0 -> 124.0 us (nearly all of a wave's vector work
    // is hidden already by the other wave of its SIMD; LDS reads and power remain).
    auto one_block = [&](auto mask_c) __attribute__((always_inline)) {
      constexpr bool kMask = decltype(mask_c)::value;
      constexpr int kSteps = D / 16, kPer = 16 / kSteps, kAhead = 2, kAll = 4 * kSteps;   // (2 * (D / 32) MFMAs of dV and of dK, as many as of S and of dP)
      // (key is masked for row (8j + 4h + t) iff key_rel > 8j + t)
      const int key_rel = a.causal ? kw0 + n - (a.q_offset + q0 + 32 * query_sb) - 4 * h : -1;
      f32x16 s_acc, dp_acc;
      f32x4 l4[4];
      bf16x8 left[kAll], right[2 * kSteps], pf[2], dsf[2];
      auto fetch = [&](int i) {
        const int j = i % kSteps;
        if (i < kSteps) {
          left[i] = lds_at<bf16x8>(row_lane + 32 * j);
          if (j >= kKRegs) right[i] = lds_at<bf16x8>(kv_at + 32 * j);
        } else if (i < 2 * kSteps) {
          left[i] = lds_at<bf16x8>(row_lane + (kDo + 32 * j));
          right[i] = lds_at<bf16x8>(kv_at + (WaveTile<D>::kRegionBytes + 32 * j));
        } else {
          left[i] = lds_tr_at<D>(tr_lane + ((i < 3 * kSteps ? kDo : 0) + j / (D / 32) * L::kRows16 + j % (D / 32) * 64));
        }
      };
#pragma unroll
      for (int i = 0; i < 16; ++i) s_acc[i] = 0.f;
#pragma unroll
      for (int i = 0; i < kAhead; ++i) fetch(i);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < kAll; ++i) {
        const int j = i % kSteps;
        if (i + kAhead < kAll) fetch(i + kAhead);
        const int rows = i - 3 * kSteps / 4;   // lse of the rows whose exp2 is kSteps / 4 MFMAs away
        if (rows >= 0 && rows < kSteps && rows % (kSteps / 4) == 0) l4[rows * 4 / kSteps] = lse_row(query_sb, rows * 4 / kSteps);
        if (i < kSteps) {
          s_acc = mfma32(left[i], j < kKRegs ? kf[j] : right[i], s_acc);
          if (2 * j >= kSteps) {   // dP starts at -delta of its rows
#pragma unroll
            for (int r = (2 * j - kSteps) * 4 / kSteps; r < (2 * j + 2 - kSteps) * 4 / kSteps; ++r) {
              const f32x4 d4 = delta_row(query_sb, r);
#pragma unroll
              for (int t = 0; t < 4; ++t) dp_acc[4 * r + t] = d4[t];
            }
          }
        } else if (i < 2 * kSteps) {
          dp_acc = mfma32(left[i], right[i], dp_acc);
#pragma unroll
          for (int e = j * kPer; e < (j + 1) * kPer; ++e) {
            s_acc[e] = fast_exp2(s_acc[e] * c - l4[e / 4][e % 4]);
            if (kMask && key_rel > 8 * (e / 4) + e % 4) s_acc[e] = 0.f;
          }
          if (2 * (j + 1) == kSteps) pf[0] = pack8(s_acc, 0);
          if (j + 1 == kSteps) pf[1] = pack8(s_acc, 8);
        } else if (i < 3 * kSteps) {
          dv_acc[j % (D / 32)] = mfma32(left[i], pf[j / (D / 32)], dv_acc[j % (D / 32)]);
#pragma unroll
          for (int e = j * kPer; e < (j + 1) * kPer; ++e) dp_acc[e] = s_acc[e] * dp_acc[e];
          if (2 * (j + 1) == kSteps) dsf[0] = pack8(dp_acc, 0);
          if (j + 1 == kSteps) dsf[1] = pack8(dp_acc, 8);
        } else {
          dk_acc[j % (D / 32)] = mfma32(left[i], dsf[j / (D / 32)], dk_acc[j % (D / 32)]);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    };

    if constexpr (QS == 2) {
      const int qs_pos = a.q_offset + q0 + 32 * query_sb;   // position of the sub-block's first query
      if constexpr (kOff) one_block(std::false_type());
      else if (!a.causal || kw0 <= qs_pos + 31) one_block(std::true_type());   // (else every pair is masked; the mask changes nothing off the diagonal)
    } else if constexpr (kOff) {
      // Every pair of this trip is visible to this wave (all trips off the diagonal): straight-line code in an order
      // that lets the wave's own phases overlap -- the matrix pipe works on the second sub-block's S / dP while the
      // vector pipe does the first one's softmax, and on the first one's dV / dK during the second one's softmax.
      f32x16 s0, d0, s1, d1;
      // Four stages; in the middle two, every pair of MFMAs is followed in program order by a share of the OTHER
      // sub-block's softmax arithmetic and by the LDS reads of a later pair.  A wave issues in order: vector
      // instructions that merely follow a batch of MFMAs start when the batch has been issued, i.e. when the matrix
      // pipe is nearly done with it, while an MFMA followed by a few vector instructions keeps both pipes busy
      // (measured on this GPU with one wave per SIMD: 16 MFMAs then 64 fma + 16 exp take 1.63x the time of the same
      // work dealt out one MFMA at a time).  The scheduling barriers pin that order slot by slot (+5 % at head_dim 128,
      // one wave per SIMD; +2.5 % at head_dim 64, where the second wave of the SIMD fills most gaps already).  The
      // head_dim 64 kernel has 256 registers: fragments are fetched one pair ahead and lse rows one slot ahead so
      // that nothing spills.
      constexpr int kPairs = D / 16;        // (S, dP) MFMA pairs per sub-block
      constexpr int kSlots = 2 * (D / 32);  // (dV, dK) MFMA pairs per sub-block
      auto softmax_part = [&](f32x16& s_acc, f32x16& dp_acc, const f32x4 (&l4)[4], int first, int count) {
#pragma unroll
        for (int i = first; i < first + count; ++i) {
          const float pv = fast_exp2(s_acc[i] * c - l4[i / 4][i % 4]);
          s_acc[i] = pv;
          dp_acc[i] = pv * dp_acc[i];
        }
      };
      // stage A: products of sub-block 0
      products(0, s0, d0);
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_setprio(1);
      // stage B: products of sub-block 1, softmax of sub-block 0 between them
      {
        // lse rows of sub-block 0 are fetched a slot ahead of the elements that need them (kPer elements per slot)
        constexpr int kPer = 16 / kPairs;
        f32x4 l4[4];
        l4[0] = lse_row(0, 0);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const f32x4 d4 = delta_row(1, j);
#pragma unroll
          for (int t = 0; t < 4; ++t) { s1[4 * j + t] = 0.f; d1[4 * j + t] = d4[t]; }
        }
        bf16x8 qa[kPairs], da[kPairs];
        auto fetch = [&](int j) {
          qa[j] = lds_at<bf16x8>(row_lane + (sub(1) + 32 * j));
          da[j] = lds_at<bf16x8>(row_lane + (kDo + sub(1) + 32 * j));
        };
        constexpr int kAhead = 1;   // fragment pairs in flight ahead of their MFMAs
#pragma unroll
        for (int j = 0; j < kAhead; ++j) fetch(j);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < kPairs; ++j) {
          if (j + kAhead < kPairs) fetch(j + kAhead);
          if (((j + 1) * kPer) % 4 == 0 && (j + 1) * kPer < 16) l4[(j + 1) * kPer / 4] = lse_row(0, (j + 1) * kPer / 4);
          s1 = mfma32(qa[j], kf[j], s1);
          d1 = mfma32(da[j], vf[j], d1);
          softmax_part(s0, d0, l4, j * kPer, kPer);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      // stage C: dV / dK of sub-block 0, softmax of sub-block 1 between them
      {
        constexpr int kPer = 16 / kSlots;
        f32x4 l4[4];
        l4[0] = lse_row(1, 0);
        bf16x8 dof[kSlots], qf[kSlots];
        auto fetch = [&](int idx) {
          const int cc = idx / (D / 32), db = idx % (D / 32);
          const uint32_t at = cc * L::kRows16 + db * 64;
          dof[idx] = lds_tr_at<D>(tr_lane + (kDo + at));
          qf[idx] = lds_tr_at<D>(tr_lane + at);
        };
        fetch(0);
        bf16x8 pf = pack8(s0, 0), dsf = pack8(d0, 0);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int idx = 0; idx < kSlots; ++idx) {
          const int db = idx % (D / 32);
          if (idx + 1 < kSlots) fetch(idx + 1);
          dv_acc[db] = mfma32(dof[idx], pf, dv_acc[db]);
          dk_acc[db] = mfma32(qf[idx], dsf, dk_acc[db]);
          if (idx + 1 == D / 32) { pf = pack8(s0, 8); dsf = pack8(d0, 8); }
          if (((idx + 1) * kPer) % 4 == 0 && (idx + 1) * kPer < 16) l4[(idx + 1) * kPer / 4] = lse_row(1, (idx + 1) * kPer / 4);
          softmax_part(s1, d1, l4, idx * kPer, kPer);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      // stage D: dV / dK of sub-block 1
      __builtin_amdgcn_s_setprio(0);
      accumulate(1, s1, d1);
    } else {
#pragma unroll
      for (int sbi = 0; sbi < (kSplit ? 1 : BM / 32); ++sbi) {
        const int sb = kSplit ? query_sb : sbi;
        const int qs_pos = a.q_offset + q0 + 32 * sb;       // position of the sub-block's first query
        if (a.causal && kw0 > qs_pos + 31) continue;        // every (query, key) pair of this block is masked
        f32x16 s_acc, dp_acc;
        products(sb, s_acc, dp_acc);
        if (a.causal && kw0 + 31 > qs_pos) softmax_grad(sb, s_acc, dp_acc, std::true_type{});
        else softmax_grad(sb, s_acc, dp_acc, std::false_type{});
        accumulate(sb, s_acc, dp_acc);
      }
    }
    buf_off ^= static_cast<uint32_t>(C::kBufBytes);
    if (has_next) stage(buf_off);
    wait_requests<0>();
    tile = tile + 1 == n_qtiles ? qt_start : tile + 1;
    __syncthreads();  // all waves are done with the buffer just read (refilled in the next trip) and the next tile is visible
  };
  // of every head the tiles on the wave's diagonal come first: loops of their own, as a branch inside the trip had the compiler move
  // the accumulators from registers to registers
  const int seen = kw0 + 31 - a.q_offset - 32 * query_sb;
  const int first_off = a.causal && seen > 0 ? (seen + BM - 1) / BM : 0;
  // (QS 4 has few trips and is better off with less code: B2 H9/3 S256 backward 22.6 -> 22.9 us with two loops)
  for (int it = 0; it < n_iter;) {
    if constexpr (QS > 2) {
      trip(std::false_type(), ++it < n_iter);
      continue;
    }
    for (; it < n_iter && tile < first_off; ++it) trip(std::false_type(), it + 1 < n_iter);
    for (; it < n_iter && tile >= first_off; ++it) trip(std::true_type(), it + 1 < n_iter);
  }

  // ---- epilogue (LDS is free now: the loop ended on a barrier)
  if constexpr (kSplit) {
    // the other waves of these keys hand their sums over, dK then dV (the loop ended on a barrier, or never ran)
    auto place = [&](int sb, int db, int i) { return reinterpret_cast<f32x4*>(smem_raw + ((sb - 1) * C::kKeyWaves + wave) * C::kExchangeBytes) + (db * 4 + i / 4) * 64 + lane; };
#pragma unroll
    for (int which = 0; which < 2; ++which) {
      f32x16 (&acc)[D / 32] = which == 0 ? dk_acc : dv_acc;
      if (query_sb > 0) {
#pragma unroll
        for (int db = 0; db < D / 32; ++db)
#pragma unroll
          for (int i = 0; i < 16; i += 4) *place(query_sb, db, i) = f32x4{acc[db][i], acc[db][i + 1], acc[db][i + 2], acc[db][i + 3]};
      }
      __syncthreads();
      if (query_sb == 0) {
#pragma unroll
        for (int sb = 1; sb < QS; ++sb)
#pragma unroll
          for (int db = 0; db < D / 32; ++db)
#pragma unroll
            for (int i = 0; i < 16; i += 4) {
              const f32x4 o = *place(sb, db, i);
#pragma unroll
              for (int t = 0; t < 4; ++t) acc[db][i + t] += o[t];
            }
      }
      __syncthreads();
    }
  }
  if (!kSplit || query_sb == 0) {
    if (kCut && parts > 1) {   // one piece of several: the sums leave as they are
      float* dst = a.pieces.ws + ((static_cast<int64_t>(blockIdx.x) * gridDim.y + blockIdx.y) * C::kKeyWaves + wave) * dkdv_piece_floats(D);
      put_acc<D / 32>(dst, dk_acc, lane);
      put_acc<D / 32>(dst + dkdv_piece_floats(D) / 2, dv_acc, lane);
      return;
    }
    unsigned char* region = smem_raw + wave * kRowRegionBytes;
    dkdv_store<D, true, true>(p, region, dk_acc, dv_acc, chunk, b, hkv, crow0 + 32 * wave, kw0, lane);
  }
}

// grid = (Hkv * B, key tiles or pairs of key tiles): the x index runs fastest in dispatch order, so all heads of
// key tile 0 (the longest under a causal mask) start first and the short tiles fill in behind them; workgroups
// of one head are a multiple of 8 apart in dispatch order and so share an XCD's L2.  With pair_ktiles a
// workgroup takes tile t and then tile n-1-t: under a causal mask every pair is the same amount of work, so a
// launch whose pairs fill the GPU once ends without a tail of short workgroups and pays the start-up of a
// workgroup (kernel arguments, first loads) half as often.
// kCut: the launch deals its trips out in pieces (see Pieces); a kernel of its own, because the loop of the whole-tile kernel
// is 1 to 2 % slower with the pieces' bookkeeping around it (in the forward and in dQ up to 10 %).
template <int D, int QS, bool kCut>
__device__ __forceinline__ void attn_bwd_dkdv_body(const BwdParams& p) {
  const Arguments<offsetof(BwdParams, dk), offsetof(BwdParams, dk_final), offsetof(BwdParams, dv), offsetof(BwdParams, dv_final), offsetof(BwdParams, dkfs),
                  sizeof(BwdParams) - 4> gradients;
  AttnArguments().arrive();
  gradients.arrive();
  using C = KvCfg<D, QS>;
  if constexpr (kCut) {
    const Piece at = find_piece(blockIdx.y, tiles_before(p.a.kv, p.a.Sk, C::BN), p.a.pieces.len, [&](int i) { return dkdv_trips(p.a, i, C::BN, C::BM); });
    attn_bwd_dkdv_tile<D, QS, true>(p, at.tile, at.part, at.parts);
  } else {
    const int first = blockIdx.y;
    attn_bwd_dkdv_tile<D, QS, false>(p, first);
    const int second = p.pair_ktiles - 1 - first;
    if (p.pair_ktiles > 0 && second != first) {
      __syncthreads();  // the epilogue's pieces of LDS are the next tile's buffers
      attn_bwd_dkdv_tile<D, QS, false>(p, second);
    }
  }
}

// D = 64 fits two workgroups per CU (<= 256 registers per lane), which lets one workgroup's MFMA
// work overlap the other's softmax / LDS phases; D = 128 needs the full register file.
template <bool kCut>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void attn_bwd_dkdv_kernel_d64(const BwdParams p) {
  attn_bwd_dkdv_body<64, 1, kCut>(p);
}
// D = 64, launches of few workgroups: eight waves, four per key block
__global__ __launch_bounds__(512) void attn_bwd_dkdv_few_kernel(const BwdParams p) { attn_bwd_dkdv_body<64, 4, false>(p); }
// D = 128: eight waves, two per key block (see KvCfg), 256 registers each
template <bool kCut>
__global__ __launch_bounds__(512) void attn_bwd_dkdv_kernel_d128(const BwdParams p) {
  attn_bwd_dkdv_body<128, 2, kCut>(p);
}

// The pieces of every cut key tile put together: grid.z 0 sums dK, 1 dV; a wave per 32 keys adds the pieces' accumulators in
// their order and ends as the kernel above does.
template <int D>
__global__ __launch_bounds__(256) void attn_bwd_dkdv_join_kernel(const BwdParams p, const int pieces_per_head) {
  using C = KvCfg<D, kUsualSplit<D>>;
  __shared__ __attribute__((aligned(16))) unsigned char smem_raw[C::kKeyWaves * kRowRegionBytes];
  const AttnParams& a = p.a;
  const int tile = static_cast<int>(blockIdx.y);
  auto trips_of = [&](int i) { return dkdv_trips(a, i, C::BN, C::BM); };
  const int parts = pieces_of(trips_of(tile), a.pieces.len);
  const KeyTile at = key_tile(a.kv, tile, C::BN);
  if (parts == 1 || (p.dk[at.chunk] == nullptr && p.dk_final[at.chunk] == nullptr)) return;
  const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int hkv = blockIdx.x % a.Hkv, b = blockIdx.x / a.Hkv;
  const int64_t first = static_cast<int64_t>(blockIdx.x) * pieces_per_head + first_piece(tile, a.pieces.len, trips_of);
  const float* src = a.pieces.ws + (first * C::kKeyWaves + wave) * dkdv_piece_floats(D) + (blockIdx.z ? dkdv_piece_floats(D) / 2 : 0);
  constexpr int64_t kStep = static_cast<int64_t>(C::kKeyWaves) * dkdv_piece_floats(D);
  f32x16 acc[D / 32];
#pragma unroll
  for (int db = 0; db < D / 32; ++db)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[db][i] = 0.f;
  for (int j = 0; j < parts; ++j) {
    f32x4 raw[D / 32][4];
    get_acc<D / 32>(src + j * kStep, raw, lane);
#pragma unroll
    for (int db = 0; db < D / 32; ++db)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[db][i] += raw[db][i / 4][i % 4];
  }
  unsigned char* region = smem_raw + wave * kRowRegionBytes;
  if (blockIdx.z == 0) dkdv_store<D, true, false>(p, region, acc, acc, at.chunk, b, hkv, at.row0 + 32 * wave, at.key0 + 32 * wave, lane);
  else dkdv_store<D, false, true>(p, region, acc, acc, at.chunk, b, hkv, at.row0 + 32 * wave, at.key0 + 32 * wave, lane);
}

template <int D, bool kCut> struct KvKernel;
template <bool kCut> struct KvKernel<64, kCut> { static constexpr auto fn = &attn_bwd_dkdv_kernel_d64<kCut>; };
template <bool kCut> struct KvKernel<128, kCut> { static constexpr auto fn = &attn_bwd_dkdv_kernel_d128<kCut>; };

// =====================================================================================  dQ
// KS > 1: KS waves share the same 32 queries and each takes one 64-key step of every staged tile (see the forward
// kernel); their dQ partial sums meet in LDS at the end.
template <int D, int NW, int KT, int KS = 1>
struct DqCfg {
  static constexpr int kThreads = 64 * NW;
  static constexpr int kQWaves = NW / KS;
  static constexpr int BM = 32 * kQWaves;  // queries per workgroup (32 per query wave)
  static_assert(NW % KS == 0 && (KS == 1 || KT == 64 * KS), "one 64-key step of every staged tile per key-split wave");
  static constexpr int BN = 64;            // keys per compute step
  static constexpr int kKT = KT;
  static constexpr int kVecPerRow = D / 8;
  static constexpr int kLoads = KT * kVecPerRow / kThreads;
  static constexpr int kSideBytes = TileLayout<D>::bytes(KT);   // a tile's K, or V; two of K, then two of V
  // workgroups that share a CU: the register budget and the plan go by it (at head_dim 128 a lane has 241 of the 256 registers that
  // two leave it; one of 332 registers was slower: 154 drawn launches of under 256 workgroups of eight waves take 0.885 of its time, B1 H12/3
  // S912 24.5 -> 21.9 us)
  static constexpr int kPerCu = NW <= 4 ? 2 : 1;
  static constexpr bool kSmall = D == 128 && NW == 8;   // products of 16 x 16 x 32 (see DqWave)
  // the tiles, double-buffered; the Q / dO fragments pass through LDS behind them where there is room, so that the first tile is
  // requested at once, and through the tile buffers otherwise
  static constexpr size_t kTiles = 4 * kSideBytes, kFragmentBytes = NW * WaveTile<D>::kRegionBytes;
  static constexpr bool kBehind = kPerCu * (kTiles + kFragmentBytes) <= 160 * 1024;
  static constexpr size_t kFragments = kBehind ? kTiles : 0, kLdsBytes = kTiles + (kBehind ? kFragmentBytes : 0);
  static_assert(kFragmentBytes <= kLdsBytes);
  static_assert(kPerCu * kLdsBytes <= 160 * 1024, "the workgroups of a CU share its LDS");
  static_assert(NW * kRowRegionBytes <= kLdsBytes, "the epilogue reuses the tile buffers");
  static_assert(KT % BN == 0 && (KT * kVecPerRow) % kThreads == 0, "tile must split evenly over the threads");
  static constexpr size_t kExchangeBytes = (D / 32) * 16 * 64 * 4;   // a wave's dQ^T accumulators
  static_assert(KS == 1 || NW * kExchangeBytes <= kLdsBytes, "the exchange reuses the tile buffers");
};

// what a wave of a piece leaves: its dQ^T accumulators
__host__ __device__ constexpr int dq_piece_floats(int D) { return (D / 32) * 16 * kWave; }

// A wave's part of dQ: 32 queries, their fragments and sums, and a trip over 64 keys, with products of 32 x 32 x 16 or of 16 x 16 x 32.
// The smaller ones take a seventh less power for the same work (a loop of products alone on normal values 1820 and 2080 TFLOP/s, on
// zeros 2475 and 2440), and as many more issue slots.  So they are for the launches that run at the power limit, eight waves at head_dim 128:
// dQ of B1 H32 S4096 169.1 -> 158.8 us, of 4096 queries and 32768 keys, 32 / 8 heads, 2264 -> 2126, of B8 H32 S1024 without a mask 197 -> 189.
// The others wait for latencies and issue slots: at head_dim 64 level (0.98 to 1.02), four waves at head_dim 128, B1 H12 S1111 without a mask 24.8
// us and 27.7, B1 H8/2 S700 16.9 and 18.7.
//
// A trip is straight-line code in an order that lets the wave's own phases overlap: exp2 needs S alone and is dealt out between the MFMAs of S
// (second 32 keys) and dP, dS between those of dP and dQ (first 32).  The fragments are requested kAhead MFMAs of 32 x 32 x 16 ahead and the scheduling
// barriers keep the order.  Forward and backward, us: B1 H4 S3000 D64 83.0 -> 81.8, B1 H32 S512 D64 49.6 -> 48.5, B1 H4 S3000 D128 85.8 -> 84,
// B2 H32 S1024 D64 71.3 -> 70.5; four MFMAs ahead is level.  Masked trips go by it as well (in the compiler's order every MFMA waited for an LDS
// round trip): dQ alone B1 H8 S293 D64 8.0 -> 7.6, B4 H4/1 S1287 D128 29.2 -> 28.7.
template <int D, bool kDelta>
struct DqOperands {   // a wave's rows of Q, dO and O, on their way
  WaveTile<D> qt, dt, ot;
  __device__ __forceinline__ void issue(const BwdParams& p, int b, int hq, int row0, int lane) {
    const AttnParams& a = p.a;
    const int64_t q_at = b * a.qs[0] + hq * a.qs[1] + static_cast<int64_t>(row0) * a.qs[2], o_at = b * a.os[0] + hq * a.os[1] + static_cast<int64_t>(row0) * a.os[2];
    const buffer_rsrc qb = make_buffer(a.q + q_at, span_bytes(a.Sq - row0, a.qs[2], D)), db = make_buffer(p.dout + o_at, span_bytes(a.Sq - row0, a.os[2], D));
    const buffer_rsrc ob = kDelta ? make_buffer(p.out + o_at, span_bytes(a.Sq - row0, a.os[2], D)) : db;
    qt.issue(qb, a.qs[2], lane);
    dt.issue(db, a.os[2], lane);
    if constexpr (kDelta) ot.issue(ob, a.os[2], lane);
  }
};

template <int D, bool kSmall> struct DqWave;
template <int D>
struct DqWave<D, false> {   // lane = query lane % 32, registers = keys
  using L = TileLayout<D>;
  static constexpr int kSteps = D / 16;
  bf16x8 qf[D / 16], dof[D / 16];
  float lse2, delta;
  int pos, first_key;   // position of the lane's query; the first of its keys of 32
  f32x16 dq[D / 32];
  static __device__ __forceinline__ uint32_t row_place(int lane) { return L::row_place(lane); }
  static __device__ __forceinline__ uint32_t column_place(int lane) { return L::column_place(lane); }
  static __device__ __forceinline__ void clear(f32x16 (&acc)[D / 32]) {
#pragma unroll
    for (int db = 0; db < D / 32; ++db)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[db][i] = 0.f;
  }
  // the fragments of the rows from row0, their lse, and delta = sum_d dO * O (context_parallel.py:145): each half of the wave holds half of
  // a row's columns; with `writes` it goes to memory, for the dK/dV kernel that is launched after this one
  template <bool kDelta>
  __device__ __forceinline__ void load(const BwdParams& p, unsigned char* region, int64_t lse_row0, int b, int hq, int row0, bool writes, int lane) {
    DqOperands<D, kDelta> rows;
    rows.issue(p, b, hq, row0, lane);
    const int qrow = row0 + lane % 32, h = lane / 32;
    const int64_t gi = lse_row0 + qrow;
    pos = p.a.causal ? p.a.q_offset + qrow : 0x7fffff00;   // (past every key)
    first_key = 4 * h;
    const uint32_t left = static_cast<uint32_t>(max(p.a.Sq - row0, 0)) * 4u, at = lane % 32 * 4u;
    const float l = buffer_load_f32(make_buffer(p.lse + lse_row0 + row0, left), at);
    delta = kDelta ? 0.f : buffer_load_f32(make_buffer(p.delta + lse_row0 + row0, left), at);
    rows.qt.fragments(region, lane, qf);
    rows.dt.fragments(region, lane, dof);
    lse2 = qrow < p.a.Sq && l != -INFINITY ? l * kLog2e : INFINITY;   // (a row that saw no key contributes nothing)
    if constexpr (kDelta) {
      bf16x8 of[D / 16];
      rows.ot.fragments(region, lane, of);
      float part = 0.f;
#pragma unroll
      for (int s = 0; s < D / 16; ++s)
#pragma unroll
        for (int e = 0; e < 8; ++e) part += static_cast<float>(dof[s][e]) * static_cast<float>(of[s][e]);
      delta = half_sum(part);
      if (qrow < p.a.Sq && h == 0 && writes) p.delta_w[gi] = delta;
    }
  }
  // the 64 keys from position key0, whose rows lie at the three places (+ kAt); kPlain: none of them is masked, otherwise those past the
  // query and from keys_end on are
  template <uint32_t kAt, bool kPlain>
  __device__ __forceinline__ void trip(uint32_t row_lane, uint32_t v_row_lane, uint32_t tr_lane, int key0, int keys_end, float c) {
    constexpr int kAll = 6 * kSteps, kAhead = 2;
    // (the rows read past a chunk are zero, but P of a zero score need not be finite beside a very negative lse): one compare with a constant per
    // element
    const int last = min(pos, keys_end - 1) - key0 - first_key;
    f32x16 s_acc[2], dp_acc[2];
    bf16x8 from[kAll], dsf[4];
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
      for (int i = 0; i < 16; ++i) { s_acc[mb][i] = 0.f; dp_acc[mb][i] = -delta; }   // dP - delta comes out of the MFMA
    auto fetch = [&](int i) {
      const int j = i % (2 * kSteps), mb = j / kSteps;   // MFMA of its product, 32-key block
      if (i < 4 * kSteps) from[i] = lds_at<bf16x8>((i < 2 * kSteps ? row_lane : v_row_lane) + (kAt + L::rows(32 * mb) + j % kSteps * 32));
      else from[i] = lds_tr_at<D>(tr_lane + (kAt + L::rows(32 * mb) + j % kSteps / (D / 32) * L::kRows16 + j % (D / 32) * 64));
    };
    auto probability = [&](int e) {
      float s = s_acc[e / 16][e % 16];
      if (!kPlain && 32 * (e / 16) + 8 * (e % 16 / 4) + e % 4 > last) s = -INFINITY;   // exp2(-inf) = 0
      s_acc[e / 16][e % 16] = fast_exp2(s * c - lse2);
    };
    auto ds = [&](int e) { dp_acc[e / 16][e % 16] = s_acc[e / 16][e % 16] * dp_acc[e / 16][e % 16]; };
#pragma unroll
    for (int i = 0; i < kAhead; ++i) fetch(i);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < kAll; ++i) {
      const int j = i % (2 * kSteps), mb = j / kSteps, s = j % kSteps;
      if (i + kAhead < kAll) fetch(i + kAhead);
      if (i < 2 * kSteps) s_acc[mb] = mfma32(from[i], qf[s], s_acc[mb]);
      else if (i < 4 * kSteps) dp_acc[mb] = mfma32(from[i], dof[s], dp_acc[mb]);
      else dq[j % (D / 32)] = mfma32(from[i], dsf[j / (D / 32)], dq[j % (D / 32)]);
      if (i >= kSteps && i < 4 * kSteps) {
#pragma unroll
        for (int e = (i - kSteps) * 32 / (3 * kSteps); e < (i + 1 - kSteps) * 32 / (3 * kSteps); ++e) probability(e);
      }
      if (i >= 3 * kSteps && i < 5 * kSteps) {
#pragma unroll
        for (int e = (i - 3 * kSteps) * 16 / kSteps; e < (i + 1 - 3 * kSteps) * 16 / kSteps; ++e) ds(e);
        const int done = (i + 1 - 3 * kSteps) * 16 / kSteps;
        if (done % 8 == 0) dsf[done / 8 - 1] = pack8(dp_acc[(done / 8 - 1) / 2], (done / 8 - 1) % 2 * 8);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
};
template <int D>
struct DqWave<D, true> {   // lane = queries lane % 16 and 16 + lane % 16, registers = keys group_row(lane / 16) ..+3 of every 16
  using L = TileLayout<D>;
  static constexpr int kSteps = D / 16;
  bf16x8 qf[2][D / 32], dof[2][D / 32];
  float lse2[2], delta[2];
  int pos, first_key;   // position of the lane's first query; the first of its keys of 16
  f32x4 dq[D / 16][2];
  static __device__ __forceinline__ uint32_t row_place(int lane) { return L::row_place16(lane); }
  static __device__ __forceinline__ uint32_t column_place(int lane) { return L::column_place16(lane); }
  static __device__ __forceinline__ void clear(f32x4 (&acc)[D / 16][2]) {
#pragma unroll
    for (int db = 0; db < D / 16; ++db)
#pragma unroll
      for (int qb = 0; qb < 2; ++qb) acc[db][qb] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  template <bool kDelta>   // (a quarter of a row's columns in each lane of it)
  __device__ __forceinline__ void load(const BwdParams& p, unsigned char* region, int64_t lse_row0, int b, int hq, int row0, bool writes, int lane) {
    DqOperands<D, kDelta> rows;
    rows.issue(p, b, hq, row0, lane);
    const int qrow = row0 + lane % 16;
    const int64_t gi = lse_row0 + qrow;
    pos = p.a.causal ? p.a.q_offset + qrow : 0x7fffff00;
    first_key = L::group_row(lane / 16);
    const uint32_t left = static_cast<uint32_t>(max(p.a.Sq - row0, 0)) * 4u;
    const buffer_rsrc lb = make_buffer(p.lse + lse_row0 + row0, left), eb = make_buffer((kDelta ? p.lse : p.delta) + lse_row0 + row0, left);
    float l[2];
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) {
      l[qb] = buffer_load_f32(lb, (lane % 16 + 16 * qb) * 4u);
      delta[qb] = kDelta ? 0.f : buffer_load_f32(eb, (lane % 16 + 16 * qb) * 4u);
    }
    rows.qt.fragments16(region, lane, qf);
    rows.dt.fragments16(region, lane, dof);
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) lse2[qb] = qrow + 16 * qb < p.a.Sq && l[qb] != -INFINITY ? l[qb] * kLog2e : INFINITY;
    if constexpr (kDelta) {
      bf16x8 of[2][D / 32];
      rows.ot.fragments16(region, lane, of);
#pragma unroll
      for (int qb = 0; qb < 2; ++qb) {
        float part = 0.f;
#pragma unroll
        for (int s = 0; s < D / 32; ++s)
#pragma unroll
          for (int e = 0; e < 8; ++e) part += static_cast<float>(dof[qb][s][e]) * static_cast<float>(of[qb][s][e]);
        delta[qb] = group_sum(part);
        if (qrow + 16 * qb < p.a.Sq && lane < 16 && writes) p.delta_w[gi + 16 * qb] = delta[qb];
      }
    }
  }
  template <uint32_t kAt, bool kPlain>
  __device__ __forceinline__ void trip(uint32_t row_lane, uint32_t v_row_lane, uint32_t tr_lane, int key0, int keys_end, float c) {
    constexpr int kAll = 6 * kSteps, kAhead = 2;
    int last[2];
    f32x4 s_acc[4][2], dp_acc[4][2];   // [16 keys][16 queries]
    bf16x8 from[kAll], dsf[4];
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) {
      last[qb] = min(pos + 16 * qb, keys_end - 1) - key0 - first_key;
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) {
        s_acc[kb][qb] = f32x4{0.f, 0.f, 0.f, 0.f};
        dp_acc[kb][qb] = f32x4{-delta[qb], -delta[qb], -delta[qb], -delta[qb]};   // dP - delta comes out of the MFMA
      }
    }
    // Fragment i of S and dP: which 16 keys, which 32 columns.  S goes through one 16 keys after the other, so that exp2 can begin early; dP, which dS
    // waits for by 32 keys, takes two 16 keys of the same columns in turn and the queries of the second the other way round, so that a sum's products are four
    // MFMAs apart instead of two and the fragment of dO stays (in the second launch below 1.5 % fewer cycles).  us, dP like S and so: B1 H32 S4096 161.0, 160.1; 4096 queries and 32768 keys with 32 / 8 heads
    // 2180, 2152; B8 H32 S1024 no mask 181.3, 179.5; 17 launches, 14 of them drawn, 0.981 to 1.001 of the time, 0.993 over all.  (S like dP, with exp2 six
    // MFMAs later, 2134.8 -> 2146.1 in the second of these; the queries of dQ's products there and back, level.)
    auto keys_of = [](int i) constexpr { return i < 2 * kSteps ? i / (D / 32) : i % (2 * kSteps) / kSteps * 2 + i % 2; };
    auto step_of = [](int i) constexpr { return i < 2 * kSteps ? i % (D / 32) : i % kSteps / 2; };
    auto fetch = [&](int i) {
      const int j = i % (2 * kSteps);   // fragment of its product
      if (i < 4 * kSteps) from[i] = lds_at<bf16x8>((i < 2 * kSteps ? row_lane : v_row_lane) + (kAt + L::rows(32 * (keys_of(i) / 2)) + keys_of(i) % 2 * L::kRows16 + L::column16(step_of(i)) * 2));
      else from[i] = lds_tr16_at<D>(tr_lane + (kAt + L::rows(32 * (j / kSteps)) + j % kSteps * 32));
    };
    // element e of a lane's 32: 16 keys, 16 queries, key
    auto probability = [&](int e) {
      const int kb = e / 8, qb = e / 4 % 2;
      float s = s_acc[kb][qb][e % 4];
      if (!kPlain && 16 * kb + e % 4 > last[qb]) s = -INFINITY;   // exp2(-inf) = 0
      s_acc[kb][qb][e % 4] = fast_exp2(s * c - lse2[qb]);
    };
    auto ds = [&](int e) {
      const int kb = e / 8, qb = e / 4 % 2;
      dp_acc[kb][qb][e % 4] = s_acc[kb][qb][e % 4] * dp_acc[kb][qb][e % 4];
    };
#pragma unroll
    for (int i = 0; i < kAhead; ++i) fetch(i);
    __builtin_amdgcn_sched_barrier(0);
    each_load<2 * kAll>([&](auto which) __attribute__((always_inline)) {   // the MFMAs: every fragment has one for each 16 queries
      constexpr int m = decltype(which)::value, i = m / 2, j = i % (2 * kSteps), kb = keys_of(i), s = step_of(i);
      constexpr int qb = i >= 2 * kSteps && i < 4 * kSteps && i % 2 ? 1 - m % 2 : m % 2;
      if constexpr (m % 2 == 0 && i + kAhead < kAll) fetch(i + kAhead);
      if constexpr (i < 2 * kSteps) s_acc[kb][qb] = mfma16(from[i], qf[qb][s], s_acc[kb][qb]);
      else if constexpr (i < 4 * kSteps) dp_acc[kb][qb] = mfma16(from[i], dof[qb][s], dp_acc[kb][qb]);
      else dq[j % kSteps][qb] = mfma16(from[i], dsf[j / kSteps * 2 + qb], dq[j % kSteps][qb]);
      // exp2 from the first 16 keys' S on, dS from the first 32 keys' dP on
      constexpr int kExp = kSteps, kDs = 6 * kSteps, kEnd = 19 * kSteps / 2;
      if constexpr (m >= kExp && m < kDs) {
#pragma unroll
        for (int e = (m - kExp) * 32 / (kDs - kExp); e < (m + 1 - kExp) * 32 / (kDs - kExp); ++e) probability(e);
      } else if constexpr (m >= kDs && m < kEnd) {
        constexpr int from_e = (m - kDs) * 32 / (kEnd - kDs), to_e = (m + 1 - kDs) * 32 / (kEnd - kDs);
#pragma unroll
        for (int e = from_e; e < to_e; ++e) ds(e);
        each_load<4>([&](auto operand) __attribute__((always_inline)) {   // 32 keys, 16 queries
          constexpr int at = decltype(operand)::value, last_e = at / 2 * 16 + 12 + at % 2 * 4;   // (all before it and its 4 are there)
          if constexpr (from_e < last_e && to_e >= last_e) dsf[at] = pack8(dp_acc[at / 2 * 2][at % 2], dp_acc[at / 2 * 2 + 1][at % 2]);
        });
      }
      __builtin_amdgcn_sched_barrier(0);
    });
  }
};
// the wave's 32 dQ rows leave through its piece of LDS as whole lines
__device__ __forceinline__ int dq_position(const BwdParams& p, int row) { return row < p.a.Sq ? p.rope.q_pos0 + row : 0; }
template <int D>
__device__ __forceinline__ void dq_unrotate(const BwdParams& p, f32x16 (&dq)[D / 32], int row0, int lane) {
  rope_unrotate_acc<D>(dq, p.rope, dq_position(p, row0 + lane % 32), lane / 32);
}
template <int D>
__device__ __forceinline__ void dq_unrotate(const BwdParams& p, f32x4 (&dq)[D / 16][2], int row0, int lane) {
  const int pos[2] = {dq_position(p, row0 + lane % 16), dq_position(p, row0 + 16 + lane % 16)};
  rope_unrotate_acc<D>(RowPair<0, D / 16, 2>{dq}, p.rope, pos, lane);
}
template <int N>
__device__ __forceinline__ const f32x16 (&rows_of(f32x16 (&acc)[N]))[N] { return acc; }
template <int N>
__device__ __forceinline__ RowPair<0, N, 2> rows_of(f32x4 (&acc)[N][2]) { return {acc}; }
template <int D, typename Acc>
__device__ __forceinline__ void dq_store(const BwdParams& p, unsigned char* region, Acc& dq, int b, int hq, int row0, int lane) {
  const AttnParams& a = p.a;
  const int64_t off = b * p.dqs[0] + hq * p.dqs[1] + static_cast<int64_t>(row0) * p.dqs[2];
  if (p.rope.cos != nullptr) dq_unrotate<D>(p, dq, row0, lane);
  if (p.dq_f32)
    wave_store_rows<D, true>(region, rows_of(dq), a.sm_scale, static_cast<float*>(p.dq) + off, p.dqs[2], a.Sq - row0, lane, p.dq_accumulate, false);
  else
    wave_store_rows<D, false>(region, rows_of(dq), a.sm_scale, static_cast<__bf16*>(p.dq) + off, p.dqs[2], a.Sq - row0, lane, false, kStreamGrads);
}

template <int D, int NW, int KT, bool kDelta, int KS, bool kCut>
__global__ __launch_bounds__(64 * NW, (DqCfg<D, NW, KT, KS>::kPerCu * NW / 4)) void attn_bwd_dq_kernel(const BwdParams p) {
  using C = DqCfg<D, NW, KT, KS>;
  using L = TileLayout<D>;
  using W = DqWave<D, C::kSmall>;
  constexpr int BM = C::BM, BN = C::BN;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];

  const Arguments<offsetof(BwdParams, dq), offsetof(BwdParams, dqs), sizeof(BwdParams) - 4> late;   // (what the epilogue uses)
  AttnArguments().arrive();
  const AttnParams& a = p.a;
  const int n_qtiles = (a.Sq + BM - 1) / BM;
  // same dispatch order as the forward kernel: every head's last (longest) query tile first
  Piece piece = {static_cast<int>(blockIdx.y), 0, 1};
  if (kCut && a.pieces.len > 0)
    piece = find_piece(blockIdx.y, n_qtiles, a.pieces.len, [&](int i) { return query_tile_trips(a, n_qtiles - 1 - i, BM, KT); });
  const int qtile = n_qtiles - 1 - piece.tile;
  const int hq = blockIdx.x % a.Hq, b = blockIdx.x / a.Hq;
  const int hkv = hq / (a.Hq / a.Hkv);
  const int q0 = qtile * BM;
  const int tid = threadIdx.x, lane = tid % 64;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);   // (a scalar: the buffer windows below are built in scalar registers)
  const int qw = wave % C::kQWaves, ks = wave / C::kQWaves;   // which queries, which 64-key step of a staged tile
  const float c = a.sm_scale * kLog2e;

  // ---- key range of this query tile
  const int q_hi = (q0 + BM < a.Sq ? q0 + BM : a.Sq);
  int kv_end = a.Sk;
  if (a.causal) {
    const int vis = a.q_offset + q_hi;
    kv_end = vis < a.Sk ? vis : a.Sk;
    if (kv_end < 0) kv_end = 0;
  }
  int t_first = 0, ntiles = kCut ? tiles_before(a.kv, kv_end, KT) : (kv_end + KT - 1) / KT;
  if (kCut && piece.parts > 1) {
    t_first = ntiles * piece.part / piece.parts;
    ntiles = ntiles * (piece.part + 1) / piece.parts - t_first;
  }

  // K / V tiles go straight to LDS, like in the forward kernel (rows past Sk read as zeros).  Besides the LDS writes at the end
  // of a trip this saves the registers of the tile: B1 H32 S4096 D128 212 -> 195 us, H32/8 S8192 720 -> 669; level at head_dim 64.
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

  // ---- the wave's queries: Q and dO fragments (B operands: fetched row-major, turned into fragments through the
  //      wave's piece of LDS; the tile buffers are filled only after the barrier below), lse and delta
  W w;
  w.template load<kDelta>(p, smem_raw + C::kFragments + wave * WaveTile<D>::kRegionBytes, (static_cast<int64_t>(b) * a.Hq + hq) * a.Sq, b, hq,
                          q0 + qw * 32, ks == 0 && piece.part == 0, lane);
  W::clear(w.dq);

  if constexpr (!C::kBehind) {
    __syncthreads();  // every wave has its Q / dO fragments: the tile buffers may be filled
    if (ntiles > 0) request_tile(0);
  }
  // While the first tile is on its way: the lane's places in the K and V tiles, and how many tiles the wave's queries see (they come
  // first, with the others it only helps, see the forward kernel).  The tiles that no mask touches have trips of their own, in loops of
  // their own, for the same reason.
  const int blk_q_lo = a.q_offset + q0 + qw * 32;  // position of this wave's first query
  const int see = max(min(a.causal ? blk_q_lo + 32 : kv_end, kv_end) - BN * ks, 0);
  int mine = min(max((kCut ? tiles_before(a.kv, see, KT) : (see + KT - 1) / KT) - t_first, 0), ntiles);
  // the wave's step of a tile is unmasked up to this first key of the tile, where keys end at `end`
  auto unmasked_end = [&](int end) { return min(a.causal ? blk_q_lo + 1 : end, end) - BN * (ks + 1); };
  int plain = unmasked_end(a.Sk);
  plain = plain >= 0 ? min(plain / KT + 1, mine) : 0;
  uint32_t row_at = W::row_place(lane), v_row_at = 2 * C::kSideBytes + W::row_place(lane), tr_at = W::column_place(lane);
  asm volatile("" : "+v"(row_at), "+v"(v_row_at), "+v"(tr_at), "+s"(mine), "+s"(plain));   // (kept, not computed again in front of the reads)
  late.arrive();
  // all loads so far are complete, the first tile among them (the barrier publishes it); stating it also keeps a
  // vmcnt(0) wait, which would hit the next tile's requests, out of the loop body
  __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);
  __syncthreads();

  // a trip on the LDS buffer `parity`, a constant, so that a lane's addresses are the same in every trip (kCut, whose runs of tiles begin
  // anywhere: on buffer t % 2)
  auto trip = [&](auto parity, auto plain_c, int t) __attribute__((always_inline)) {
    constexpr uint32_t kAt = decltype(parity)::value * C::kSideBytes;
    const uint32_t moved = kCut ? t % 2 * C::kSideBytes : 0;
    constexpr bool kPlain = decltype(plain_c)::value;   // no key of the wave's step is masked
    static_assert(kAt + L::rows(KT - 32) + L::kRows16 + L::kRows8 + 2 * D <= 65535, "offsets of LDS reads");
    const int tile_key0 = kCut ? pos.key0 : t * KT, keys_end = kCut ? pos.end : a.Sk;
    if constexpr (kCut) pos.next(a.kv, KT);
    if (t + 1 < ntiles) request_tile(kCut ? 1 - t % 2 : 1 - decltype(parity)::value);
    static_assert(KT == BN * KS && BN == 64);
    const uint32_t step_at = moved + (KS > 1 ? static_cast<uint32_t>(ks) * L::kRows64 : 0);
    w.template trip<kAt, kPlain>(row_at + step_at, v_row_at + step_at, tr_at + step_at, tile_key0 + BN * ks, keys_end, c);
    wait_requests<0>();
    __syncthreads();
  };
  int t = 0;
  if constexpr (kCut) {
    // Chunk after chunk, whose last tile may be a partial one.  (With masked trips alone where chunks end inside tiles, 150 drawn launches took
    // 1.12 of the time at head_dim 64 and 1.07 at 128: B4 H9/3 S1582 of 4 x 1582 keys D64 160.6 -> 139.5 us, B1 H32 S2275 of 4 x 568 45.9 -> 42.4.)
    while (t < mine) {
      int run = unmasked_end(pos.end) - pos.key0;
      run = run >= 0 ? min(t + run / KT + 1, mine) : t;
      if (t >= run) trip(std::integral_constant<int, 0>(), std::false_type(), t++);
      while (t < run) trip(std::integral_constant<int, 0>(), std::true_type(), t++);
    }
  } else {
    while (t < plain) {
      trip(std::integral_constant<int, 0>(), std::true_type(), t++);
      if (t >= plain) break;
      trip(std::integral_constant<int, 1>(), std::true_type(), t++);
    }
    if (t % 2 == 1 && t < mine) trip(std::integral_constant<int, 1>(), std::false_type(), t++);
    while (t < mine) {
      trip(std::integral_constant<int, 0>(), std::false_type(), t++);
      if (t >= mine) break;
      trip(std::integral_constant<int, 1>(), std::false_type(), t++);
    }
  }
  for (; t < ntiles; ++t) {
    if (t + 1 < ntiles) request_tile((t + 1) % 2);
    wait_requests<0>();
    __syncthreads();
  }

  // ---- key split: the partial sums of the waves ks > 0 are added to the wave ks == 0 of the same queries through LDS
  //      (the loop ended on a barrier: the tile buffers are free; the store pieces used below lie in front of the
  //      exchange areas of the ks > 0 waves)
  if constexpr (KS > 1) {
    if (ks > 0) put_acc(reinterpret_cast<float*>(smem_raw + wave * C::kExchangeBytes), w.dq, lane);
    __syncthreads();
    if (ks > 0) return;
#pragma unroll
    for (int j = 1; j < KS; ++j) add_acc(w.dq, reinterpret_cast<const float*>(smem_raw + (qw + j * C::kQWaves) * C::kExchangeBytes), lane);
    static_assert(kRowRegionBytes <= C::kExchangeBytes, "store pieces lie below the exchange areas read above");
  }

  if (kCut && piece.parts > 1) {   // one piece of several: the sums leave as they are
    put_acc(a.pieces.ws + ((static_cast<int64_t>(blockIdx.x) * gridDim.y + blockIdx.y) * C::kQWaves + qw) * dq_piece_floats(D), w.dq, lane);
    return;
  }
  dq_store<D>(p, smem_raw + wave * kRowRegionBytes, w.dq, b, hq, q0 + qw * 32, lane);
}

// The pieces of every cut query tile put together (see attn_bwd_dkdv_join_kernel).
template <int D, int QW, int KT, bool kSmall>
__global__ __launch_bounds__(64 * QW) void attn_bwd_dq_join_kernel(const BwdParams p, const int pieces_per_head) {
  __shared__ __attribute__((aligned(16))) unsigned char smem_raw[QW * kRowRegionBytes];
  const AttnParams& a = p.a;
  constexpr int BM = 32 * QW;
  const int n_qtiles = (a.Sq + BM - 1) / BM, tile = static_cast<int>(blockIdx.y);
  auto trips_of = [&](int i) { return query_tile_trips(a, n_qtiles - 1 - i, BM, KT); };
  const int parts = pieces_of(trips_of(tile), a.pieces.len);
  if (parts == 1) return;
  const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int hq = blockIdx.x % a.Hq, b = blockIdx.x / a.Hq;
  const int64_t first = static_cast<int64_t>(blockIdx.x) * pieces_per_head + first_piece(tile, a.pieces.len, trips_of);
  const float* src = a.pieces.ws + (first * QW + wave) * dq_piece_floats(D);
  constexpr int64_t kStep = static_cast<int64_t>(QW) * dq_piece_floats(D);
  decltype(DqWave<D, kSmall>::dq) dq;
  DqWave<D, kSmall>::clear(dq);
  for (int j = 0; j < parts; ++j) add_acc(dq, src + j * kStep, lane);
  dq_store<D>(p, smem_raw + wave * kRowRegionBytes, dq, b, hq, (n_qtiles - 1 - tile) * BM + wave * 32, lane);
}

// delta[row] = sum_d dO * O, one 16-byte vector of each per lane, D/8 lanes per row.
template <int D, typename TO>
__global__ __launch_bounds__(256) void attn_bwd_preprocess_kernel(const __bf16* __restrict__ dout,
                                                                  const TO* __restrict__ out, float* __restrict__ delta,
                                                                  float* __restrict__ dq_acc, int B, int H, int S,
                                                                  int64_t sb, int64_t sh, int64_t ss) {
  constexpr int LPR = D / 8;  // lanes per row
  const int64_t idx = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  const int64_t rows = static_cast<int64_t>(B) * H * S;
  const int64_t row = idx / LPR;
  const int v = static_cast<int>(idx % LPR);
  float part = 0.f;
  if (row < rows) {
    const int s = static_cast<int>(row % S);
    const int hh = static_cast<int>((row / S) % H);
    const int64_t bb = row / (static_cast<int64_t>(S) * H);
    const int64_t off = bb * sb + hh * sh + s * ss + v * 8;
    float d8[8], o8[8];
    io<__bf16>::load(dout + off, d8);
    if constexpr (sizeof(TO) == 2) {
      io<__bf16>::load(out + off, o8);
    } else {
      float t[4];
      io<float>::load(out + off, t);
#pragma unroll
      for (int e = 0; e < 4; ++e) o8[e] = t[e];
      io<float>::load(out + off + 4, t);
#pragma unroll
      for (int e = 0; e < 4; ++e) o8[4 + e] = t[e];
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) part += d8[e] * o8[e];
    if (dq_acc != nullptr) {
      const f32x4 z = {0.f, 0.f, 0.f, 0.f};
      *reinterpret_cast<f32x4*>(dq_acc + row * D + v * 8) = z;
      *reinterpret_cast<f32x4*>(dq_acc + row * D + v * 8 + 4) = z;
    }
  }
#pragma unroll
  for (int off = LPR / 2; off > 0; off >>= 1) part += __shfl_xor(part, off, kWave);
  if (row < rows && v == 0) delta[row] = part;
}

// How the dK/dV launch is run: key tiles singly, in pairs, or cut into pieces.
struct DkdvPlan {
  bool few = false;    // attn_bwd_dkdv_few_kernel
  bool roles = false;  // attn_bwd_roles.hip
  bool pair = false;
  int len = 0;
  int64_t ws_bytes = 0;
};
template <int D>
DkdvPlan make_dkdv_plan(const AttnParams& a) {
  using C = KvCfg<D, kUsualSplit<D>>;
  DkdvPlan plan;
  const int64_t heads = static_cast<int64_t>(a.Hkv) * a.B;
  const int n_ktiles = tiles_before(a.kv, a.Sk, C::BN);
  // pairs only when they still fill most of the GPU (two workgroups per CU for D = 64, one for D = 128; at D = 64 three
  // quarters of the places are enough: rank 2 of 4 of B4 H32 S1024, 384 pairs, 21.2 -> 20.3 us; with 256 pairs single tiles
  // are up to 30 % faster)
  // Few workgroups with short chains: the kernel whose chain is a quarter as long.  It takes 6.6 us + 0.92 per trip (of 128
  // queries) while its workgroups have a CU each, the usual one 5.3 + 1.25 per trip (of 64): B2 H9/3 S256 20.3 -> 12.1, B2 H32
  // S256 (256 workgroups) 10.4 -> 8.6, B8 H9/3 S512 (12 trips) 22.1 -> 18.3.  With longer chains the usual kernel's pieces win
  // (B3 H9/3 S777, 21 trips: 25.2, here 26.4), with more workgroups its two per CU (B4 H32 S256 10.7, here 14.0).
  if constexpr (D == 64) {
    using F = KvCfg<64, 4>;
    if (heads * tiles_before(a.kv, a.Sk, F::BN) <= 256 && dkdv_trips(a, 0, F::BN, F::BM) <= 14) {
      plan.few = true;
      return plan;
    }
  }
  plan.pair = a.causal && n_ktiles >= 2 && heads * ((n_ktiles + 1) / 2) >= (D == 64 ? 384 : 256);
  TripCost cost = {1.1, 1.0, 1.0, C::kPerCu, 0.0};
  if (D == 128) cost = {1.65, 2.05, 1.0, C::kPerCu, 0.0};
  cost.piece_bytes = 4.0 * C::kKeyWaves * dkdv_piece_floats(D);
  auto trips_of = [&](int i) { return dkdv_trips(a, i, C::BN, C::BM); };
  plan.len = choose_pieces(heads, n_ktiles, cost, plan.pair, trips_of);
  // Key tiles of 256 (attn_bwd_roles.hip) where the estimate says so, by a sixth: the line lies under the first launch that loses.  Of 115 launches whose estimate
  // is under the others' (113 of them drawn), the 72 below the line take 0.69 to 0.993 of the time of the others, 0.86 in the mean.  The first above it is at
  // 0.844 and loses (B8 H6/2 S2057 without a mask 263 -> 269 us; B4 H16 S1100 causal, at 0.844 too, would gain, 63 -> 58), and from there to 1 so do 16 of 43, up to
  // 1.06 (0.96 in the mean: masked and unmasked trips have one price here, and an estimate that tells them apart could take more).  Few workgroups lose, and are cut: B1
  // H32 S1024 28.6 us, 46.4 so; B1 H32 S2048 causal, one round of unequal lengths, 71.8 and 92.9.  A trip (64 queries) takes 2.6 us with half of the GPU idle and 3.15 with
  // all of it busy.
  if constexpr (D == 128) {
    using R = RoleTiles;
    auto role_trips = [&](int i) { return dkdv_trips(a, i, R::BN, R::BM); };
    const double us = launch_us(heads, n_ktiles, cost, plan.len, plan.len == 0 && plan.pair, trips_of);
    const double roles_us = launch_us(heads, tiles_before(a.kv, a.Sk, R::BN), {2.6, 3.15, 1.0, R::kPerCu, 0.0}, 0, false, role_trips);
    if (roles_us < 0.84 * us) {
      plan = DkdvPlan();
      plan.roles = true;
      return plan;
    }
  }
  if (plan.len > 0) plan.ws_bytes = static_cast<int64_t>(heads * count_pieces(n_ktiles, plan.len, trips_of) * cost.piece_bytes);
  return plan;
}
template <int D>
const DkdvPlan& plan_dkdv(const AttnParams& a) {
  static thread_local PlanTable<DkdvPlan> table;
  return table.get(a, D, [&] { return make_dkdv_plan<D>(a); });
}

template <int D, bool kCut>
int launch_dkdv_impl(const BwdParams& p, int grid_y, hipStream_t s) {
  using C = KvCfg<D, kUsualSplit<D>>;
  static LdsOnce lds_reserved;
  if (!reserve_lds_once(lds_reserved, reinterpret_cast<const void*>(KvKernel<D, kCut>::fn), C::kLdsBytes))
    return fail(PICO_ERR_LAUNCH, "pico_attn_bwd(dk/dv): cannot reserve %zu bytes of LDS", C::kLdsBytes);
  hipLaunchKernelGGL((KvKernel<D, kCut>::fn), dim3(p.a.Hkv * p.a.B, grid_y), dim3(C::kThreads), C::kLdsBytes, s, p);
  return PICO_OK;
}
template <int D>
int launch_dkdv(const BwdParams& p, float* ws, int64_t ws_bytes, hipStream_t s) {
  using C = KvCfg<D, kUsualSplit<D>>;
  const DkdvPlan& plan = plan_dkdv<D>(p.a);
  if constexpr (D == 64) {
    if (plan.few) {
      using F = KvCfg<64, 4>;
      static LdsOnce reserved;
      if (!reserve_lds_once(reserved, reinterpret_cast<const void*>(&attn_bwd_dkdv_few_kernel), F::kLdsBytes))
        return fail(PICO_ERR_LAUNCH, "pico_attn_bwd(dk/dv): cannot reserve %zu bytes of LDS", F::kLdsBytes);
      BwdParams q = p;
      q.pair_ktiles = 0;
      hipLaunchKernelGGL(attn_bwd_dkdv_few_kernel, dim3(p.a.Hkv * p.a.B, tiles_before(p.a.kv, p.a.Sk, F::BN)), dim3(F::kThreads), F::kLdsBytes, s, q);
      return PICO_OK;
    }
  }
  if constexpr (D == 128) {
    if (plan.roles) return launch_dkdv_roles(p, s);
  }
  const int n_ktiles = tiles_before(p.a.kv, p.a.Sk, C::BN);
  BwdParams q = p;
  if (plan.len == 0 || !ws || ws_bytes < plan.ws_bytes) {
    q.pair_ktiles = plan.pair ? n_ktiles : 0;
    return launch_dkdv_impl<D, false>(q, plan.pair ? (n_ktiles + 1) / 2 : n_ktiles, s);
  }
  q.a.pieces = Pieces{plan.len, ws};
  const int n = count_pieces(n_ktiles, plan.len, [&](int i) { return dkdv_trips(p.a, i, C::BN, C::BM); });
  if (int rc = launch_dkdv_impl<D, true>(q, n, s)) return rc;
  hipLaunchKernelGGL(attn_bwd_dkdv_join_kernel<D>, dim3(p.a.Hkv * p.a.B, n_ktiles, 2), dim3(256), 0, s, q, n);
  return PICO_OK;
}

template <int D, int NW, int KT, bool kDelta, int KS, bool kCut>
int launch_dq_impl(const BwdParams& p, hipStream_t s) {
  using C = DqCfg<D, NW, KT, KS>;
  static LdsOnce lds_reserved;
  if (!reserve_lds_once(lds_reserved, reinterpret_cast<const void*>(&attn_bwd_dq_kernel<D, NW, KT, kDelta, KS, kCut>), C::kLdsBytes))
    return fail(PICO_ERR_LAUNCH, "pico_attn_bwd(dq): cannot reserve %zu bytes of LDS", C::kLdsBytes);
  const int heads = p.a.Hq * p.a.B, n_qtiles = (p.a.Sq + C::BM - 1) / C::BM, len = p.a.pieces.len;
  const int n = count_pieces(n_qtiles, len, [&](int i) { return query_tile_trips(p.a, n_qtiles - 1 - i, C::BM, KT); });
  hipLaunchKernelGGL((attn_bwd_dq_kernel<D, NW, KT, kDelta, KS, kCut>), dim3(heads, n), dim3(C::kThreads), C::kLdsBytes, s, p);
  if (kCut && len > 0)
    hipLaunchKernelGGL((attn_bwd_dq_join_kernel<D, C::kQWaves, KT, C::kSmall>), dim3(heads, n_qtiles), dim3(64 * C::kQWaves), 0, s, p, n);
  return PICO_OK;
}

template <int D, int NW, int KT, int KS = 1>
int launch_dq(const BwdParams& p, hipStream_t s) {
  const bool cut = p.a.pieces.len > 0 || ends_inside_tile(p.a.kv, KT);
  if (p.out) return cut ? launch_dq_impl<D, NW, KT, true, KS, true>(p, s) : launch_dq_impl<D, NW, KT, true, KS, false>(p, s);
  return cut ? launch_dq_impl<D, NW, KT, false, KS, true>(p, s) : launch_dq_impl<D, NW, KT, false, KS, false>(p, s);
}

// How the dQ launch is run: which kernel, and whether its query tiles are cut into pieces.
struct DqPlan {
  enum { kWaves4, kWaves8, kSplit4, kSplit8 } kernel;
  int len = 0;
  int64_t ws_bytes = 0;
};
DqPlan make_dq_plan(const AttnParams& a, int D) {
  DqPlan plan;
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
  if (D == 64) {
    const int64_t visible_keys = a.causal ? std::min<int64_t>(a.Sk, static_cast<int64_t>(a.q_offset) + a.Sq) : a.Sk;
    // the forward's rules: eight waves per workgroup also for rectangular launches (every query sees at least as many
    // keys as there are queries) with fewer workgroups than the square ones need
    const bool rectangular = !a.causal || a.q_offset >= a.Sq;
    // several generations of workgroups over short key ranges (a few trips each): two four-wave workgroups per CU hide
    // each other's prologues and epilogues, which one eight-wave workgroup per CU cannot (B8 S768 51.3 -> 44.3 us,
    // B16 S512 54.4 -> 48.1, B8 S1024 78.5 -> 72.9, B8 S1536 147.8 -> 144.3; from S2048 on, and with 512 workgroups,
    // the eight-wave kernel is level or ahead)
    if (groups(256) >= 768 && visible_keys <= 1536) plan.kernel = DqPlan::kWaves4;
    else if (groups(256) >= 512) plan.kernel = DqPlan::kWaves8;
    else if (groups(128) >= 512) plan.kernel = rectangular && groups(256) >= 256 ? DqPlan::kWaves8 : DqPlan::kWaves4;
    // few waves in all: two waves per 32 queries, 64 keys of every 128 each (rank 3 of 4 of B4 H32 S1024 with eight waves
    // per workgroup: 18.8 -> 17.9 us)
    else plan.kernel = groups(128) >= 256 && rectangular && visible_keys >= 512 ? DqPlan::kSplit8 : DqPlan::kSplit4;
    switch (plan.kernel) {
      case DqPlan::kWaves8: use(DqCfg<64, 8, 64>(), 1.7, 1.5, 1.0); break;
      case DqPlan::kWaves4: use(DqCfg<64, 4, 64>(), 0.89, 0.44, 1.18); break;
      case DqPlan::kSplit8: use(DqCfg<64, 8, 128, 2>(), 1.6, 1.5, 1.0); break;
      case DqPlan::kSplit4: use(DqCfg<64, 4, 128, 2>(), 1.25, 0.8, 1.0); break;
    }
  } else {
    // The forward's rule (see there), with other lines.  Four waves and eight, us: up to 384 workgroups of eight waves B8 H8 S769 27, 32, B1 H32 S1918
    // 55, 65, B8 H8 S1418 without a mask 96, 114, B4 H8 S3063 109, 111.5; then eight (432: 97, 96; 448: 145, 135); just over two rounds B8 H12 S1403
    // 78, 87, B4 H8 S4386 205, 214; beyond them by a few percent one way or the other (B8 H32 S5246 2918, 2610).  One workgroup to a head either way:
    // B64 H32 S128 70, 103; B128 H32/8 S64 67, 122; B48 H32/8 128 x 4096 518, 930.  The line at 8192 keys is the forward's and costs less on either
    // side (288 workgroups of 8192 x 10240 498, 521, x 16384 767, 825, shifted 612, 587, x 32768 1560, 1549), and so does its absence under one
    // round of workgroups of eight (12 heads of 4096 x 16384 484, 443; 9 of 4096 x 8192 172, 171; whole sequences of 14 heads 99, 112).
    const bool rectangular = !a.causal || a.q_offset >= a.Sq;
    const int64_t wide = groups(256), narrow = groups(128);
    const bool idle = wide <= 384 && !(rectangular && wide == 256), third = wide > 512 && wide <= 640, padded = narrow <= 1024 && 10 * narrow <= 18 * wide;
    plan.kernel = wide < 256 || narrow == wide || (a.Sk <= 8192 && (idle || third || padded)) ? DqPlan::kWaves4 : DqPlan::kWaves8;
    if (plan.kernel == DqPlan::kWaves8) use(DqCfg<128, 8, 64>(), 1.15, 2.81, 1.01);
    else {
      // The estimates put short walks in pieces 2 to 7 us too high (what the second kernel adds up is still in L2), so half of the time of a launch
      // is asked for.  That cuts 27 of 589 drawn launches more, walks of 11 to 22 key tiles, to 0.76 to 0.98 of their time (one 1.024): B2 H4 S1168
      // 25.2 us whole, 19.0 cut; B4 H2 S480 x 960 20.9, 16.9; B1 H4 S877 20.2, 17.0.  (2.0 would cut heads in eights of 14 tiles as well, whose sums
      // stay on their XCD, B1 H8 S859 20.1, 16.8, but also B1 H9/3 S890 19.7, 21.2.)
      use(DqCfg<128, 4, 64>(), 1.4, 0.9, 1.15);
      cost.launch_us = 2.5;
    }
  }
  const int n_qtiles = (a.Sq + bm - 1) / bm;
  cost.piece_bytes = 4.0 * (bm / 32) * dq_piece_floats(D);
  auto trips_of = [&](int i) { return query_tile_trips(a, n_qtiles - 1 - i, bm, kt); };
  plan.len = choose_pieces(heads, n_qtiles, cost, false, trips_of);
  if (plan.len > 0) plan.ws_bytes = static_cast<int64_t>(heads * count_pieces(n_qtiles, plan.len, trips_of) * cost.piece_bytes);
  return plan;
}
const DqPlan& plan_dq(const AttnParams& a, int D) {
  static thread_local PlanTable<DqPlan> table;
  return table.get(a, D, [&] { return make_dq_plan(a, D); });
}

}  // namespace
}  // namespace pico

using namespace pico;

extern "C" int pico_attn_bwd_preprocess(const pico_attn_desc* desc, const void* dout, const void* out, int out_dtype,
                                        float* delta, float* dq_acc, void* stream) {
  if (int rc = check_attn_desc("pico_attn_bwd_preprocess", desc)) return rc;
  if (out_dtype != PICO_BF16 && out_dtype != PICO_F32)
    return fail(PICO_ERR_DTYPE, "pico_attn_bwd_preprocess: out dtype code %d not supported", out_dtype);
  if (desc->B == 0 || desc->Sq == 0) return PICO_OK;
  if (!dout || !out || !delta) return fail(PICO_ERR_NULL, "pico_attn_bwd_preprocess: dout, out and delta are required");
  if (!aligned16(dout) || !aligned16(out) || !aligned16(dq_acc))
    return fail(PICO_ERR_ALIGN, "pico_attn_bwd_preprocess: dout, out and dq_acc must be 16-byte aligned");
  const int64_t rows = static_cast<int64_t>(desc->B) * desc->Hq * desc->Sq;
  const int64_t total = rows * (desc->D / 8);
  const unsigned grid = static_cast<unsigned>((total + 255) / 256);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int64_t* os = desc->o_stride;
#define PICO_PRE(DD, TO)                                                                                   \
  hipLaunchKernelGGL((attn_bwd_preprocess_kernel<DD, TO>), dim3(grid), dim3(256), 0, s,                    \
                     static_cast<const __bf16*>(dout), static_cast<const TO*>(out), delta, dq_acc, desc->B, \
                     desc->Hq, desc->Sq, os[0], os[1], os[2])
  if (desc->D == 64) { if (out_dtype == PICO_BF16) PICO_PRE(64, __bf16); else PICO_PRE(64, float); }
  else               { if (out_dtype == PICO_BF16) PICO_PRE(128, __bf16); else PICO_PRE(128, float); }
#undef PICO_PRE
  return check_launch("pico_attn_bwd_preprocess");
}

namespace {

// Shared body of the backward entry points.  With `out` (bf16 forward output) the dQ kernel computes delta itself,
// writes it to `delta_w`, and runs BEFORE the dK/dV kernel, which reads it from there.
int run_bwd(const char* fn, const pico_attn_desc* desc, const void* q, const pico_kv_chunks* kv, const void* dout,
            const float* lse, const float* delta, const void* out, float* delta_w, void* dq, const int64_t* dq_stride,
            int dq_dtype, int dq_accumulate, const int64_t* dkv_stride, int dkv_dtype, void* stream,
            const RopeArgs* rope = nullptr, float* ws = nullptr, int64_t ws_bytes = 0) {
  if ((dkv_dtype != PICO_BF16 && dkv_dtype != PICO_F32) || (dq_dtype != PICO_BF16 && dq_dtype != PICO_F32))
    return fail(PICO_ERR_DTYPE, "%s: gradient dtype codes %d / %d not supported", fn, dq_dtype, dkv_dtype);
  if (dq_accumulate && dq_dtype != PICO_F32) return fail(PICO_ERR_DTYPE, "%s: accumulate needs fp32 gradients", fn);
  BwdParams p;
  p.a = make_params(desc, q, nullptr, nullptr);
  if (int rc = set_chunks(fn, desc, kv, p.a, false)) return rc;
  if (desc->B == 0) return PICO_OK;
  // a gradient that is not wanted is passed as NULL and its kernel (or its chunk's workgroups) is skipped
  bool want_dkv = false;
  p.dkv_accumulate = 0;
  for (int c = 0; c < kMaxChunks; ++c) {
    p.dk[c] = p.dv[c] = nullptr;
    p.dk_final[c] = p.dv_final[c] = nullptr;
  }
  bool any_final = false;
  for (int c = 0; c < kv->count; ++c) {
    if ((kv->dk[c] == nullptr) != (kv->dv[c] == nullptr) || (kv->dk_final[c] == nullptr) != (kv->dv_final[c] == nullptr))
      return fail(PICO_ERR_NULL, "%s: dk and dv (and dk_final and dv_final) must be given together (chunk %d)", fn, c);
    if (!aligned16(kv->dk_final[c]) || !aligned16(kv->dv_final[c]))
      return fail(PICO_ERR_ALIGN, "%s: chunk %d: dk_final and dv_final must be 16-byte aligned", fn, c);
    p.dk[c] = kv->dk[c];
    p.dv[c] = kv->dv[c];
    p.dk_final[c] = static_cast<__bf16*>(kv->dk_final[c]);
    p.dv_final[c] = static_cast<__bf16*>(kv->dv_final[c]);
    const bool acc = kv->dk[c] && ((kv->accumulate_mask >> c) & 1u);
    if (kv->dk[c] || kv->dk_final[c]) want_dkv = true;
    if (acc) p.dkv_accumulate |= 1u << c;
    if (kv->dk_final[c]) {
      any_final = true;
      if (acc && dkv_dtype != PICO_F32)
        return fail(PICO_ERR_DTYPE, "%s: chunk %d: the sums that dk_final completes must be fp32", fn, c);
    }
  }
  for (int i = 0; i < 3; ++i) {
    p.dkfs[i] = any_final ? kv->final_stride[i] : 0;
    if (any_final && (p.dkfs[i] < 0 || p.dkfs[i] % 4 != 0))
      return fail(PICO_ERR_STRIDE, "%s: final_stride must hold non-negative multiples of 4 elements", fn);
  }
  if (p.dkv_accumulate && dkv_dtype != PICO_F32) return fail(PICO_ERR_DTYPE, "%s: accumulate needs fp32 gradients", fn);
  const bool want_dq = dq != nullptr;
  const bool have_q = desc->Sq > 0 && want_dq, have_k = desc->Sk > 0 && want_dkv;
  if ((have_q || have_k) && desc->Sq > 0 && (!q || !dout || !lse || !delta))
    return fail(PICO_ERR_NULL, "%s: q, dout, lse and delta are required", fn);
  if ((have_q || have_k) && desc->Sk > 0)
    for (int c = 0; c < kv->count; ++c)
      if (!kv->k[c] || !kv->v[c]) return fail(PICO_ERR_NULL, "%s: k / v of chunk %d are NULL", fn, c);
  if (!aligned16(q) || !aligned16(dout) || !aligned16(dq) || !aligned16(out))
    return fail(PICO_ERR_ALIGN, "%s: q, dout, out and dq must be 16-byte aligned", fn);
  p.dout = static_cast<const __bf16*>(dout);
  p.lse = lse; p.delta = delta; p.dq = dq;
  p.out = static_cast<const __bf16*>(out);
  p.delta_w = delta_w;
  p.dq_f32 = dq_dtype == PICO_F32;
  p.dq_accumulate = dq_accumulate != 0;
  p.dkv_f32 = dkv_dtype == PICO_F32;
  p.pair_ktiles = 0;
  p.rope = rope ? *rope : RopeArgs{nullptr, nullptr, 0, 0, 0, 0};
  auto strides = [&](const int64_t* given, int heads, int seq, int64_t (&st)[3], int align) -> bool {
    if (given) {
      for (int i = 0; i < 3; ++i) {
        if (given[i] < 0 || given[i] % align != 0) return false;
        st[i] = given[i];
      }
    } else {
      st[2] = desc->D;
      st[1] = static_cast<int64_t>(seq) * desc->D;
      st[0] = st[1] * heads;
    }
    return true;
  };
  if (!strides(dq_stride, desc->Hq, desc->Sq, p.dqs, p.dq_f32 ? 4 : 8) || !strides(dkv_stride, desc->Hkv, kv->chunk_len, p.dks, 8))
    return fail(PICO_ERR_STRIDE, "%s: dq strides must be non-negative multiples of 4 (fp32) or 8 (bf16), dk/dv strides of 8", fn);
  hipStream_t s = static_cast<hipStream_t>(stream);
  auto run_dkdv = [&]() -> int {
    if (!have_k) return PICO_OK;
    // without queries the dK/dV kernel still runs: it writes (or adds) zeros
    if (int rc = desc->D == 64 ? launch_dkdv<64>(p, ws, ws_bytes, s) : launch_dkdv<128>(p, ws, ws_bytes, s)) return rc;
    return check_launch("pico_attn_bwd(dk/dv)");
  };
  auto run_dq = [&]() -> int {
    if (!have_q) return PICO_OK;
    // without keys the dQ kernel still runs: it writes (or adds) zeros
    const DqPlan& plan = plan_dq(p.a, desc->D);
    BwdParams p_dq = p;
    p_dq.a.pieces = Pieces{ws && ws_bytes >= plan.ws_bytes ? plan.len : 0, ws};
    int rc;
    if (desc->D == 64) {
      if (plan.kernel == DqPlan::kWaves8) rc = launch_dq<64, 8, 64>(p_dq, s);
      else if (plan.kernel == DqPlan::kWaves4) rc = launch_dq<64, 4, 64>(p_dq, s);
      else if (plan.kernel == DqPlan::kSplit8) rc = launch_dq<64, 8, 128, 2>(p_dq, s);
      else rc = launch_dq<64, 4, 128, 2>(p_dq, s);
    } else {
      rc = plan.kernel == DqPlan::kWaves8 ? launch_dq<128, 8, 64>(p_dq, s) : launch_dq<128, 4, 64>(p_dq, s);
    }
    if (rc) return rc;
    return check_launch("pico_attn_bwd(dq)");
  };
  if (p.out) {  // the dQ kernel produces delta for the dK/dV kernel
    if (int rc = run_dq()) return rc;
    return run_dkdv();
  }
  if (int rc = run_dkdv()) return rc;
  return run_dq();
}

pico_kv_chunks one_chunk(const pico_attn_desc* desc, const void* k, const void* v, void* dk, void* dv, int accumulate) {
  pico_kv_chunks kv = {};
  kv.count = 1;
  kv.chunk_len = desc->Sk;
  kv.k[0] = k;
  kv.v[0] = v;
  kv.dk[0] = dk;
  kv.dv[0] = dv;
  kv.accumulate_mask = accumulate ? 1u : 0u;
  return kv;
}

// delta inside the dQ kernel needs that kernel to run and a bf16 out; otherwise the pre-pass computes it
int run_bwd_with_out(const char* fn, const pico_attn_desc* desc, const void* q, const pico_kv_chunks* kv, const void* dout,
                     const void* out, int out_dtype, const float* lse, float* delta, void* dq, const int64_t* dq_stride,
                     int dq_dtype, int dq_accumulate, const int64_t* dkv_stride, int dkv_dtype, void* stream,
                     const RopeArgs* rope, float* ws = nullptr, int64_t ws_bytes = 0) {
  if (out_dtype != PICO_BF16 && out_dtype != PICO_F32)
    return fail(PICO_ERR_DTYPE, "%s: out dtype code %d not supported", fn, out_dtype);
  if (desc->B == 0) return PICO_OK;
  if (desc->Sq > 0 && (!out || !delta)) return fail(PICO_ERR_NULL, "%s: out and delta are required", fn);
  const bool in_kernel = out_dtype == PICO_BF16 && dq != nullptr && desc->Sq > 0;
  if (!in_kernel) {
    if (int rc = pico_attn_bwd_preprocess(desc, dout, out, out_dtype, delta, nullptr, stream)) return rc;
    return run_bwd(fn, desc, q, kv, dout, lse, delta, nullptr, nullptr, dq, dq_stride, dq_dtype, dq_accumulate, dkv_stride,
                   dkv_dtype, stream, rope, ws, ws_bytes);
  }
  return run_bwd(fn, desc, q, kv, dout, lse, delta, out, delta, dq, dq_stride, dq_dtype, dq_accumulate, dkv_stride, dkv_dtype,
                 stream, rope, ws, ws_bytes);
}

int rope_args(const char* fn, const pico_attn_desc* desc, const pico_rope_tables* rope, int q_pos_offset, int k_pos_offset,
              RopeArgs& r) {
  if (q_pos_offset < 0 || k_pos_offset < 0) return fail(PICO_ERR_SHAPE, "%s: position offsets must be >= 0", fn);
  const int64_t last = std::max(static_cast<int64_t>(q_pos_offset) + desc->Sq, static_cast<int64_t>(k_pos_offset) + desc->Sk) - 1;
  if (int rc = check_rope_tables(fn, rope, desc->D, last)) return rc;
  r = RopeArgs{rope->cos, rope->sin, rope->pitch, rope->dtype == PICO_F32, q_pos_offset, k_pos_offset};
  return PICO_OK;
}

}  // namespace

extern "C" int pico_attn_bwd(const pico_attn_desc* desc, const void* q, const void* k, const void* v, const void* dout,
                             const float* lse, const float* delta, void* dq, const int64_t* dq_stride, int dq_dtype,
                             int dq_accumulate, void* dk, void* dv, const int64_t* dkv_stride, int dkv_dtype,
                             int dkv_accumulate, void* stream) {
  if (int rc = check_attn_desc("pico_attn_bwd", desc)) return rc;
  if (dkv_accumulate && dkv_dtype != PICO_F32) return fail(PICO_ERR_DTYPE, "pico_attn_bwd: accumulate needs fp32 gradients");
  const pico_kv_chunks kv = one_chunk(desc, k, v, dk, dv, dkv_accumulate);
  return run_bwd("pico_attn_bwd", desc, q, &kv, dout, lse, delta, nullptr, nullptr, dq, dq_stride, dq_dtype, dq_accumulate,
                 dkv_stride, dkv_dtype, stream);
}

extern "C" int pico_attn_bwd_fused(const pico_attn_desc* desc, const void* q, const void* k, const void* v,
                                   const void* dout, const void* out, int out_dtype, const float* lse, float* delta,
                                   void* dq, const int64_t* dq_stride, int dq_dtype, int dq_accumulate, void* dk, void* dv,
                                   const int64_t* dkv_stride, int dkv_dtype, int dkv_accumulate, void* stream) {
  const char* fn = "pico_attn_bwd_fused";
  if (int rc = check_attn_desc(fn, desc)) return rc;
  if (dkv_accumulate && dkv_dtype != PICO_F32) return fail(PICO_ERR_DTYPE, "%s: accumulate needs fp32 gradients", fn);
  const pico_kv_chunks kv = one_chunk(desc, k, v, dk, dv, dkv_accumulate);
  return run_bwd_with_out(fn, desc, q, &kv, dout, out, out_dtype, lse, delta, dq, dq_stride, dq_dtype, dq_accumulate,
                          dkv_stride, dkv_dtype, stream, nullptr);
}

extern "C" int pico_attn_bwd_rope(const pico_attn_desc* desc, const void* q_rot, const void* k_rot, const void* v,
                                  const void* dout, const void* out, const float* lse, float* delta, void* dq,
                                  const int64_t* dq_stride, int dq_dtype, int dq_accumulate, void* dk, void* dv,
                                  const int64_t* dkv_stride, int dkv_dtype, int dkv_accumulate,
                                  const pico_rope_tables* rope, int q_pos_offset, int k_pos_offset, void* stream) {
  const char* fn = "pico_attn_bwd_rope";
  if (int rc = check_attn_desc(fn, desc)) return rc;
  if (desc->B == 0) return PICO_OK;
  RopeArgs r;
  if (int rc = rope_args(fn, desc, rope, q_pos_offset, k_pos_offset, r)) return rc;
  if (!dq || !dk || !dv) return fail(PICO_ERR_NULL, "%s: dq, dk and dv are required", fn);
  if (dkv_accumulate && dkv_dtype != PICO_F32) return fail(PICO_ERR_DTYPE, "%s: accumulate needs fp32 gradients", fn);
  const pico_kv_chunks kv = one_chunk(desc, k_rot, v, dk, dv, dkv_accumulate);
  return run_bwd_with_out(fn, desc, q_rot, &kv, dout, out, PICO_BF16, lse, delta, dq, dq_stride, dq_dtype, dq_accumulate,
                          dkv_stride, dkv_dtype, stream, &r);
}

namespace {

// what a plan is made from, without operands; false: there is nothing to launch
bool plan_params(const pico_attn_desc* desc, int chunk_count, AttnParams& a) {
  if (!desc || chunk_count < 1 || (desc->D != 64 && desc->D != 128) || desc->B <= 0 || desc->Hkv <= 0 || desc->Hq % desc->Hkv != 0 ||
      desc->Hq <= 0 || desc->Sq <= 0 || desc->Sk <= 0)
    return false;
  a = make_params(desc, nullptr, nullptr, nullptr);
  a.kv.count = chunk_count;
  a.kv.len = desc->Sk / chunk_count;
  return true;
}

}  // namespace

extern "C" int64_t pico_attn_bwd_workspace_bytes(const pico_attn_desc* desc, int chunk_count) {
  AttnParams a;
  if (!plan_params(desc, chunk_count, a)) return 0;
  const int64_t dkdv = desc->D == 64 ? plan_dkdv<64>(a).ws_bytes : plan_dkdv<128>(a).ws_bytes;
  return std::max(dkdv, plan_dq(a, desc->D).ws_bytes);   // (the two kernels run one after the other)
}

extern "C" int pico_attn_dkdv_plan(const pico_attn_desc* desc, int chunk_count, int32_t* out) {
  if (!out) return fail(PICO_ERR_NULL, "pico_attn_dkdv_plan: the plan is NULL");
  AttnParams a;
  if (!plan_params(desc, chunk_count, a)) return fail(PICO_ERR_SHAPE, "pico_attn_dkdv_plan: no launch for this descriptor");
  const DkdvPlan& plan = desc->D == 64 ? plan_dkdv<64>(a) : plan_dkdv<128>(a);
  out[0] = plan.roles ? RoleTiles::BN : plan.few ? KvCfg<64, 4>::BN : 128;
  out[1] = plan.pair && plan.len == 0 ? 2 : 1;
  out[2] = plan.len;
  return PICO_OK;
}

extern "C" int pico_attn_dq_plan(const pico_attn_desc* desc, int chunk_count, int32_t* out) {
  if (!out) return fail(PICO_ERR_NULL, "pico_attn_dq_plan: the plan is NULL");
  AttnParams a;
  if (!plan_params(desc, chunk_count, a)) return fail(PICO_ERR_SHAPE, "pico_attn_dq_plan: no launch for this descriptor");
  const DqPlan& plan = plan_dq(a, desc->D);
  out[0] = plan.kernel == DqPlan::kWaves8 || plan.kernel == DqPlan::kSplit8 ? 8 : 4;
  out[1] = plan.kernel == DqPlan::kSplit4 || plan.kernel == DqPlan::kSplit8 ? 2 : 1;
  out[2] = plan.len;
  return PICO_OK;
}

extern "C" int pico_attn_bwd_chunks_ws(const pico_attn_desc* desc, const void* q, const pico_kv_chunks* kv, const void* dout,
                                       const void* out, int out_dtype, const float* lse, float* delta, void* dq,
                                       const int64_t* dq_stride, int dq_dtype, int dq_accumulate, const int64_t* dkv_stride,
                                       int dkv_dtype, const pico_rope_tables* rope, int q_pos_offset, int k_pos_offset,
                                       void* workspace, int64_t workspace_bytes, void* stream) {
  const char* fn = "pico_attn_bwd_chunks";
  if (int rc = check_attn_desc(fn, desc)) return rc;
  if (!kv) return fail(PICO_ERR_NULL, "%s: the chunk list is NULL", fn);
  if (!aligned16(workspace)) return fail(PICO_ERR_ALIGN, "%s: the workspace must be 16-byte aligned", fn);
  if (desc->B == 0) return PICO_OK;
  RopeArgs r;
  if (rope) {
    if (int rc = rope_args(fn, desc, rope, q_pos_offset, k_pos_offset, r)) return rc;
  }
  float* ws = static_cast<float*>(workspace);
  if (out)
    return run_bwd_with_out(fn, desc, q, kv, dout, out, out_dtype, lse, delta, dq, dq_stride, dq_dtype, dq_accumulate, dkv_stride,
                            dkv_dtype, stream, rope ? &r : nullptr, ws, workspace_bytes);
  return run_bwd(fn, desc, q, kv, dout, lse, delta, nullptr, nullptr, dq, dq_stride, dq_dtype, dq_accumulate, dkv_stride, dkv_dtype,
                 stream, rope ? &r : nullptr, ws, workspace_bytes);
}

extern "C" int pico_attn_bwd_chunks(const pico_attn_desc* desc, const void* q, const pico_kv_chunks* kv, const void* dout,
                                    const void* out, int out_dtype, const float* lse, float* delta, void* dq,
                                    const int64_t* dq_stride, int dq_dtype, int dq_accumulate, const int64_t* dkv_stride,
                                    int dkv_dtype, const pico_rope_tables* rope, int q_pos_offset, int k_pos_offset,
                                    void* stream) {
  return pico_attn_bwd_chunks_ws(desc, q, kv, dout, out, out_dtype, lse, delta, dq, dq_stride, dq_dtype, dq_accumulate, dkv_stride,
                                 dkv_dtype, rope, q_pos_offset, k_pos_offset, nullptr, 0, stream);
}
