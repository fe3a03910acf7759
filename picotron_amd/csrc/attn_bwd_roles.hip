// dK / dV at head_dim 128: one workgroup owns 256 keys of one kv head and walks the queries that see them, 32 at a time.
// Its eight waves work in pairs (waves w and w + 4, which share a SIMD) on 64 keys; each wave of a pair has two of the four products:
//   S wave:   S = Q K^T, P = exp2(S c - lse log2e), dV^T += dO^T P
//   dP wave:  dP = dO V^T - delta, dS = P (dP - delta), dK^T += Q^T dS
// so a wave holds the fragments of one operand (K or V) and one set of accumulators (dV or dK) for 64 keys in 256 registers, and every fragment of Q
// and dO that it reads from LDS has four MFMAs.  P goes from the one to the other through LDS, in fp32 and in the order of their registers; the dP wave is
// a step behind the S wave, so one barrier per step is enough.
//
// What this split gives over waves that have all four products of 32 keys (attn_bwd_dkdv_kernel_d128), us: B1 H32 S4096 causal 239 -> 216, 4096 queries and
// 32768 keys with 32 / 8 heads 3470 -> 3010, B8 H32 S1024 without a mask 279 -> 240, B3 H32 S777 64 -> 44; 70 drawn launches 0.874 of the time.
// LDS: 22 reads and 4 writes of 16 bytes (a transposing pair is one) for 64 MFMAs of 16 x 16 x 32, 34 instructions, where there were 49 reads, 65 instructions,
// for 32 of twice the work each; products of 16 x 16 x 32 take a seventh less power (see DqWave).  For 4096 queries and 32768 keys the clock rose from 1.77 to 2.16 GHz
// by it (dQ, whose matrix pipe is fuller, 1.88), with the matrix pipe busy for 0.61 of the cycles instead of 0.65: what is left is the length of the two waves' own
// chains, 2700 and 2400 of a step's 3400 cycles when the other wave does
// nothing (LDS latency behind the barrier 100 to 180, exp2 and what waits for P 1000 to 1300, dV or dK 600, the step's scalar work 160).
// Taken out one at a time from B8 H32 S1024, us: P's way through LDS 250 -> 231, exp2 243, requests 216, most of dV and dK 194.
// Two bodies in turn for the halves of a tile, or a branch between them, spill: the walk has 256 registers and needs 250 to 256 in every form.
#include "attn_bwd.h"

namespace pico {
namespace {

struct RoleCfg : RoleTiles {
  static constexpr int D = 128, NW = 8, kThreads = 64 * NW, kPairs = 4;
  // of a tile's keys pair w has 64 kb + 16 w .. + 15 for kb < 4, so that all pairs see as much of a diagonal; a trip's queries are a tile of LDS, two steps
  using L = TileLayout<D>;
  static constexpr int kSide = L::bytes(BM), kLoads = BM * (D / 8) / kThreads;
  static constexpr int kRowsAt = 2 * kSide;                      // lse (in log2) and -delta of a tile's rows, behind Q and dO
  static constexpr int kBufBytes = 2 * kSide + 2 * BM * 4;
  static constexpr int kTileBytes = 2 * kBufBytes;
  static constexpr int kPairBytes = 32 * 64 * 4, kPBytes = kPairs * kPairBytes;   // P of a step
  static constexpr int kFragmentBytes = NW * WaveTile<D>::kRegionBytes;          // K and V pass through the place of P, 32 rows at a time
  static constexpr size_t kLdsBytes = kTileBytes + (2 * kPBytes > kFragmentBytes ? 2 * kPBytes : kFragmentBytes);
  static_assert(kLdsBytes <= 160 * 1024);
  static_assert(NW * kRowRegionBytes <= kTileBytes, "the epilogue reuses the tile buffers");
};
// dK (kDk) or dV of a wave's 64 keys, from row `row0` of their chunk and position `key0` on 16 of every 64
template <bool kDk>
__device__ __forceinline__ void role_store(const BwdParams& p, unsigned char* region, f32x4 (&acc)[8][4], int chunk, int b, int hkv, int row0, int key0, int lane) {
  constexpr int D = RoleCfg::D;
  const AttnParams& a = p.a;
  const float scale = kDk ? a.sm_scale : 1.f;
  const bool accumulate = (p.dkv_accumulate >> chunk) & 1u;
  each_load<2>([&](auto half) __attribute__((always_inline)) {
    constexpr int kb = 2 * decltype(half)::value;
    const RowPair<kb, 8, 4> part = {acc};
    const int row = row0 + 64 * kb, rows_live = a.kv.len - row;
    if (rows_live <= 0) return;
    if (kDk && p.rope.cos != nullptr) {
      const int n = lane % 16;
      const int pos[2] = {n < rows_live ? p.rope.k_pos0 + key0 + 64 * kb + n : 0, n + 64 < rows_live ? p.rope.k_pos0 + key0 + 64 * (kb + 1) + n : 0};
      rope_unrotate_acc<D>(part, p.rope, pos, lane);
    }
    const int64_t off = b * p.dks[0] + hkv * p.dks[1] + static_cast<int64_t>(row) * p.dks[2];
    void* const dst = kDk ? p.dk[chunk] : p.dv[chunk];
    __bf16* const total = kDk ? p.dk_final[chunk] : p.dv_final[chunk];
    if (p.dk_final[chunk] != nullptr) {
      // the last block this chunk's gradient was waiting for: total = travelling sums + this block, rounded once
      const int64_t foff = b * p.dkfs[0] + hkv * p.dkfs[1] + static_cast<int64_t>(row) * p.dkfs[2];
      wave_store_rows_total<D, 64>(region, part, scale, accumulate ? static_cast<const float*>(dst) + off : nullptr, p.dks[2], total + foff, p.dkfs[2], rows_live, lane);
    } else if (p.dkv_f32) {
      wave_store_rows<D, true, 64>(region, part, scale, static_cast<float*>(dst) + off, p.dks[2], rows_live, lane, accumulate, false);
    } else {
      wave_store_rows<D, false, 64>(region, part, scale, static_cast<__bf16*>(dst) + off, p.dks[2], rows_live, lane, false, kStreamGrads);
    }
  });
}

__device__ __forceinline__ void role_clear(f32x4 (&acc)[8][4]) {
#pragma unroll
  for (int db = 0; db < 8; ++db)
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) acc[db][kb] = f32x4{0.f, 0.f, 0.f, 0.f};
}

// Where a workgroup's walk is: (query head of the group) x (tiles of 64 queries that see its first key)
struct RoleWalk {
  int b, hkv, head_first, qt_start, n_qtiles, n_tiles;
};

template <bool kDk>   // the wave that has dP and dK, or the one that has S and dV
__device__ __forceinline__ void role_walk(const BwdParams& p, const KeyTile& at, const RoleWalk& walk, f32x4 (&acc)[8][4]) {
  using C = RoleCfg;
  using L = C::L;
  constexpr int D = C::D, BM = C::BM;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  const AttnParams& a = p.a;
  const int tid = threadIdx.x, lane = tid % 64, wave_id = __builtin_amdgcn_readfirstlane(tid / 64), pair = wave_id % C::kPairs;
  // (scalars, and below the lane's offsets and constants worked out where they are used: the walk needs every register)
  const float c = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(a.sm_scale * kLog2e)));

  // ---- the fragments of the wave's 64 keys of K, or of V (B operand: lane = key, 8 consecutive d per k step), fetched row-major; the
  //      first tile's loads follow before anything waits
  bf16x8 kv[4][D / 32];
  WaveTile<D> rows[2];
  {
    const int64_t* const stride = kDk ? a.vs : a.ks;
    const __bf16* const base = (kDk ? a.kv.v[at.chunk] : a.kv.k[at.chunk]) + walk.b * stride[0] + walk.hkv * stride[1];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int row0 = at.row0 + 128 * i + 16 * pair;
      rows[i].template issue<64>(make_buffer(base + static_cast<int64_t>(row0) * stride[2], span_bytes(a.kv.len - row0, stride[2], D)), stride[2], lane);
    }
  }

  // ---- tiles of Q and dO straight to LDS, their lse (by the first S wave) and delta (the first dP wave) through a register, see attn_bwd_dkdv_tile
  const uint32_t q_step = static_cast<uint32_t>(BM * a.qs[2] * 2), do_step = static_cast<uint32_t>(BM * a.os[2] * 2);
  struct Cursor {
    int tile, head;                  // query tile within the head, query head
    const char *q, *dout;            // first row of the tile
    const float* per_row;            // its lse or delta
    uint32_t q_left, do_left, rows_left;  // bytes from there to the end of the head's rows
  } cur;
  auto seek = [&](int head, int tile) {
    const int q0 = tile * BM;
    cur.tile = tile;
    cur.head = head;
    cur.q = reinterpret_cast<const char*>(a.q + walk.b * a.qs[0] + head * a.qs[1] + static_cast<int64_t>(q0) * a.qs[2]);
    cur.dout = reinterpret_cast<const char*>(p.dout + walk.b * a.os[0] + head * a.os[1] + static_cast<int64_t>(q0) * a.os[2]);
    cur.per_row = (kDk ? p.delta : p.lse) + (static_cast<int64_t>(walk.b) * a.Hq + head) * a.Sq + q0;
    cur.q_left = span_bytes(a.Sq - q0, a.qs[2], D);
    cur.do_left = span_bytes(a.Sq - q0, a.os[2], D);
    cur.rows_left = static_cast<uint32_t>(a.Sq - q0) * 4u;
  };
  auto advance = [&]() {
    if (cur.tile + 1 == walk.n_qtiles) {
      seek(cur.head + 1, walk.qt_start);
    } else {
      ++cur.tile;
      cur.q += q_step;  cur.q_left -= q_step;
      cur.dout += do_step;  cur.do_left -= do_step;
      cur.per_row += BM;  cur.rows_left -= BM * 4;
    }
  };
  auto request_tile = [&](uint32_t buf_off, float& row_reg) __attribute__((always_inline)) {
    if (pair == 0) row_reg = buffer_load_f32(make_buffer(cur.per_row, cur.rows_left), lane_here() * 4u);
    // (a wave's second KiB of a tile holds the rows two behind its first's: the same offsets in a window that begins two rows later)
    static_assert(C::kLoads == 2);
    const int lane = lane_here(), r = L::row(wave_id, lane), cv = L::column(lane);
    auto request = [&](const char* first, uint32_t left, int64_t stride, uint32_t to) __attribute__((always_inline)) {
      const uint32_t off = (static_cast<uint32_t>(r) * static_cast<uint32_t>(stride) + cv) * 2;
      const uint64_t base = reinterpret_cast<uint64_t>(first), two_rows = static_cast<uint64_t>(stride) * 4;
      request16_to<0>(to, request_window(base, left), off);
      request16_to<C::NW * L::kPitch>(to, request_window(base + two_rows, left > two_rows ? left - static_cast<uint32_t>(two_rows) : 0), off);
    };
    const uint32_t to = buf_off + wave_id * L::kPitch;
    request(cur.q, cur.q_left, a.qs[2], to);
    request(cur.dout, cur.do_left, a.os[2], to + C::kSide);
  };
  auto stage = [&](uint32_t buf_off, float row_reg) __attribute__((always_inline)) {   // (the tile still under the cursor)
    if (pair != 0) return;
    float v = -row_reg;   // -delta: dP starts there (0 past Sq)
    // rows past Sq, and rows whose lse is -inf (they saw no key), get lse = +inf so that P = 0
    const uint32_t at = lane_here() * 4u;
    if constexpr (!kDk) {
      uint32_t inf = 0x7f800000;
      asm volatile("" : "+s"(inf));
      v = at < cur.rows_left && row_reg != -INFINITY ? row_reg * kLog2e : __uint_as_float(inf);
    }
    *reinterpret_cast<float*>(smem_raw + buf_off + C::kRowsAt + (kDk ? BM * 4 : 0) + at) = v;
  };

  seek(walk.head_first, walk.qt_start);
  float first_row = 0.f;
  request_tile(0, first_row);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    bf16x8 f[2][D / 32];
    rows[i].fragments16(smem_raw + C::kTileBytes + wave_id * WaveTile<D>::kRegionBytes, lane, f);
#pragma unroll
    for (int s = 0; s < D / 32; ++s) { kv[2 * i][s] = f[0][s]; kv[2 * i + 1][s] = f[1][s]; }
  }
  stage(0, first_row);
  // the lane's places: in Q's or dO's rows (S: Q's, dP: dO's), for the transposing reads of the other, in its rows' lse or -delta, in P
  uint32_t row_at = (kDk ? C::kSide : 0) + L::row_place16(lane), tr_at = (kDk ? 0 : C::kSide) + L::column_place16(lane);
  uint32_t per_row_at = C::kRowsAt + (kDk ? BM * 4 : 0) + L::group_row(lane / 16) * 4, p_at = C::kTileBytes + pair * C::kPairBytes + lane * 16;
  asm volatile("" : "+v"(row_at), "+v"(tr_at), "+v"(per_row_at), "+v"(p_at));
  __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);
  __syncthreads();
  role_clear(acc);

  // A head's walk is counted in steps of 32 queries, u; `left` tiles follow the one that the wave is in.
  int u = 2 * walk.qt_start, left = walk.n_tiles - 1;
  uint32_t buf_off = 0;          // the wave's tile of LDS
  const int base = at.key0 + 16 * pair - a.q_offset;   // the step position (times 32) at which the wave's first key is the first query
  bf16x8 from[2][4];
  f32x4 first_start;
  auto fetch = [&](int qb, int s) { from[qb][s] = lds_at<bf16x8>(row_at + (qb * L::kRows16 + L::column16(s) * 2)); };
  auto first_fetch = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int s = 0; s < 4; ++s) fetch(0, s);
    first_start = lds_at<f32x4>(per_row_at);   // lse, or -delta
  };
  // One step: kKb of the four key blocks have a query that sees them (0: none, and only the step's duties are done).
  auto step = [&](auto kb_c, auto mask_c) __attribute__((always_inline)) {
    constexpr int kKb = decltype(kb_c)::value;
    constexpr bool kMask = decltype(mask_c)::value;
    const int second = u & 1;   // half of a tile
    // the next tile goes where the dP waves were done a step ago with the last one: while the S waves have the second half of a tile
    const bool requests = second == (kDk ? 0 : 1) && left > 0;
    float row_reg;   // (of this step alone: a value that outlives it is copied, and waited for, where it was asked for)
    auto request_next = [&]() __attribute__((always_inline)) {
      if (requests) {
        advance();
        request_tile(buf_off ^ static_cast<uint32_t>(C::kBufBytes), row_reg);
      }
    };
    if constexpr (kKb == 0) request_next();
    // (the places move in their registers: another of each kind would not fit)
    const int flip = buf_off == 0 ? C::kBufBytes : -C::kBufBytes, rows = second ? flip - L::kRows32 : L::kRows32;
    auto move_on = [&]() __attribute__((always_inline)) {
      row_at += rows;
      per_row_at += second ? flip - 128 : 128;
      p_at += second ? -C::kPBytes : C::kPBytes;
    };
    if constexpr (kKb > 0) {
      // Block after block of 16 queries x 16 keys; the vector work of the block before is dealt out between a block's four MFMAs.  The fragments of
      // a product's 16 queries are held for its kKb blocks, and those of the next are requested where they are last used.
      constexpr int kBlocks = 2 * kKb, kAhead = 2;
      bf16x8 tr[8];
      auto fetch_tr = [&](int db) { tr[db] = lds_tr16_at<D>(tr_at + db * 32); };
      f32x4 x[kBlocks], start[2], prob[kBlocks];
      u32x4 right[kKb];   // P or dS, rounded: 32 queries and 16 keys, an operand
      // (the dP wave comes second at every turn, being the younger of its SIMD, and is the one that its pair waits for)
      if constexpr (!kDk) first_fetch();
      else __builtin_amdgcn_s_setprio(1);
      start[0] = first_start;
      // (a key is masked for the query of register i iff key_rel > i)
      int key_rel = -0x10000000;
      if constexpr (kMask && !kDk) {
        const int lane = lane_here();
        if (a.causal) key_rel = base + lane % 16 - 32 * u - L::group_row(lane / 16);
      }
      auto read_p = [&](auto block_c) __attribute__((always_inline)) {
        constexpr int block = decltype(block_c)::value;
        if constexpr (kDk) prob[block] = lds_at<f32x4>(p_at + (block / kKb * 4 + block % kKb) * 1024);
      };
      read_p(std::integral_constant<int, 0>());
      // element i of a block: S -> P, or dP -> dS; with its last one it is rounded, and P goes to the dP wave
      auto element = [&](auto block_c, auto i_c) __attribute__((always_inline)) {
        constexpr int block = decltype(block_c)::value, qb = block / kKb, kb = block % kKb, i = decltype(i_c)::value;
        if constexpr (kDk) {
          x[block][i] *= prob[block][i];
        } else {
          x[block][i] = fast_exp2(x[block][i] * c - start[qb][i]);
          if (kMask && key_rel + 64 * kb - 16 * qb > i) x[block][i] = 0.f;
        }
        if constexpr (i == 3) {
          if constexpr (!kDk) *reinterpret_cast<__attribute__((address_space(3))) f32x4*>(p_at + (qb * 4 + kb) * 1024) = x[block];
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
            uint32_t two = __builtin_bit_cast(uint32_t, bf16x2{static_cast<__bf16>(x[block][2 * j]), static_cast<__bf16>(x[block][2 * j + 1])});
            asm volatile("" : "+v"(two));   // (rounded here: at its place the four values would be held till then)
            right[kb][2 * qb + j] = two;
          }
        }
      };
      __builtin_amdgcn_sched_barrier(0);
      each_load<kBlocks>([&](auto block_c) __attribute__((always_inline)) {
        constexpr int block = decltype(block_c)::value, qb = block / kKb, kb = block % kKb;
        each_load<4>([&](auto s_c) __attribute__((always_inline)) {
          constexpr int s = decltype(s_c)::value;
          const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
          x[block] = mfma16(from[qb][s], kv[kb][s], s == 0 ? (kDk ? start[qb] : zero) : x[block]);
          if constexpr (block == kKb - 1) fetch(1, s);
          if constexpr (kDk ? block == kKb - 1 && s == 0 : block == kKb && s == 2) start[1] = lds_at<f32x4>(per_row_at + 64);
          if constexpr (s == 3 && block + 1 < kBlocks) read_p(std::integral_constant<int, (block + 1 < kBlocks ? block + 1 : 0)>());
          if constexpr (block == kBlocks - 1 && s == 3) fetch_tr(0);
          if constexpr (block == 0 && s == 3) request_next();   // (scalar work for the most part: behind products that are on their way)
          // (an MFMA behind the block's last: its results are there then)
          if constexpr (kDk) {   // (two at a time, which frees P of the block for the next)
            if constexpr (block > 0 && (s == 1 || s == 2)) {
              constexpr int prev = block > 0 ? block - 1 : 0, first = s == 2 ? 2 : 0;
              element(std::integral_constant<int, prev>(), std::integral_constant<int, first>());
              element(std::integral_constant<int, prev>(), std::integral_constant<int, first + 1>());
            }
          } else {
            if constexpr (block > 0 && s > 0) element(std::integral_constant<int, (block > 0 ? block - 1 : 0)>(), std::integral_constant<int, (s > 0 ? s - 1 : 0)>());
            if constexpr (block > 1 && s == 0) element(std::integral_constant<int, (block > 1 ? block - 2 : 0)>(), std::integral_constant<int, 3>());
          }
          __builtin_amdgcn_sched_barrier(0);
        });
      });
      fetch_tr(1);
      if constexpr (kDk) __builtin_amdgcn_s_setprio(0);
      if constexpr (!kDk) element(std::integral_constant<int, kBlocks - 2>(), std::integral_constant<int, 3>());
      each_load<4>([&](auto i_c) __attribute__((always_inline)) { element(std::integral_constant<int, kBlocks - 1>(), i_c); });
      __builtin_amdgcn_sched_barrier(0);
      each_load<8>([&](auto block) __attribute__((always_inline)) {
        constexpr int db = decltype(block)::value;
        if constexpr (db + kAhead < 8) fetch_tr(db + kAhead);
        if constexpr (db == 2) move_on();
        if constexpr (db == 6) tr_at += rows;
        if constexpr (db == 6 && kDk) first_fetch();
        // (key blocks there and back: from each product to the next one operand stays.  17 launches 0.998 of the time, 4096 queries and 32768 keys with
        // 32 / 8 heads 3060 -> 3045 us)
#pragma unroll
        for (int to = 0; to < kKb; ++to) {
          const int kb = db % 2 ? kKb - 1 - to : to;
          acc[db][kb] = mfma16(tr[db], __builtin_bit_cast(bf16x8, right[kb]), acc[db][kb]);
        }
        __builtin_amdgcn_sched_barrier(0);
      });
    }
    if constexpr (kKb == 0) {
      move_on();
      tr_at += rows;
      if constexpr (kDk) first_fetch();
    }
    if (requests) stage(buf_off ^ static_cast<uint32_t>(C::kBufBytes), row_reg);
    buf_off ^= second ? static_cast<uint32_t>(C::kBufBytes) : 0u;
    left -= second ? 1 : 0;
    ++u;
    // (the compiler has to see this wait: for the row's load, which it cannot tell is always waited for, it would wait in front of the products)
    __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);
    __syncthreads();
  };
  auto only_duties = [&]() { __builtin_amdgcn_s_waitcnt(kWaitVmcnt0); __syncthreads(); };

  // Key blocks with rows in the chunk, and those of them that a step's last query sees: one more every two steps of a head's walk.  Each number has
  // a loop of its own: a branch inside a step has the compiler move the accumulators.
  const int live = min(max((a.kv.len - at.row0 - 16 * pair + 63) / 64, 0), 4);
  constexpr int kNever = 1 << 30;
  auto from_step = [&](int kb) { return kb > live ? kNever : a.causal ? (base >> 5) + 2 * (kb - 1) : 0; };   // the first that sees kb blocks
  const int plain_from = live < 4 ? kNever : a.causal ? (base + 3 * 64 + 15 + 31) >> 5 : 0;                  // ... all pairs of four
  auto steps = [&](auto kb_c, auto mask_c, int upto) __attribute__((always_inline)) {
    while (u < upto) step(kb_c, mask_c);
  };
  if (kDk) {
    only_duties();
    first_fetch();
  }
  while (true) {
    const int end = min(2 * walk.n_qtiles, u + 2 * left + 2);   // (a head begins and ends with a tile)
    steps(std::integral_constant<int, 0>(), std::true_type(), min(from_step(1), end));
    steps(std::integral_constant<int, 1>(), std::true_type(), min(from_step(2), end));
    steps(std::integral_constant<int, 2>(), std::true_type(), min(from_step(3), end));
    steps(std::integral_constant<int, 3>(), std::true_type(), min(from_step(4), end));
    steps(std::integral_constant<int, 4>(), std::true_type(), min(plain_from, end));
    steps(std::integral_constant<int, 4>(), std::false_type(), end);
    if (left < 0) break;
    u = 2 * walk.qt_start;
  }
  if (!kDk) only_duties();
}

// grid = (Hkv * B, key tiles of 256): every head's first tile, the longest under a causal mask, first
__global__ __launch_bounds__(512, 2) void attn_bwd_roles_kernel(const BwdParams p) {
  const Arguments<offsetof(BwdParams, dk), offsetof(BwdParams, dk_final), offsetof(BwdParams, dv), offsetof(BwdParams, dv_final), offsetof(BwdParams, dkfs),
                  sizeof(BwdParams) - 4> gradients;
  AttnArguments().arrive();
  gradients.arrive();
  using C = RoleCfg;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  const AttnParams& a = p.a;
  // what the workgroup does (found again after the walk, which leaves no registers for it)
  struct Task {
    KeyTile at;
    RoleWalk walk;
  };
  auto find = [&]() __attribute__((always_inline)) {
    int x = blockIdx.x, y = blockIdx.y;
    asm volatile("" : "+s"(x), "+s"(y));
    Task t;
    t.at = key_tile(a.kv, y, C::BN);
    RoleWalk& walk = t.walk;
    walk.hkv = x % a.Hkv;
    walk.b = x / a.Hkv;
    walk.n_qtiles = (a.Sq + C::BM - 1) / C::BM;
    walk.qt_start = first_query_tile(a, t.at.key0, C::BM);
    walk.n_tiles = max(walk.n_qtiles - walk.qt_start, 0) * (a.Hq / a.Hkv);
    walk.head_first = walk.hkv * (a.Hq / a.Hkv);
    return t;
  };
  f32x4 acc[8][4];
  const int wave_id = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), pair = wave_id % C::kPairs;
  const bool is_dk = wave_id >= C::kPairs;
  {
    const Task t = find();
    if (p.dk[t.at.chunk] == nullptr && p.dk_final[t.at.chunk] == nullptr) return;   // this chunk's gradient is not wanted (uniform over the workgroup)
    if (t.walk.n_tiles == 0) role_clear(acc);
    else if (is_dk) role_walk<true>(p, t.at, t.walk, acc);
    else role_walk<false>(p, t.at, t.walk, acc);
  }
  // (LDS is free now: the walk ended on a barrier)
  const Task t = find();
  const int lane = lane_here();
  unsigned char* const region = smem_raw + wave_id * kRowRegionBytes;
  if (is_dk) role_store<true>(p, region, acc, t.at.chunk, t.walk.b, t.walk.hkv, t.at.row0 + 16 * pair, t.at.key0 + 16 * pair, lane);
  else role_store<false>(p, region, acc, t.at.chunk, t.walk.b, t.walk.hkv, t.at.row0 + 16 * pair, t.at.key0 + 16 * pair, lane);
}

}  // namespace

int launch_dkdv_roles(const BwdParams& p, hipStream_t s) {
  using C = RoleCfg;
  static LdsOnce reserved;
  if (!reserve_lds_once(reserved, reinterpret_cast<const void*>(&attn_bwd_roles_kernel), C::kLdsBytes))
    return fail(PICO_ERR_LAUNCH, "pico_attn_bwd(dk/dv): cannot reserve %zu bytes of LDS", C::kLdsBytes);
  hipLaunchKernelGGL(attn_bwd_roles_kernel, dim3(p.a.Hkv * p.a.B, tiles_before(p.a.kv, p.a.Sk, C::BN)), dim3(C::kThreads), C::kLdsBytes, s, p);
  return PICO_OK;
}

}  // namespace pico
