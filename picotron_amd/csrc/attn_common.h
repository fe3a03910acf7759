// Pieces shared by the attention forward and backward kernels (gfx950, wave64, MFMA 32x32x16 and 16x16x32 bf16).
//
// MFMA 32x32x16 operand layout (verified on hardware): lane l, half h = l / 32, n = l % 32
//   A[m][k]  : lane holds m = n, k = 8h .. 8h+7          (8 bf16)
//   B[k][n]  : lane holds n,     k = 8h .. 8h+7          (8 bf16)
//   C[m][n]  : lane holds column n, register i holds row 8*(i/4) + 4h + i%4   (16 fp32)
// The sum over k does not care which physical index sits in slot k as long as A and B agree, so a
// C tile can be fed back as the k-operand of the next MFMA straight from registers: registers
// 8c .. 8c+7 of a lane hold rows {16c + 8jj + 4h + t : jj < 2, t < 4}, and the partner operand is
// fetched with that same row order.
//
// MFMA 16x16x32: lane l, group g = l / 16, n = l % 16
//   A[m][k]  : lane holds m = n, k = 8g .. 8g+7          (8 bf16)
//   B[k][n]  : lane holds n,     k = 8g .. 8g+7          (8 bf16)
//   C[m][n]  : lane holds column n, register i holds row 4g + i                   (4 fp32)
// Two C tiles' registers are 8 slots k of the next product, 4 rows of the one and 4 of the other.  Which row and which columns of a tile in
// LDS stand for m and k is TileLayout's (group_row, column16 and group_column, the same in A and B).
//
// ds_read_b64_tr_b16 (verified on hardware): within a group of 16 lanes, lane p supplies the address
// of 4 consecutive 16-bit elements; lane p receives element p%4 of lanes {p/4, 4 + p/4, 8 + p/4, 12 + p/4}.
// With lane p pointing at tile[row0 + p/4][col0 + 4*(p%4)] every lane p ends up with
// tile[row0 .. row0+3][col0 + p]: a 4-deep column of a row-major tile, which is what an MFMA operand
// needs when the contraction index is the tile's row.
#pragma once
#include <type_traits>
#include "common.h"

namespace pico {

typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

__device__ __forceinline__ f32x16 mfma32(bf16x8 a, bf16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mfma16(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// 4 rows x 1 column of a row-major bf16 tile in LDS, transposed into the lane (see header comment).
// `p` must point at tile[row0 + (lane%16)/4][col0 + 4*(lane%4)].
__device__ __forceinline__ s16x4 lds_read_tr(const __bf16* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p));
}

// Two transposed reads -> the 8 k-slots of an MFMA operand.  Slots 0-3 come from rows
// row0 .. row0+3, slots 4-7 from rows row0+8 .. row0+11 (the register order of a C tile): the second read lies `step` elements
// after the first (rows need not be evenly spaced).
__device__ __forceinline__ bf16x8 lds_read_tr_pair_step(const __bf16* p, int step) {
  s16x4 lo = lds_read_tr(p);
  s16x4 hi = lds_read_tr(p + step);
  typedef __attribute__((ext_vector_type(8))) short s16x8;
  s16x8 v = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  return __builtin_bit_cast(bf16x8, v);
}

// s_waitcnt immediate for "vmcnt(0)" with the other counters left at their maxima (gfx9 encoding:
// vmcnt[3:0] | expcnt[6:4] | lgkmcnt[11:8] | vmcnt_hi[15:14])
constexpr int kWaitVmcnt0 = 0x0F70;

// ---- buffer loads.  A buffer resource (4 SGPRs: base, byte count) plus a 32-bit per-lane byte offset replaces
// 64-bit per-lane addresses; a lane whose offset is past the byte count reads zeros, which is how tile rows
// past the end of a sequence become zero rows without clamps or selects.
using buffer_rsrc = __amdgpu_buffer_rsrc_t;
// `bytes` is the exact size of the window: the entry points reject tensors whose rows of one head span 4 GiB or more
__device__ __forceinline__ buffer_rsrc make_buffer(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, static_cast<int>(bytes), 0x00020000);
}
// bytes from the first element of row 0 to the end of row rows-1, for rows of D bf16 elements `stride` elements apart
__device__ __forceinline__ uint32_t span_bytes(int rows, int64_t stride, int D) {
  return rows <= 0 ? 0u : static_cast<uint32_t>((static_cast<int64_t>(rows - 1) * stride + D) * 2);
}
__device__ __forceinline__ u32x4 buffer_load_b128(buffer_rsrc r, uint32_t byte_off) {
  return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, static_cast<int>(byte_off), 0, 0));
}
__device__ __forceinline__ float buffer_load_f32(buffer_rsrc r, uint32_t byte_off) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, static_cast<int>(byte_off), 0, 0));
}

// ---- loads that go to LDS without passing the registers: 16 bytes per lane, lane after lane from m0 on; zeros past the window.
// In assembly, because the compiler makes every later read of LDS wait for the builtin: the caller waits by hand
// (wait_requests) before the barrier that publishes the tile.  A spill to scratch would be counted in a request's place, and
// the kernel's dynamic LDS has to start at 0 (no static LDS): the build refuses kernels that have either.  m0 is an output of what
// writes it and an operand of what reads it, so that the compiler keeps nothing of its own there across a request and puts nothing
// there between the two statements.
template <int kPlus>
__device__ __forceinline__ uint32_t aim_request(uint32_t lds_off) {   // one instruction has to lie between this and the request
  uint32_t aim;
  asm volatile("s_add_u32 %0, %1, %2" : "={m0}"(aim) : "s"(lds_off), "n"(kPlus) : "scc", "memory");
  return aim;
}
__device__ __forceinline__ void request16(uint32_t aim, u32x4 window, uint32_t off) {
  asm volatile("buffer_load_dwordx4 %0, %1, 0 offen lds" ::"v"(off), "s"(window), "{m0}"(aim) : "memory");
}
template <int kPlus>
__device__ __forceinline__ void request16_to(uint32_t lds_off, u32x4 window, uint32_t off) {
  uint32_t aim;
  asm volatile("s_add_u32 %0, %1, %2\n\ts_nop 0\n\tbuffer_load_dwordx4 %3, %4, 0 offen lds"
               : "=&{m0}"(aim) : "s"(lds_off), "n"(kPlus), "v"(off), "s"(window) : "scc", "memory");
}
// all but the wave's newest N vector memory operations are complete
template <int N>
__device__ __forceinline__ void wait_requests() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// a buffer resource in scalar registers, for the requests (base and bytes uniform over the wave)
__device__ __forceinline__ u32x4 request_window(uint64_t base, uint32_t bytes) {
  u32x4 r;
  r[0] = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(base));
  r[1] = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(base >> 32) & 0xffffu);
  r[2] = __builtin_amdgcn_readfirstlane(bytes);
  r[3] = 0x00020000;
  return r;
}

// How K, V, Q and dO tiles lie in LDS, 64 rows at a time.  A request puts 1 KiB of consecutive addresses there, lane after lane, and
// every lane can ask for any 16 bytes of the tile; the KiBs lie 16 bytes further apart than they are long.  Rows share a KiB such that
// 16 consecutive ones start at 16 different places of the 64 banks, so reads by rows (16 lanes at a time: one piece of 16 rows) have no
// bank conflicts, and rows 4 g .. 4 g + 3 a quarter of the banks apart, so transposing ones (32 lanes at a time: 4 rows x 64 bytes) have
// none either.  And a lane's piece of any group of rows, any columns, lies at a constant distance from its first: one register per
// kind of read holds all addresses.  Before, dense rows whose pieces changed places with the row: eight addresses per kind of read
// at head_dim 128, kept in registers or flipped anew, and an addition in front of every read.  Forward at head_dim 128 221 -> 171
// registers, 16 of 180 vector instructions per trip less: B1 H32 S4096 136.2 -> 133.3 us in a long row of launches (D64 86.5 -> 84.3), its dK/dV 19 % fewer
// of them and 257 -> 250 us (matrix work at the power limit: 4 % fewer cycles); small launches gain more, B3 H9/3 S777 D64 12.4 -> 10.7,
// one rank's B1 H32 256 x 1024 13.3 -> 11.0.
// (Counted conflicts say how LDS takes a read: 16 lanes of a 16-byte one at a time, 32 of an 8-byte one.  A layout that spread the
// requests only over all 64 lanes doubled the pipe's cycles.)
template <int D>
struct TileLayout {
  static constexpr int kBlocks = D / 8, kPitch = 1024 + 16;   // KiBs of 64 rows, and from one to the next
  static constexpr int kRows64 = kBlocks * kPitch, kRows32 = 512, kRows16 = 256, kRows8 = 2 * kPitch;   // so many rows further
  static constexpr int rows(int n) { return n / 64 * kRows64 + n % 64 / 32 * kRows32; }
  static constexpr int bytes(int n) { return n / 64 * kRows64; }
  // the row and first column of what lane `lane` of the request of KiB `block` brings
  static __device__ __forceinline__ int row(int block, int lane) {
    const int at = block % kBlocks, slot = lane / (D / 8), r = D == 128 ? 16 * slot : 16 * (slot / 2) + 2 * (slot % 2);
    return block / kBlocks * 64 + at / 4 + 4 * (at % 4) + r;
  }
  static __device__ __forceinline__ int column(int lane) { return lane % (D / 8) * 8; }
  static __device__ __forceinline__ uint32_t place(int r) {   // of a row, of the first 64
    return D == 128 ? (r % 4 * 4 + r / 4 % 4) * kPitch + r / 16 * 256 : (r % 2 * 4 + r / 4 % 4) * kPitch + r / 16 * 256 + r % 4 / 2 * 128;
  }
  // the lane's place for reads by rows: row lane % 32, columns 8 (lane / 32) ..+7 (32 bytes further: the next 16 columns)
  static __device__ __forceinline__ uint32_t row_place(int lane) { return place(lane % 32) + lane / 32 * 16; }
  // ... and for transposing reads: row 4 (lane / 32) + lane % 16 / 4, columns 16 (lane / 16 % 2) + 4 (lane % 4) ..+3 (64 bytes further:
  // the next 32 columns)
  static __device__ __forceinline__ uint32_t column_place(int lane) { return place(4 * (lane / 32) + lane % 16 / 4) + lane / 16 % 2 * 32 + lane % 4 * 8; }
  // For products of 16 x 16 x 32, whose results have rows 4 (lane / 16) ..+3 in a lane: there the four groups of lanes stand for the rows from
  // 0, 8, 4 and 12, so that the 32 lanes of a transposing read, which fetch 8 rows x 32 bytes, have no bank conflicts (rows 0 .. 7 would share banks
  // in twos).  A 16-byte read is taken 16 lanes at a time, lanes 0-3, 12-15, 20-27 and 4-11, 16-19, 28-31 of each half: it has none if lanes 16 apart
  // read columns 32 apart, so a fragment's 32 columns of the contraction are 0-7, 32-39, 8-15, 40-47 (the next one's 16 further on), in both operands.
  // (With 32 consecutive columns every such read took eight cycles instead of four.)
  static __device__ __forceinline__ int group_row(int group) { return group % 2 * 8 + group / 2 * 4; }
  static __device__ __forceinline__ int group_column(int group) { return group % 2 * 32 + group / 2 * 8; }
  static constexpr int column16(int s) { return s / 2 * 64 + s % 2 * 16; }   // fragment s: columns column16(s) + group_column(lane / 16) ..+7
  // the lane's row of a read by rows; the first of its rows in a result is group_row(lane / 16); and of a transposing read, columns 4 (lane % 4) ..+3
  // (32 bytes further: the next 16 columns)
  static __device__ __forceinline__ uint32_t row_place16(int lane) { return place(group_row(lane / 4 % 4) + lane % 4) + group_column(lane / 16) * 2; }
  static __device__ __forceinline__ uint32_t column_place16(int lane) { return place(group_row(lane / 16) + lane % 16 / 4) + lane % 4 * 8; }
};
// LDS at a byte offset (the kernels' LDS starts at 0, see request16): through a pointer to the array the compiler adds its address,
// which it does not know to be 0, to every lane offset
template <typename T>
__device__ __forceinline__ T lds_at(uint32_t off) {
  return *reinterpret_cast<const __attribute__((address_space(3))) T*>(off);
}
// the 8 k-slots of an MFMA operand by two transposing reads: 4 rows at `off`, and 4 at 8 rows further
template <int D>
__device__ __forceinline__ bf16x8 lds_tr_at(uint32_t off) {
  const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<lds_s16x4*>(off));
  const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<lds_s16x4*>(off + TileLayout<D>::kRows8));
  typedef __attribute__((ext_vector_type(8))) short s16x8;
  return __builtin_bit_cast(bf16x8, static_cast<s16x8>(__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7)));
}

// ... of a 16 x 16 x 32 product: 16 rows at `off`, 4 of each lane, and the 16 rows after them
template <int D>
__device__ __forceinline__ bf16x8 lds_tr16_at(uint32_t off) {
  const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<lds_s16x4*>(off));
  const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<lds_s16x4*>(off + TileLayout<D>::kRows16));
  typedef __attribute__((ext_vector_type(8))) short s16x8;
  return __builtin_bit_cast(bf16x8, static_cast<s16x8>(__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7)));
}

// fn(integral_constant) for 0 .. N - 1
template <int N, typename Fn, int i = 0>
__device__ __forceinline__ void each_load(const Fn& fn) {
  if constexpr (i < N) {
    fn(std::integral_constant<int, i>());
    each_load<N, Fn, i + 1>(fn);
  }
}

__device__ __forceinline__ bf16x8 pack8(const f32x16& c, int base) {
  bf16x8 r;
#pragma unroll
  for (int e = 0; e < 8; ++e) r[e] = static_cast<__bf16>(c[base + e]);
  return r;
}

__device__ __forceinline__ bf16x8 pack8(const f32x4& lo, const f32x4& hi) {
  bf16x8 r;
#pragma unroll
  for (int e = 0; e < 4; ++e) { r[e] = static_cast<__bf16>(lo[e]); r[4 + e] = static_cast<__bf16>(hi[e]); }
  return r;
}

// max / sum of a value across the two 32-lane halves of a wave (lane l with lane l^32)
__device__ __forceinline__ float half_max(float v) {
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float half_sum(float v) {
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// ... across the four groups of 16 lanes (lanes l, l^16, l^32, l^48)
__device__ __forceinline__ float group_sum(float v) {
  auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return half_sum(__uint_as_float(r[0]) + __uint_as_float(r[1]));
}

// ---- reading a wave's 32 x D operand tile as MFMA fragments.  Fetched straight in fragment layout (lane =
// row, 16 bytes per lane) one instruction touches 32 different lines; fetched row-major -- 16 bytes per lane,
// 8 or 16 consecutive lanes per row -- the same bytes arrive in a quarter of the line requests, and a detour
// through a 32 x (D + 8) piece of LDS private to the wave turns them into fragments: lane n gets row n % 32,
// and for k step s the elements 16s + 8h ..+7 (h = lane / 32).  Rows past the end of the window read as zeros.
template <int D>
struct WaveTile {
  static constexpr int kChunks = D / 16;                 // 16-byte pieces per lane
  static constexpr int kRegionBytes = 32 * (D + 8) * 2;
  u32x4 raw[kChunks];
  template <int kSecond = 16>   // where the second 16 rows are, counted from the first
  __device__ __forceinline__ void issue(buffer_rsrc window, int64_t row_stride, int lane) {
#pragma unroll
    for (int i = 0; i < kChunks; ++i) {
      const int idx = lane + 64 * i, r = idx / (D / 8) + (2 * i >= kChunks ? kSecond - 16 : 0), cv = idx % (D / 8);
      raw[i] = buffer_load_b128(window, static_cast<uint32_t>((static_cast<int64_t>(r) * row_stride + cv * 8) * 2));
    }
  }
  static constexpr int kPitch = (D + 8) * 2;
  __device__ __forceinline__ void put(unsigned char* region, int lane) const {
#pragma unroll
    for (int i = 0; i < kChunks; ++i) {
      const int idx = lane + 64 * i, r = idx / (D / 8), cv = idx % (D / 8);
      *reinterpret_cast<u32x4*>(region + r * kPitch + cv * 16) = raw[i];
    }
  }
  __device__ __forceinline__ void fragments(unsigned char* region, int lane, bf16x8 (&frag)[D / 16]) const {
    put(region, lane);
    const int n = lane % 32, h = lane / 32;
#pragma unroll
    for (int s = 0; s < D / 16; ++s)
      frag[s] = *reinterpret_cast<const bf16x8*>(region + n * kPitch + (16 * s + 8 * h) * 2);
  }
  // ... of 16 x 16 x 32 products: frag[b][s] holds row 16 b + lane % 16, eight columns as TileLayout says
  __device__ __forceinline__ void fragments16(unsigned char* region, int lane, bf16x8 (&frag)[2][D / 32]) const {
    put(region, lane);
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int s = 0; s < D / 32; ++s)
        frag[b][s] = *reinterpret_cast<const bf16x8*>(region + (16 * b + lane % 16) * kPitch + (TileLayout<D>::column16(s) + TileLayout<D>::group_column(lane / 16)) * 2);
  }
};

// ---- writing a wave's 32 result rows.  The accumulators of the transposed products hold, per lane, one row
// (lane % 32) and, in registers 4j..4j+3 of block db, columns 32db + 8j + 4h ..+3 (h = lane / 32).  Stored
// straight from that layout a wave would touch 32 different 128-byte lines with 8 or 16 bytes each per
// instruction; instead the rows take a detour through a 32 x 144-byte piece of LDS that belongs to the wave
// (the caller guarantees that every wave of the workgroup is done with the tile buffers) and leave as whole
// 128-byte lines, 16 bytes per lane.  One pass moves 128 bytes of every row: 32 fp32 or 64 bf16 columns.
//   dst_row0: address of column 0 of the wave's first row; row_stride in elements; rows_live rows exist.
//   accumulate (fp32 only) adds to what is there; all its reads are issued before the first write.
//   streaming marks bf16 stores non-temporal (the data is not read again by the kernels that follow soon).
constexpr int kRowRegionBytes = 32 * 144;
// four columns of a row, scaled, to the wave's piece of LDS
template <bool kF32>
__device__ __forceinline__ void put_columns(unsigned char* region, int row, int col, f32x4 v4, float scale) {
  if constexpr (kF32) {
    *reinterpret_cast<f32x4*>(region + row * 144 + col * 4) = f32x4{v4[0] * scale, v4[1] * scale, v4[2] * scale, v4[3] * scale};
  } else {
    bf16x4 b4;
#pragma unroll
    for (int t = 0; t < 4; ++t) b4[t] = static_cast<__bf16>(v4[t] * scale);
    *reinterpret_cast<bf16x4*>(region + row * 144 + col * 2) = b4;
  }
}
// columns c0 .. c0 + kCols - 1 of the 32 rows
template <bool kF32, int kCols, int N>   // products of 32 x 32
__device__ __forceinline__ void put_rows(unsigned char* region, const f32x16 (&acc)[N], float scale, int c0, int lane) {
#pragma unroll
  for (int db = c0 / 32; db < (c0 + kCols) / 32; ++db)
#pragma unroll
    for (int j = 0; j < 4; ++j)
      put_columns<kF32>(region, lane % 32, 32 * db + 8 * j + 4 * (lane / 32) - c0,
                        f32x4{acc[db][4 * j], acc[db][4 * j + 1], acc[db][4 * j + 2], acc[db][4 * j + 3]}, scale);
}
// of 16 x 16: acc[db][kFrom + b] holds row 16 b + lane % 16, columns 16 db + 4 (lane / 16) ..+3
template <int kFrom, int N, int M>
struct RowPair {
  f32x4 (&acc)[N][M];
};
template <bool kF32, int kCols, int kFrom, int N, int M>
__device__ __forceinline__ void put_rows(unsigned char* region, const RowPair<kFrom, N, M>& rows, float scale, int c0, int lane) {
#pragma unroll
  for (int db = c0 / 16; db < (c0 + kCols) / 16; ++db)
#pragma unroll
    for (int b = 0; b < 2; ++b) put_columns<kF32>(region, 16 * b + lane % 16, 16 * db + 4 * (lane / 16) - c0, rows.acc[db][kFrom + b], scale);
}
// (kSecond: where the second 16 rows are, counted from the first)
template <int D, bool kF32, int kSecond = 16, typename Acc>
__device__ __forceinline__ void wave_store_rows(unsigned char* region, const Acc& acc, float scale,
                                                void* dst_row0, int64_t row_stride, int rows_live, int lane,
                                                bool accumulate, bool streaming) {
  constexpr int kPitch = 144;
  constexpr int kColsPerPass = kF32 ? 32 : 64;
#pragma unroll
  for (int c0 = 0; c0 < D; c0 += kColsPerPass) {
    put_rows<kF32, kColsPerPass>(region, acc, scale, c0, lane);
    // 32 rows x 8 pieces of 16 bytes = 4 pieces per lane; 8 consecutive lanes cover one row's line
    unsigned char* g[4];
    u32x4 v[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int idx = lane + 64 * t, ch = idx % 8, r = idx / 8 + t / 2 * (kSecond - 16);
      v[t] = *reinterpret_cast<const u32x4*>(region + idx / 8 * kPitch + ch * 16);
      g[t] = r < rows_live ? static_cast<unsigned char*>(dst_row0) +
                                 (static_cast<int64_t>(r) * row_stride + c0) * (kF32 ? 4 : 2) + ch * 16
                           : nullptr;
    }
    if constexpr (kF32) {
      f32x4 old[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) old[t] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (accumulate) {
#pragma unroll
        for (int t = 0; t < 4; ++t)
          if (g[t]) old[t] = *reinterpret_cast<const f32x4*>(g[t]);
      }
#pragma unroll
      for (int t = 0; t < 4; ++t)
        if (g[t]) *reinterpret_cast<f32x4*>(g[t]) = __builtin_bit_cast(f32x4, v[t]) + old[t];
    } else {
#pragma unroll
      for (int t = 0; t < 4; ++t)
        if (g[t]) {
          if (streaming) __builtin_nontemporal_store(v[t], reinterpret_cast<u32x4*>(g[t]));
          else *reinterpret_cast<u32x4*>(g[t]) = v[t];
        }
    }
  }
}

// The same rows as the sum of an fp32 buffer and the accumulators, rounded once to bf16 and written somewhere else:
// the last block of a ring adds itself to the travelling fp32 sums (`old_row0`, nullptr: nothing to add) and hands
// the total back in the dtype of the inputs.  32 columns per pass (fp32 staging), 8-byte bf16 pieces per lane.
template <int D, int kSecond = 16, typename Acc>
__device__ __forceinline__ void wave_store_rows_total(unsigned char* region, const Acc& acc, float scale,
                                                      const float* old_row0, int64_t old_stride, __bf16* dst_row0,
                                                      int64_t dst_stride, int rows_live, int lane) {
  constexpr int kPitch = 144;
#pragma unroll
  for (int c0 = 0; c0 < D; c0 += 32) {
    put_rows<true, 32>(region, acc, scale, c0, lane);
    f32x4 v[4], old[4];
    int row[4], piece[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int idx = lane + 64 * t;
      row[t] = idx / 8 + t / 2 * (kSecond - 16);
      piece[t] = idx % 8;
      v[t] = *reinterpret_cast<const f32x4*>(region + idx / 8 * kPitch + piece[t] * 16);
      old[t] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (old_row0 != nullptr && row[t] < rows_live)
        old[t] = *reinterpret_cast<const f32x4*>(old_row0 + static_cast<int64_t>(row[t]) * old_stride + c0 + piece[t] * 4);
    }
#pragma unroll
    for (int t = 0; t < 4; ++t)
      if (row[t] < rows_live) {
        bf16x4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = static_cast<__bf16>(v[t][e] + old[t][e]);
        __builtin_nontemporal_store(__builtin_bit_cast(u32x2, o),
                                    reinterpret_cast<u32x2*>(dst_row0 + static_cast<int64_t>(row[t]) * dst_stride + c0 + piece[t] * 4));
      }
  }
}

// ---- RoPE inside the attention kernels (non-interleaved: column d pairs with d + D/2; model.py:12-19).
// Tables are [rows, >= D/2 columns] with `pitch` elements between rows, bf16 or fp32; row index = position.
struct RopeArgs {
  const void* cos;   // nullptr: no rotation
  const void* sin;
  int64_t pitch;
  int f32;
  int q_pos0, k_pos0;   // position of query row 0 / key row 0
};
// n (4 or 8) consecutive table entries starting at column `col` of row `pos`
template <int N>
__device__ __forceinline__ void rope_load(const RopeArgs& r, const void* table, int pos, int col, float (&out)[N]) {
  if (r.f32) {
    const float* t = static_cast<const float*>(table) + static_cast<int64_t>(pos) * r.pitch + col;
#pragma unroll
    for (int e = 0; e < N; e += 4) {
      const f32x4 v = *reinterpret_cast<const f32x4*>(t + e);
#pragma unroll
      for (int u = 0; u < 4; ++u) out[e + u] = v[u];
    }
  } else {
    const __bf16* t = static_cast<const __bf16*>(table) + static_cast<int64_t>(pos) * r.pitch + col;
#pragma unroll
    for (int e = 0; e < N; e += 4) {
      const u32x2 v = *reinterpret_cast<const u32x2*>(t + e);
      out[e] = __uint_as_float(v[0] << 16);  out[e + 1] = __uint_as_float(v[0] & 0xffff0000u);
      out[e + 2] = __uint_as_float(v[1] << 16);  out[e + 3] = __uint_as_float(v[1] & 0xffff0000u);
    }
  }
}
// Rotates a lane's operand fragments in place: fragment s holds columns 16 s + 8 h ..+7 of the lane's row, its partner
// (column + D/2) is fragment s + D/32.  fp32 arithmetic, one rounding, the formula of the stand-alone kernel.
template <int D>
__device__ __forceinline__ void rope_rotate_fragments(bf16x8 (&f)[D / 16], const RopeArgs& r, int pos, int h) {
#pragma unroll
  for (int s = 0; s < D / 32; ++s) {
    float c[8], sn[8];
    rope_load<8>(r, r.cos, pos, 16 * s + 8 * h, c);
    rope_load<8>(r, r.sin, pos, 16 * s + 8 * h, sn);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float lo = static_cast<float>(f[s][e]), hi = static_cast<float>(f[s + D / 32][e]);
      f[s][e] = static_cast<__bf16>(lo * c[e] - hi * sn[e]);
      f[s + D / 32][e] = static_cast<__bf16>(hi * c[e] + lo * sn[e]);
    }
  }
}
// Un-rotates (rotation by the negative angle: the backward of RoPE) a lane's row of a transposed-product accumulator:
// registers 4j..4j+3 of block db hold columns 32 db + 8 j + 4 h ..+3; the partner of block db is block db + D/64.
template <int D>
__device__ __forceinline__ void rope_unrotate_acc(f32x16 (&acc)[D / 32], const RopeArgs& r, int pos, int h) {
#pragma unroll
  for (int db = 0; db < D / 64; ++db)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float c[4], sn[4];
      rope_load<4>(r, r.cos, pos, 32 * db + 8 * j + 4 * h, c);
      rope_load<4>(r, r.sin, pos, 32 * db + 8 * j + 4 * h, sn);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const float lo = acc[db][4 * j + t], hi = acc[db + D / 64][4 * j + t];
        acc[db][4 * j + t] = lo * c[t] + hi * sn[t];
        acc[db + D / 64][4 * j + t] = hi * c[t] - lo * sn[t];
      }
    }
}

// ... of 16 x 16 products, whose rows are at positions pos[b]
template <int D, int kFrom, int N, int M>
__device__ __forceinline__ void rope_unrotate_acc(const RowPair<kFrom, N, M>& rows, const RopeArgs& r, const int (&pos)[2], int lane) {
#pragma unroll
  for (int db = 0; db < D / 32; ++db)
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      f32x4 &first = rows.acc[db][kFrom + b], &second = rows.acc[db + D / 32][kFrom + b];
      float c[4], sn[4];
      rope_load<4>(r, r.cos, pos[b], 16 * db + 4 * (lane / 16), c);
      rope_load<4>(r, r.sin, pos[b], 16 * db + 4 * (lane / 16), sn);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const float lo = first[t], hi = second[t];
        first[t] = lo * c[t] + hi * sn[t];
        second[t] = hi * c[t] - lo * sn[t];
      }
    }
}

// K / V as a list of equally long chunks that lie one after another along the key axis: key j of the launch is row
// j % len of chunk j / len.  One chunk of len = Sk is the plain case.  A staged key tile belongs to one chunk: with a len
// that is no multiple of the tile the last tile of every chunk is a partial one (its rows past the chunk read as zeros and
// are masked), and tiles are counted chunk by chunk.
constexpr int kMaxChunks = PICO_MAX_KV_CHUNKS;
struct KvChunks {
  const __bf16* k[kMaxChunks];
  const __bf16* v[kMaxChunks];
  int count, len;
};

// A launch that is cut into pieces: too few workgroups for the GPU, or a few long ones among many short (under a causal
// mask, and with the query heads of a GQA group walked by one workgroup in dK/dV).  The trips of an output tile are dealt
// to ceil(trips / len) workgroups; where that is more than one, each leaves its accumulators in `ws` as they lie in its
// registers, and a second launch adds the pieces of a tile in their order and runs the kernel's own epilogue on the sum.
// Before and after, us: dK/dV of B1 H8/2 S2048 D64 144 -> 31, B2 H32/8 S1531 D128 143 -> 97, B8 H4/1 S7729 D64 655 -> 505,
// B1 H12/4 S3000 D128 200 -> 87; forward and dQ of one head of 4000 rows 48 -> 21 and 44 -> 19.
struct Pieces {
  int len;     // most trips of a piece; 0: tiles are not cut
  float* ws;
};

struct AttnParams {
  const __bf16* q;
  KvChunks kv;
  int B, Hq, Hkv, Sq, Sk;
  int causal, q_offset;
  float sm_scale;
  int64_t qs[3], ks[3], vs[3], os[3];
  Pieces pieces;
};

__host__ __device__ inline int pieces_of(int trips, int len) { return len <= 0 || trips <= len ? 1 : (trips + len - 1) / len; }

// The lane, counted anew where it is used: kept in a register (threadIdx is one) it costs the kernels that need all of theirs.
__device__ __forceinline__ int lane_here() {
  uint32_t all = ~0u;
  asm volatile("" : "+s"(all));
  return __builtin_amdgcn_mbcnt_hi(all, __builtin_amdgcn_mbcnt_lo(all, 0));
}

// Which (tile, piece) workgroup `y` of a head is, tiles in order, and how many pieces its tile has.  64 tiles at a time, one
// per lane: a prefix sum over their numbers of pieces and a ballot.  All lanes of the wave take part.
struct Piece {
  int tile, part, parts;
};
template <typename F>
__device__ __forceinline__ Piece find_piece(int y, int n_tiles, int len, const F& trips_of) {
  const int lane = lane_here();
  for (int base = 0; base < n_tiles; base += kWave) {
    const int mine = base + lane < n_tiles ? pieces_of(trips_of(base + lane), len) : 0;
    int sum = mine;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
      const int left = __shfl_up(sum, off, kWave);
      if (lane >= off) sum += left;
    }
    const uint64_t past = __ballot(sum > y);
    if (past != 0) {
      const int at = __builtin_ctzll(past);
      const int parts = __builtin_amdgcn_readlane(mine, at), upto = __builtin_amdgcn_readlane(sum, at);
      return {base + at, y - (upto - parts), parts};
    }
    y -= __builtin_amdgcn_readlane(sum, kWave - 1);
  }
  return {n_tiles - 1, 0, 0};   // (not reached: the grid has as many workgroups as there are pieces)
}
// the number of pieces in front of `tile`, i.e. the y of its first one
template <typename F>
__device__ __forceinline__ int first_piece(int tile, int len, const F& trips_of) {
  const int lane = threadIdx.x % kWave;
  int sum = 0;
  for (int i = lane; i < tile; i += kWave) sum += pieces_of(trips_of(i), len);
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) sum += __shfl_xor(sum, off, kWave);
  return __builtin_amdgcn_readfirstlane(sum);
}

// Host: the piece length for a launch, from what its workgroups cost.  A trip takes `alone_us` in a workgroup that has its
// CU to itself and `full_us` of a CU's time where `per_cu` workgroups share each, `cut` times that in the kernel that can cut
// (see kCut of the forward); `per_cu` is the number the kernel's registers and LDS are budgeted for.
// (Fitted to every piece length of some thousand launches, 1 to 256 heads and 200 to 8192 rows; of 16714 others 22 ran over 1.03 of the whole
// launch's time, 1.07 at worst, where they would be level.  Since then the uncut kernels gained more than the cutting ones: of 6179 launches of
// 2136 drawn shapes 62 are over 1.03 now, the worst forwards of few heads at head_dim 64 (B1 H6/2 S4629 35.7 us whole, 44.1 cut; both were
// slower before, 46.6 and 48.8).  The lengths chosen run within 0.1 to 2.5 % of the best ones in the geometric mean, dK/dV at head_dim 64 4 %:
// constants that came nearer there made every twentieth launch 3 to 12 % slower than these did.  The four-wave dQ at head_dim 64 is
// never faster cut, which its own loss, 1.18, says: with 1.02 it was cut eight times in 218, B2 H8 S4096 64.1 whole, 71.1.  The four-wave dQ at
// head_dim 128, whose workgroups came to share a CU later, has costs of its own: over 589 launches and every length within 1.6 % of the best, 6
// over 1.03 of the whole launch; of 180 other sets of its three costs the twelve that come within 1.45 % have 8 to 21 there, 1.17 at worst.)
struct TripCost {
  double alone_us, full_us, cut;
  int per_cu;
  double piece_bytes;
  double launch_us = 5.0;   // by how much a cut has to win by the estimate (see choose_pieces)
};
// When the last of a launch's workgroups ends: they are dealt in grid order, tile by tile, to whichever place is free first.
struct Places {
  static constexpr int kMost = 64;   // groups of places that become free together (beyond that the latest two are merged)
  double at[kMost];
  int64_t count[kMost];
  int n;
  explicit Places(int64_t places) : n(1) { at[0] = 0.0; count[0] = places; }
  void run(int64_t workgroups, double us) {
    while (workgroups > 0) {
      const double start = at[0];
      const int64_t k = std::min(count[0], workgroups);
      workgroups -= k;
      count[0] -= k;
      if (count[0] == 0) {
        --n;
        for (int i = 0; i < n; ++i) { at[i] = at[i + 1]; count[i] = count[i + 1]; }
      }
      const double end = start + us;
      int i = n;
      while (i > 0 && at[i - 1] > end + 1e-6) --i;
      if (i > 0 && at[i - 1] > end - 1e-6) { count[i - 1] += k; continue; }
      if (n == kMost) { count[n - 1] += k; at[n - 1] = std::max(at[n - 1], end); continue; }
      for (int j = n; j > i; --j) { at[j] = at[j - 1]; count[j] = count[j - 1]; }
      at[i] = end;
      count[i] = k;
      ++n;
    }
  }
  double last() const { return at[n - 1]; }
};
template <typename F>
double launch_us(int64_t heads, int n_tiles, const TripCost& c, int len, bool pairs, const F& trips_of) {
  constexpr int64_t kCus = 256;
  constexpr double kFixedUs = 4.0, kPairFixedUs = 5.2, kJoinUs = 3.0, kJoinPartUs = 1.0, kBytesPerUs = 4e6;
  int64_t workgroups = 0, cut = 0;
  int most = 1;
  for (int i = 0; i < n_tiles; ++i) {
    const int k = pieces_of(trips_of(i), len);
    workgroups += heads * k;
    if (k > 1) { cut += heads * k; most = std::max(most, k); }
  }
  if (pairs) workgroups = heads * ((n_tiles + 1) / 2);
  const double shared = c.per_cu > 1 ? std::min(1.0, std::max(0.0, (workgroups - kCus) / static_cast<double>(kCus)))
                                     : std::min(1.0, workgroups / static_cast<double>(kCus));
  const double trip = (c.alone_us + (std::max(c.alone_us, c.full_us * c.per_cu) - c.alone_us) * shared) * (len > 0 ? c.cut : 1.0);
  Places places(kCus * c.per_cu);
  if (pairs) {
    for (int i = 0; i < (n_tiles + 1) / 2; ++i) {
      const int j = n_tiles - 1 - i;
      places.run(heads, (trips_of(i) + (j != i ? trips_of(j) : 0)) * trip + kPairFixedUs);
    }
  } else {
    for (int i = 0; i < n_tiles; ++i) {
      const int t = trips_of(i), k = pieces_of(t, len);
      places.run(heads * k, t * trip / k + kFixedUs);
    }
  }
  return places.last() + (cut ? kJoinUs + kJoinPartUs * most + 2.0 * cut * c.piece_bytes / kBytesPerUs : 0.0);
}
template <typename F>
int choose_pieces(int64_t heads, int n_tiles, const TripCost& c, bool pairs, const F& trips_of) {
  if (heads * n_tiles > 4 * 512) return 0;   // enough workgroups that their lengths even out
  // a cut has to win 5 % by the estimate (so that few of the launches above lose) and the time in which a
  // host launches the second kernel: where the host is the slower side a shorter kernel gains nothing (B2 H9/3 S256 D64, forward and backward: 33 us
  // of kernels cut to 29 took 38 us for 35)
  const double uncut_us = launch_us(heads, n_tiles, c, 0, pairs, trips_of);
  double best_us = std::min(0.95 * uncut_us, uncut_us - c.launch_us);
  int best = 0, longest = 0;
  for (int i = 0; i < n_tiles; ++i) longest = std::max(longest, trips_of(i));
  for (int len : {2, 3, 4, 6, 8, 12, 16, 24, 32, 48, 64, 96, 128, 192, 256}) {
    if (len >= longest) break;
    int64_t n = 0;
    for (int i = 0; i < n_tiles; ++i) n += pieces_of(trips_of(i), len);
    if (n > 65535 || heads * n * c.piece_bytes > static_cast<double>(PICO_ATTN_MAX_WORKSPACE)) continue;
    const double us = launch_us(heads, n_tiles, c, len, false, trips_of);
    if (us < best_us) {
      best_us = us;
      best = len;
    }
  }
  return best;
}
template <typename F>
int count_pieces(int n_tiles, int len, const F& trips_of) {
  if (len <= 0) return n_tiles;
  int n = 0;
  for (int i = 0; i < n_tiles; ++i) n += pieces_of(trips_of(i), len);
  return n;
}

// A launch's plan depends on its sizes alone and is worked out once per thread and shape (some microseconds): `make` for the
// sizes in `key`, kept in a small direct-mapped table.
template <typename Plan>
struct PlanTable {
  struct Entry {
    int key[10];
    bool used = false;
    Plan plan;
  } entries[64];
  template <typename Make>
  const Plan& get(const AttnParams& a, int D, const Make& make) {
    const int key[10] = {a.B, a.Hq, a.Hkv, a.Sq, a.Sk, D, a.causal, a.q_offset, a.kv.count, a.kv.len};
    uint32_t h = 2166136261u;
    for (int v : key) h = (h ^ static_cast<uint32_t>(v)) * 16777619u;
    Entry& e = entries[(h ^ (h >> 15)) % 64];
    if (!e.used || !std::equal(key, key + 10, e.key)) {
      e.plan = make();
      std::copy(key, key + 10, e.key);
      e.used = true;
    }
    return e.plan;
  }
};

// accumulators in register order, 16 bytes per lane and piece of a row block: what a cut tile's pieces leave in memory
template <int N>
__device__ __forceinline__ void put_acc(float* dst, const f32x16 (&acc)[N], int lane) {
#pragma unroll
  for (int db = 0; db < N; ++db)
#pragma unroll
    for (int j = 0; j < 4; ++j)
      *reinterpret_cast<f32x4*>(dst + ((db * 4 + j) * kWave + lane) * 4) =
          f32x4{acc[db][4 * j], acc[db][4 * j + 1], acc[db][4 * j + 2], acc[db][4 * j + 3]};
}
template <int N>
__device__ __forceinline__ void get_acc(const float* src, f32x4 (&raw)[N][4], int lane) {
#pragma unroll
  for (int db = 0; db < N; ++db)
#pragma unroll
    for (int j = 0; j < 4; ++j) raw[db][j] = *reinterpret_cast<const f32x4*>(src + ((db * 4 + j) * kWave + lane) * 4);
}

template <int N, int M>   // of 16 x 16 products
__device__ __forceinline__ void put_acc(float* dst, const f32x4 (&acc)[N][M], int lane) {
#pragma unroll
  for (int db = 0; db < N; ++db)
#pragma unroll
    for (int b = 0; b < M; ++b) *reinterpret_cast<f32x4*>(dst + ((db * M + b) * kWave + lane) * 4) = acc[db][b];
}
template <int N, int M>
__device__ __forceinline__ void get_acc(const float* src, f32x4 (&raw)[N][M], int lane) {
#pragma unroll
  for (int db = 0; db < N; ++db)
#pragma unroll
    for (int b = 0; b < M; ++b) raw[db][b] = *reinterpret_cast<const f32x4*>(src + ((db * M + b) * kWave + lane) * 4);
}
// what put_acc left, added
template <int N>
__device__ __forceinline__ void add_acc(f32x16 (&acc)[N], const float* src, int lane) {
  f32x4 raw[N][4];
  get_acc<N>(src, raw, lane);
#pragma unroll
  for (int db = 0; db < N; ++db)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[db][i] += raw[db][i / 4][i % 4];
}
template <int N, int M>
__device__ __forceinline__ void add_acc(f32x4 (&acc)[N][M], const float* src, int lane) {
  f32x4 raw[N][M];
  get_acc(src, raw, lane);
#pragma unroll
  for (int db = 0; db < N; ++db)
#pragma unroll
    for (int b = 0; b < M; ++b) acc[db][b] += raw[db][b];
}

// How many key tiles of KT keys lie in front of position `end`, counted chunk by chunk.
__host__ __device__ inline int tiles_before(const KvChunks& kv, int end, int KT) {
  if (kv.count == 1) return (end + KT - 1) / KT;
  const int whole = end / kv.len, rest = end - whole * kv.len;
  return whole * ((kv.len + KT - 1) / KT) + (rest + KT - 1) / KT;
}

// Key tiles of KT keys that query tile `qtile` of BM queries sees: the trips of a forward or dQ workgroup.
__host__ __device__ inline int query_tile_trips(const AttnParams& a, int qtile, int BM, int KT) {
  int end = a.Sk;
  if (a.causal) {
    const int hi = (qtile + 1) * BM < a.Sq ? (qtile + 1) * BM : a.Sq, vis = a.q_offset + hi;
    end = vis < a.Sk ? vis : a.Sk;
  }
  return tiles_before(a.kv, end, KT);
}

// do chunks end inside key tiles of KT rows that further chunks follow?
inline bool ends_inside_tile(const KvChunks& kv, int KT) { return kv.count > 1 && kv.len % KT != 0; }

// A cursor over the key tiles of KT keys, in order, across the chunks: wave-uniform, so it lives in scalar registers;
// stepping inside a chunk is four adds, a new chunk re-reads its base addresses from the kernel arguments.
template <int D>
struct KvCursor {
  const char *k, *v;            // first row of the next tile
  uint32_t k_left, v_left;      // bytes from there to the end of the chunk's rows of this head
  uint32_t k_step, v_step;
  int tiles_left, chunk, tiles_per_chunk;
  int64_t k_head, v_head;       // element offset of the (batch, kv head) inside every chunk
  // opens at the tile `tile` of the launch
  __device__ __forceinline__ void open(const AttnParams& a, int tile, int b, int hkv, int KT) {
    k_head = b * a.ks[0] + hkv * a.ks[1];
    v_head = b * a.vs[0] + hkv * a.vs[1];
    k_step = static_cast<uint32_t>(KT * a.ks[2] * 2);
    v_step = static_cast<uint32_t>(KT * a.vs[2] * 2);
    tiles_per_chunk = (a.kv.len + KT - 1) / KT;
    chunk = 0;
    if (tile > 0 && a.kv.count > 1) chunk = tile / tiles_per_chunk;
    enter(a);
    if (tile > 0) {
      const int skip = tile - chunk * tiles_per_chunk;
      k += static_cast<int64_t>(skip) * k_step;  k_left -= static_cast<uint32_t>(skip) * k_step;
      v += static_cast<int64_t>(skip) * v_step;  v_left -= static_cast<uint32_t>(skip) * v_step;
      tiles_left -= skip;
    }
  }
  __device__ __forceinline__ void enter(const AttnParams& a) {
    k = reinterpret_cast<const char*>(a.kv.k[chunk] + k_head);
    v = reinterpret_cast<const char*>(a.kv.v[chunk] + v_head);
    k_left = span_bytes(a.kv.len, a.ks[2], D);
    v_left = span_bytes(a.kv.len, a.vs[2], D);
    tiles_left = tiles_per_chunk;
  }
  __device__ __forceinline__ void next(const AttnParams& a) {
    if (--tiles_left == 0 && chunk + 1 < a.kv.count) {
      ++chunk;
      enter(a);
    } else {
      k += k_step;  k_left -= k_step;
      v += v_step;  v_left -= v_step;
    }
  }
};
// The positions of the tile being computed: its first key, and the end of its chunk (keys from there on do not exist).
struct KvPosition {
  int key0, end;
  __device__ __forceinline__ void open(const KvChunks& kv, int tile, int KT) {
    const int per = (kv.len + KT - 1) / KT, chunk = tile > 0 && kv.count > 1 ? tile / per : 0;
    key0 = chunk * kv.len + (tile - chunk * per) * KT;
    end = (chunk + 1) * kv.len;
  }
  __device__ __forceinline__ void next(const KvChunks& kv, int KT) {
    key0 += KT;
    if (key0 >= end) {   // (also where the tile ended exactly with its chunk)
      key0 = end;
      end += kv.len;
    }
  }
};

// The arguments of a launch of one chunk (see Arguments).  Forward, dQ, dK/dV alone, us: B4 H32 256 x 1024 D64 15.3 -> 14.8, 18.0 -> 17.7, 25.3 -> 23.6;
// B2 H9/3 S256 D64 5.9 -> 5.7, 6.5 -> 6.3, 11.5 -> 11.1; B4 H32 S1024 D64 27.4 -> 26.3, 36.8 -> 36.4, 42.7 -> 42.6.  (All 18 lines of the backward's
// arguments, or loads that the compiler may move behind others, gain less, and the forward lost up to 4 %.)
using AttnArguments = Arguments<0, offsetof(AttnParams, kv.v), offsetof(AttnParams, kv.count), offsetof(AttnParams, kv.count) + 64, sizeof(AttnParams) + 4>;

int check_attn_desc(const char* fn, const pico_attn_desc* d);
// tables usable for head_dim D and positions 0 .. last_pos?
int check_rope_tables(const char* fn, const pico_rope_tables* t, int D, int64_t last_pos);
// one chunk of d->Sk keys
AttnParams make_params(const pico_attn_desc* d, const void* q, const void* k, const void* v);
// the chunk list checked against the descriptor (count, length, tile multiple, alignment; with need_kv also that no
// k / v pointer is NULL) and copied into `a`
int set_chunks(const char* fn, const pico_attn_desc* d, const pico_kv_chunks* kv, AttnParams& a, bool need_kv);

}  // namespace pico
