// What the products whose operands go to LDS without passing the registers share: an operand's tile in LDS and the window of the
// matrix that it is requested from.
#pragma once
#include "attn_common.h"

namespace pico {
namespace {

constexpr int kStep = 64;   // contraction per step

// One operand's tile of kRows rows and kStep of contraction.  kSlow false: rows of the tile are rows of the matrix (contraction
// contiguous), 128 bytes in LDS, whose 16-byte pieces change places with the row; true: the matrix lies with its contraction as
// the slow axis and is staged that way, and the 32-byte pieces change places.
template <bool kSlow, int kRows, int kThreads>
struct Tile {
  static constexpr int kPitch = kSlow ? kRows * 2 : kStep * 2, kBytes = kRows * kStep * 2;
  static constexpr int kPieces = kBytes / 16 / kThreads;
  static_assert(kBytes % (16 * kThreads) == 0 && kRows % 32 == 0);
  // kSlow: a transposing read takes 32 bytes of 16 rows, 0 .. 3 and every 8 further; where rows of this pitch start in the banks
  // decides which of them have to differ
  static __device__ __forceinline__ int twist(int k) {
    return kRows % 128 == 0 ? (k & 3) | (k >> 3 & 1) << 2 : kRows % 64 == 0 ? (k >> 1 & 1) | (k >> 3 & 1) << 1 : k >> 3 & 1;
  }
  // byte offset in the matrix of what lies at 16 (tid + kThreads i) in LDS
  static __device__ __forceinline__ uint32_t offset(int64_t ld, int tid, int i) {
    const int idx = tid + kThreads * i;
    if constexpr (kSlow) {
      const int k = idx / (kRows / 8), c = idx % (kRows / 8);
      return static_cast<uint32_t>((k * ld + (c / 2 ^ twist(k)) * 16 + c % 2 * 8) * 2);
    } else {
      const int r = idx / 8, c = idx % 8 ^ (r / 2 & 7);
      return static_cast<uint32_t>((r * ld + c * 8) * 2);
    }
  }
  // lane l gets row `first` + l % 16, contraction 32 s + 8 (l / 16) ..+7
  static __device__ __forceinline__ bf16x8 fragment(const unsigned char* tile, int first, int s, int lane) {
    const int n = lane % 16, h = lane / 16;
    if constexpr (kSlow) {
      const int k = 8 * h + n / 4;
      return lds_read_tr_pair_step(reinterpret_cast<const __bf16*>(tile + (32 * s + k) * kPitch + (first / 16 ^ twist(k)) * 32 + n % 4 * 8),
                                   2 * kPitch);
    } else {
      return *reinterpret_cast<const bf16x8*>(tile + (first + n) * kPitch + ((4 * s + h) ^ (n / 2 & 7)) * 16);
    }
  }
};

// the bytes of a tile that are left from the step on that is requested next
struct Window {
  uint64_t base;
  uint32_t bytes;
};
template <bool kSlow>
__device__ __forceinline__ Window open_window(const __bf16* p, int64_t ld, int first, int side, int rows, int k, int K) {
  const int left = min(side, rows - first);
  return {reinterpret_cast<uint64_t>(p) + (kSlow ? first + k * ld : first * ld + k) * 2,
          static_cast<uint32_t>((kSlow ? (K - k - 1) * ld + left : (left - 1) * ld + K - k) * 2)};
}
__device__ __forceinline__ void advance(Window& w, uint32_t bytes) {
  w.base += bytes;
  w.bytes = w.bytes > bytes ? w.bytes - bytes : 0;
}
__device__ __forceinline__ u32x4 resource(const Window& w) { return request_window(w.base, w.bytes); }

}  // namespace
}  // namespace pico
