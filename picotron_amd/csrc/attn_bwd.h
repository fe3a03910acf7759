// What the attention backward's kernels share.
#pragma once
#include "attn_common.h"

namespace pico {

struct BwdParams {
  AttnParams a;
  const __bf16* dout;
  const float* lse;
  const float* delta;
  const __bf16* out;   // fused-delta mode of the dQ kernel: the forward output, addressed like dout
  float* delta_w;      //   ... and where that kernel writes delta = sum_d dO * O for the dK/dV kernel
  void* dq;
  void* dk[kMaxChunks];      // per K / V chunk; nullptr: that chunk's gradient is not wanted
  void* dv[kMaxChunks];
  __bf16* dk_final[kMaxChunks];   // per chunk, optional: the chunk's total (fp32 dk[c] if its accumulate bit is set, plus this
  __bf16* dv_final[kMaxChunks];   //   launch's block) leaves here in bf16; dk[c] / dv[c] are only read
  int64_t dkfs[3];                // element strides (b, h, s) of dk_final / dv_final
  uint32_t dkv_accumulate;   // bit c: chunk c's dk / dv are added to (fp32)
  int dq_f32, dq_accumulate;
  int dkv_f32;
  int pair_ktiles;                  // > 0: every workgroup does key tile blockIdx.y and this number - 1 - blockIdx.y
  int64_t dqs[3];  // element strides (b, h, s) of dq
  int64_t dks[3];  // element strides (b, h, s) of dk and dv
  RopeArgs rope;   // rope.cos != nullptr: q and k are rotated tensors; dq and dk leave un-rotated (RoPE's backward)
};

// bf16 gradients leave with streaming (non-temporal) stores: nothing on this GPU reads them back soon
constexpr bool kStreamGrads = true;

// key tile `ktile` (counted chunk by chunk): its chunk, its first row there and that row's position in the launch
struct KeyTile {
  int chunk, row0, key0;
};
__host__ __device__ inline KeyTile key_tile(const KvChunks& kv, int ktile, int BN) {
  if (kv.count == 1) return {0, ktile * BN, ktile * BN};
  const int per = (kv.len + BN - 1) / BN, chunk = ktile / per, row0 = (ktile - chunk * per) * BN;
  return {chunk, row0, chunk * kv.len + row0};
}
// first query tile of BM queries that sees position key0
__host__ __device__ inline int first_query_tile(const AttnParams& a, int key0, int BM) {
  const int first_q = a.causal ? key0 - a.q_offset : 0;
  return first_q > 0 ? first_q / BM : 0;
}
// trips of a key tile: (query heads of the group) x (query tiles that see it)
__host__ __device__ inline int dkdv_trips(const AttnParams& a, int ktile, int BN, int BM) {
  const int n = (a.Sq + BM - 1) / BM, start = first_query_tile(a, key_tile(a.kv, ktile, BN).key0, BM);
  return n > start ? (n - start) * (a.Hq / a.Hkv) : 0;
}

// dK/dV at head_dim 128 in key tiles of 256 (attn_bwd_roles.hip)
struct RoleTiles {
  static constexpr int BN = 256, BM = 64, kPerCu = 1;   // keys of a tile, queries of a trip, workgroups that share a CU
};
int launch_dkdv_roles(const BwdParams& p, hipStream_t s);

}  // namespace pico
