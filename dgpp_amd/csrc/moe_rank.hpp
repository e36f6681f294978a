// The rank of a decode slot among (expert key, slot) pairs and the wavefront's prefix sum, shared by the router, the
// grouping and the tiled product kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <limits.h>
#include <stdint.h>

namespace dgpp_amd {

// Ranks by (key, slot) as one integer: key << 10 | slot (slots < 1024, keys <= n_experts < 2^16), unique per slot.
__device__ __forceinline__ int32_t slot_sort_key(int key, int slot) { return (key << 10) | slot; }
// Rank of a slot among `padded` such integers (a multiple of 4; pad entries hold INT_MAX): how many are below
// `mine`. Four per LDS read, one compare and one add each: the ranking is bound by the vector ALU.
__device__ __forceinline__ int slot_rank(const int32_t* __restrict__ sort_keys, int padded, int32_t mine) {
  const int4* k4 = reinterpret_cast<const int4*>(sort_keys);
  int pos = 0;
#pragma unroll 4
  for (int o = 0; o < padded / 4; ++o) {
    const int4 v = k4[o];
    pos += (v.x < mine) + (v.y < mine) + (v.z < mine) + (v.w < mine);
  }
  return pos;
}

template <int kCtrl, int kRowMask>
__device__ __forceinline__ int dpp_take(int v) {   // lanes the move does not reach read 0
  return __builtin_amdgcn_update_dpp(0, v, kCtrl, kRowMask, 0xF, false);
}
// Inclusive prefix sum over the wavefront: four shifts inside each row of sixteen lanes, then the two row
// broadcasts that carry a row's total into the rows after it.
__device__ __forceinline__ int wave_prefix_incl(int v) {
  v += dpp_take<0x111, 0xF>(v);   // row_shr:1
  v += dpp_take<0x112, 0xF>(v);   // row_shr:2
  v += dpp_take<0x114, 0xF>(v);   // row_shr:4
  v += dpp_take<0x118, 0xF>(v);   // row_shr:8
  v += dpp_take<0x142, 0xA>(v);   // row_bcast:15 into rows 1 and 3
  v += dpp_take<0x143, 0xC>(v);   // row_bcast:31 into rows 2 and 3
  return v;
}

}  // namespace dgpp_amd
