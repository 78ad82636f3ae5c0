// tile_dma.hpp -- device helpers of the kernels whose operands are staged in
// LDS by direct loads (global_load_lds).
#pragma once

#include <hip/hip_runtime.h>

#include "tile_shapes.hpp"

namespace occxc {
namespace {

// Tiles that the contractions run for a wavefront's half block (half_tiles); one
// tile runs as the 2-tile shape (their shapes start at 2, and the second tile's
// operands are in LDS whatever the width of the block).
__device__ __forceinline__ int live_tiles(int valid, int half) {
  const int t = half_tiles(valid, half);
  return t == 1 ? 2 : t;
}

// Barrier after this wavefront's vector memory loads but the newest N are
// done (and its LDS accesses): the s_waitcnt immediate holds vmcnt in bits
// 3:0 and 15:14, expcnt (no wait) in 6:4 and lgkmcnt (0) in 11:8.
template <int N>
__device__ __forceinline__ void vmcnt_barrier() {
  static_assert(N >= 0 && N < 64, "vmcnt is six bits");
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt((N & 0xF) | (0x7 << 4) | ((N >> 4) << 14));
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Workgroup barrier for LDS hand-offs only: waits for this wavefront's LDS
// accesses (lgkmcnt) but not for its outstanding global memory operations
// (__syncthreads would wait for them).  The empty asm statements keep the
// compiler from moving memory accesses across it.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xc07f);  // vmcnt and expcnt: no wait; lgkmcnt(0)
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

} // namespace
} // namespace occxc
