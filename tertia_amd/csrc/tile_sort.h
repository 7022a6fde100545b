// tile_sort.h — bitonic sort of 256 int keys held one per thread of a
// 256-thread work-group.  Every compare-exchange distance is a compile-time
// constant: distances 1, 2, 4 and 8 exchange through DPP lane moves, 16 and 32
// through permlane swaps (no LDS round trip), and the two cross-wave distances
// (64, 128) through LDS (sh, 256 ints).  Used by the
// tiled push kernels to order deposit (and adjoint scatter) events by cell.
#pragma once

#include <hip/hip_runtime.h>

namespace qss_tile {

// value held by lane (lane ^ J) of this wave64
template <int J>
__device__ inline int xor_lane(int v, int t) {
  if constexpr (J == 1) {
    return __builtin_amdgcn_mov_dpp(v, 0xB1, 0xF, 0xF, false);   // quad_perm [1,0,3,2]
  } else if constexpr (J == 2) {
    return __builtin_amdgcn_mov_dpp(v, 0x4E, 0xF, 0xF, false);   // quad_perm [2,3,0,1]
  } else if constexpr (J == 4) {
    // row_ror:n makes lane i read lane (i - n) mod 16 of its row
    const int from_minus4 = __builtin_amdgcn_mov_dpp(v, 0x124, 0xF, 0xF, false);
    const int from_plus4 = __builtin_amdgcn_mov_dpp(v, 0x12C, 0xF, 0xF, false);
    return (t & 4) ? from_minus4 : from_plus4;
  } else {
    static_assert(J == 8, "distances within a row of 16");
    return __builtin_amdgcn_mov_dpp(v, 0x128, 0xF, 0xF, false);  // row_ror:8
  }
}

template <int K, int J>
__device__ inline int bitonic_stage(int key, int *sh, int t) {
  const bool up = (t & K) == 0;
  const bool lower = (t & J) == 0;
  if constexpr (J == 16 || J == 32) {
    // swapping a register with its own copy leaves the lane's key in one and its
    // partner's in the other, in either order
    const auto r = J == 32 ? __builtin_amdgcn_permlane32_swap(key, key, false, false)
                           : __builtin_amdgcn_permlane16_swap(key, key, false, false);
    const int a = (int)r[0], b = (int)r[1];
    return (lower == up) ? min(a, b) : max(a, b);
  } else {
    int other;
    if constexpr (J >= 64) {
      sh[t] = key;
      __syncthreads();
      other = sh[t ^ J];
      __syncthreads();
    } else {
      other = xor_lane<J>(key, t);
    }
    // lower element keeps min if ascending block, max otherwise
    const int mn = min(key, other), mx = max(key, other);
    return (lower == up) ? mn : mx;
  }
}

template <int K, int J>
__device__ inline int bitonic_merge(int key, int *sh, int t) {
  key = bitonic_stage<K, J>(key, sh, t);
  if constexpr (J > 1) key = bitonic_merge<K, J / 2>(key, sh, t);
  return key;
}

template <int K>
__device__ inline int bitonic_sort(int key, int *sh, int t) {
  if constexpr (K > 2) key = bitonic_sort<K / 2>(key, sh, t);
  return bitonic_merge<K, K / 2>(key, sh, t);
}

// The thread index passes through a register the compiler cannot see into: it would
// otherwise keep every stage's lane masks (36 pairs of scalar registers) alive over
// the caller's whole loop and spill what the loop needs.
__device__ inline int sort256(int key, int *sh) {
  int t = threadIdx.x;
  asm volatile("" : "+v"(t));
  return bitonic_sort<256>(key, sh, t);
}

}  // namespace qss_tile
