// tile_sort.h — bitonic sort of 256 int keys held one per thread of a
// 256-thread work-group.  Every compare-exchange distance is a compile-time
// constant: distances 1, 2, 4 and 8 exchange through DPP lane moves, 16 and 32
// through permlane swaps (no LDS round trip), and the two cross-wave distances
// (64, 128) through LDS (sh, 256 ints).  Used by the
// tiled push kernels to order deposit (and adjoint scatter) events by cell.
#pragma once

#include <hip/hip_runtime.h>

namespace qss_tile {

// threadIdx.x through a register the compiler cannot see into, where the masks and
// addresses it gives should be remade in each round: kept over the chunk loop they
// spill what the loop needs
__device__ inline int thread_index() {
  int t = threadIdx.x;
  asm volatile("" : "+v"(t));
  return t;
}

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
  return bitonic_sort<256>(key, sh, thread_index());
}

// Where the event at sorted position i lies.  Neighbouring lanes walk the runs of
// neighbouring cells, and runs of 16 events put them 16 apart, on two of the banks:
// with the row of 16 mixed into the place they are on different ones.
__device__ inline int run_slot(int i) { return i ^ i >> 4; }

// Events of a cell that one lane sums: the bytes of one 8-byte list (indices of the
// round's 256 events), put in the order of the indices by networks of 4 or 8.
constexpr int kCell = 8;

template <int N>
__device__ inline void sort_network(int *v) {
  const auto cx = [&](int i, int j) {
    const int a = v[i], b = v[j];
    v[i] = min(a, b);
    v[j] = max(a, b);
  };
  if constexpr (N == 4) {
    cx(0, 1); cx(2, 3); cx(0, 2); cx(1, 3); cx(1, 2);
  } else {   // 19 exchanges for 8
    static_assert(N == 8, "networks for 4 and 8");
    cx(0, 2); cx(1, 3); cx(4, 6); cx(5, 7); cx(0, 4); cx(1, 5); cx(2, 6); cx(3, 7);
    cx(0, 1); cx(2, 3); cx(4, 5); cx(6, 7); cx(2, 4); cx(3, 5); cx(1, 4); cx(3, 6);
    cx(1, 2); cx(3, 4); cx(5, 6);
  }
}

// the list's indices in order, sentinels past n
template <int N>
__device__ inline void cell_order(uint2 bytes, int n, int *e) {
#pragma unroll
  for (int i = 0; i < N; ++i)
    e[i] = i < n ? (int)((i < 4 ? bytes.x >> 8 * i : bytes.y >> 8 * (i - 4)) & 255) : 256 + i;
  sort_network<N>(e);
}

}  // namespace qss_tile
