// What kernels of ONE workgroup of 1024 threads share that keep a whole small problem in LDS
// (gs_minibatch.hip, the small relabel of gs_unique.hip).
#pragma once

#include "gs_common.hpp"

namespace gs {

constexpr int kOneThreads = 1024;
constexpr int kOneWaves = kOneThreads / kWave;

// A barrier that orders LDS only: the stores to the outputs, which no thread reads back, go on
// under it (a full barrier waits until memory has acknowledged them).
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <int CTRL, int ROWS>
__device__ __forceinline__ int scan_step(int v) {
  return v + __builtin_amdgcn_update_dpp(0, v, CTRL, ROWS, 0xf, false);
}

// sum over the lanes of a wave up to and including this one, in lane moves of the vector ALU
__device__ __forceinline__ int wave_inclusive_sum(int v) {
  v = scan_step<0x111, 0xf>(v);  // from 1, 2, 4 and 8 lanes below in a row of 16
  v = scan_step<0x112, 0xf>(v);
  v = scan_step<0x114, 0xf>(v);
  v = scan_step<0x118, 0xf>(v);
  v = scan_step<0x142, 0xa>(v);  // row 0's sum to row 1, row 2's to row 3
  return scan_step<0x143, 0xc>(v);  // rows 0 and 1's to rows 2 and 3
}

// Exclusive prefix of v over the workgroup and its total: one barrier, the wave part in lane
// moves of the vector ALU.  `which` alternates from call to call (the two halves of s_scan).
__device__ __forceinline__ int one_scan(int v, int* total, int (*s_scan)[kOneWaves], int which) {
  const int incl = wave_inclusive_sum(v);
  const int wave = threadIdx.x / kWave;
  if ((threadIdx.x & (kWave - 1)) == kWave - 1) s_scan[which][wave] = incl;
  lds_barrier();
  int before = 0, sum = 0;
#pragma unroll
  for (int w = 0; w < kOneWaves; ++w) {
    const int t = s_scan[which][w];
    before += w < wave ? t : 0;
    sum += t;
  }
  *total = sum;
  return before + incl - v;
}

// whether an id fits the 32 bits a table's one-word slots keep of it
template <typename IdT>
__device__ __forceinline__ bool fits_slot(IdT id) {
  return sizeof(IdT) == 4 || (static_cast<unsigned long long>(id) >> 32) == 0ull;
}

}  // namespace gs
