// Which of a column's edges a uniform sample takes, for kernels that give a column to a group of
// lanes (gs_sampling.hip, gs_minibatch.hip).
#pragma once

#include "gs_common.hpp"

namespace gs {

__device__ __forceinline__ bool valid_col(int64_t c, int64_t num_cols) {
  return static_cast<uint64_t>(c) < static_cast<uint64_t>(num_cols);
}

// lanes that share a column: one for every four picks
inline int group_lanes_for(int64_t fanout) {
  return fanout <= 4 ? 1 : (fanout <= 8 ? 2 : (fanout <= 16 ? 4 : 8));
}

// the value lane `owner` of every G-lane group holds (owner is a constant after unrolling)
template <int G>
__device__ __forceinline__ uint32_t group_broadcast(uint32_t v, int owner) {
  if (G == 1) return v;
  const int x = static_cast<int>(v);
  if (G == 2) {  // pairs inside a quad: lanes (0,1) read lane owner, lanes (2,3) lane 2 + owner
    return static_cast<uint32_t>(owner == 0 ? __builtin_amdgcn_update_dpp(0, x, 0xA0, 0xF, 0xF, false)
                                            : __builtin_amdgcn_update_dpp(0, x, 0xF5, 0xF, 0xF, false));
  }
  if (G == 4) {
    switch (owner) {
      case 0: return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, x, 0x00, 0xF, 0xF, false));
      case 1: return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, x, 0x55, 0xF, 0xF, false));
      case 2: return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, x, 0xAA, 0xF, 0xF, false));
      default: return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, x, 0xFF, 0xF, 0xF, false));
    }
  }
  return static_cast<uint32_t>(__shfl(x, ((threadIdx.x & (kWave - 1)) & ~(G - 1)) | owner, kWave));
}

// Floyd's selection of k < deg of a column's edges by the column's G lanes together: mine[u] =
// position of output 4 * sub + u inside the column (all of them, in order, when deg <= k).  Lane s
// makes the Philox block of draws 4s..4s+3 and reduces them to their ranges; the "already chosen?"
// chain runs step by step with one lane move per step.  replay: the column's draws, or nullptr.
template <int G>
__device__ __forceinline__ void floyd_picks(uint64_t seed, int64_t row, int sub, int k, int64_t deg,
                                            const uint32_t* replay, uint32_t (&mine)[4]) {
  constexpr int KMAX = 4 * G;
  if (deg <= k) {
#pragma unroll
    for (int u = 0; u < 4; ++u) mine[u] = static_cast<uint32_t>(4 * sub + u);
    return;
  }
  const uint32_t lowest = static_cast<uint32_t>(deg - k);  // step i draws from [0, lowest + i]
  uint32_t t[4] = {0u, 0u, 0u, 0u};
  if (4 * sub < k) {
    U4 blk;
    if (replay) {
#pragma unroll
      for (int u = 0; u < 4; ++u) blk.v[u] = 4 * sub + u < k ? replay[4 * sub + u] : 0u;
    } else {
      blk = draw_block(seed, kTagUniform, static_cast<uint64_t>(row), static_cast<uint64_t>(sub));
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) t[u] = blk.v[u] % (lowest + static_cast<uint32_t>(4 * sub + u) + 1u);
  }
  uint32_t chosen[KMAX];
#pragma unroll
  for (int i = 0; i < KMAX; ++i) {
    if (i < k) {
      const uint32_t ti = t[i & 3];  // the owner's lane holds the step's draw
      bool taken = false;
#pragma unroll
      for (int m = 0; m < i; ++m) taken |= chosen[m] == ti;
      const uint32_t c = group_broadcast<G>(taken ? lowest + static_cast<uint32_t>(i) : ti, i >> 2);
      chosen[i] = c;
      if (sub == (i >> 2)) mine[i & 3] = c;
    }
  }
}

}  // namespace gs
