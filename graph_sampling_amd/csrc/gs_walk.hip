// Uniform random walks and metapath walks on gfx950, one lane per walker.
//
// Replaces impl::fusion::FusedRandomWalkCUDA (reference
// src/cuda/fusion/random_walk.cu:52) and FusedMetapathRandomWalkCUDA
// (src/cuda/fusion/metapath_random_walk.cu:49).
//
// The trace is step-major, [length+1][n] (random_walk.cu:21,32,42), which is
// also the coalesced layout for one lane per walker: at every step the 64 lanes
// of a wave store 64 consecutive ids.  The walker keeps its current node in a
// register (the reference re-reads it from the trace, random_walk.cu:32).  A
// step is two dependent random reads (the indptr pair, then one neighbour).  With
// enough walkers the kernel is bound by lines fetched behind the L2s: random reads
// that miss run at 48-55 G/s on this machine, in the memory-side cache or not (hits
// at 255 G/s), and a million walkers on a graph of 4 M nodes and 200 M edges miss
// 66 M times in 47 M steps.  With few it is latency: 256 threads per workgroup, no
// LDS, ~24 VGPRs, as many waves as there are.  One Philox block feeds four steps.
#include "gs_common.hpp"

namespace gs {
namespace {

constexpr int kThreads = 256;

// Neighbour arrays from this size on are read as streams (the line is the first to leave the
// L2): hardly one of their lines is met again, and the offsets, which are, stay longer.
// Arrays that the L2s and the memory-side cache hold in good part lose by it.  38 steps, three graphs
// in turn, plain / as a stream, us, by walkers:
//                               66 k       131 k       400 k       1 M
//   280 MB (70 M edges, 32-bit)   66/65      86/97     266/281    632/662
//   400 MB (100 M, 32-bit)        69/67      93/104    289/307    687/724
//   720 MB (90 M, 64-bit)         73/66      95/98     301/291    710/704
//   800 MB (200 M, 32-bit)        70/67      98/102    307/301    727/708
//   1.1 GB (139 M, 64-bit)        72/66      96/96     296/286    693/688
constexpr int64_t kStreamBytes = int64_t(5) << 27;
// The same for a relation of a metapath, when the path has two such: three of 400 MB, 20 steps, 200 k
// walkers 89 -> 85 us, 1 M walkers 411 -> 383.
constexpr int64_t kStreamRelationBytes = int64_t(256) << 20;
// A metapath's relations have to be looked up for it in front of the first step, 1.0 to 1.4 us that
// only long work earns back: 1 M walkers, 4 steps 93 -> 92 us, 200 k walkers, 20 steps 87 -> 85,
// but 400 k walkers, 8 steps 70 -> 71, 18 k walkers, 8 steps 12.9 -> 13.8.
constexpr int64_t kStreamSteps = int64_t(1) << 22;

// A node outside [0, num_nodes) has no neighbours (the walker dies there), so a
// stray seed can never turn into a wild read.
template <typename IdT>
__device__ __forceinline__ int64_t step_from(const int64_t* __restrict__ indptr,
                                             const IdT* __restrict__ indices, int64_t num_nodes,
                                             int64_t curr, uint32_t x, bool stream) {
  if (static_cast<uint64_t>(curr) >= static_cast<uint64_t>(num_nodes)) return -1;
  const int64_t start = indptr[curr];
  const int64_t deg = indptr[curr + 1] - start;
  if (deg <= 0) return -1;
  const IdT* at = indices + start + static_cast<int64_t>(x % static_cast<uint32_t>(deg));
  IdT next;
  if (stream) {
    // (held apart from the other by two empty statements, or the compiler makes one plain load
    // of the two)
    asm volatile("" : "+v"(at));
    next = __builtin_nontemporal_load(at);
    asm volatile("" : "+v"(next));
  } else {
    next = *at;
  }
  return static_cast<int64_t>(next);
}

template <typename IdT>
__global__ void __launch_bounds__(kThreads)
random_walk_kernel(const int64_t* __restrict__ indptr, const IdT* __restrict__ indices,
                   int64_t num_nodes, const IdT* __restrict__ seeds, int64_t n, int64_t length, uint64_t seed,
                   const uint32_t* __restrict__ replay, IdT* __restrict__ trace) {
  const int64_t w = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
  if (w >= n) return;
  int64_t curr = static_cast<int64_t>(seeds[w]);
  trace[w] = static_cast<IdT>(curr);
  const bool stream = indptr[num_nodes] >= kStreamBytes / static_cast<int64_t>(sizeof(IdT));
  U4 x;
  for (int64_t t = 0; t < length; ++t) {
    if (!replay && (t & 3) == 0)
      x = draw_block(seed, kTagWalk, static_cast<uint64_t>(w), static_cast<uint64_t>(t >> 2));
    int64_t pick = -1;
    if (curr >= 0) {
      const uint32_t xv = replay ? replay[t * n + w] : x.v[t & 3];
      pick = step_from(indptr, indices, num_nodes, curr, xv, stream);
    }
    trace[(t + 1) * n + w] = static_cast<IdT>(pick);
    curr = pick;
  }
}

// LONG_WORK: large neighbour arrays are looked for and read as streams
template <typename IdT, bool LONG_WORK>
__global__ void __launch_bounds__(kThreads)
metapath_walk_kernel(const int64_t* const* __restrict__ all_indptr,
                     const IdT* const* __restrict__ all_indices,
                     const int64_t* __restrict__ all_num_nodes,
                     const int64_t* __restrict__ metapath, int64_t length,
                     const IdT* __restrict__ seeds, int64_t n, uint64_t seed,
                     const uint32_t* __restrict__ replay, IdT* __restrict__ trace) {
  const int64_t w = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
  if (w >= n) return;
  int64_t curr = static_cast<int64_t>(seeds[w]);
  trace[w] = static_cast<IdT>(curr);
  U4 x;
  unsigned long long streams = 0ull;  // bit t: the relation of step t (mod 64) is read as a stream
  for (int64_t t = 0; t < length; ++t) {
    if (LONG_WORK && (t & (kWave - 1)) == 0) {  // a lane per step of the next 64
      const int64_t step = t + (threadIdx.x & (kWave - 1));
      const int64_t rel = metapath[step < length ? step : length - 1];
      const int64_t bytes = all_indptr[rel][all_num_nodes[rel]] * static_cast<int64_t>(sizeof(IdT));
      const unsigned long long large = __ballot(bytes >= kStreamRelationBytes);
      const int64_t one = __shfl(rel, large ? __ffsll(static_cast<long long>(large)) - 1 : 0, kWave);
      const bool two = __ballot(bytes >= kStreamRelationBytes && rel != one) != 0ull;
      streams = two ? large : __ballot(bytes >= kStreamBytes);
    }
    if (!replay && (t & 3) == 0)
      x = draw_block(seed, kTagWalk, static_cast<uint64_t>(w), static_cast<uint64_t>(t >> 2));
    int64_t pick = -1;
    if (curr >= 0) {
      const int64_t rel = metapath[t];  // uniform over the wave: scalar loads
      const uint32_t xv = replay ? replay[t * n + w] : x.v[t & 3];
      pick = step_from(all_indptr[rel], all_indices[rel], all_num_nodes[rel], curr, xv,
                       LONG_WORK && ((streams >> (t & (kWave - 1))) & 1ull));
    }
    trace[(t + 1) * n + w] = static_cast<IdT>(pick);
    curr = pick;
  }
}

}  // namespace
}  // namespace gs

using namespace gs;

extern "C" {

int gs_random_walk(const int64_t* indptr, int64_t num_nodes, const void* indices, int id_bytes,
                   const void* seeds, int64_t n, int64_t length, uint64_t seed, const uint32_t* replay,
                   void* trace, void* stream) {
  GS_REQUIRE(n >= 0 && length >= 0 && num_nodes >= 0, "gs_random_walk: negative size");
  GS_REQUIRE(n == 0 || (indptr && seeds && trace), "gs_random_walk: null pointer");
  GS_REQUIRE(valid_id_bytes(id_bytes), "gs_random_walk: id_bytes must be 4 or 8, got %d", id_bytes);
  if (n == 0) return GS_OK;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const dim3 grid(blocks_for(n, kThreads));
  ProfileScope prof("random_walk", st);
  if (id_bytes == 8)
    hipLaunchKernelGGL((random_walk_kernel<int64_t>), grid, dim3(kThreads), 0, st, indptr,
                       static_cast<const int64_t*>(indices), num_nodes,
                       static_cast<const int64_t*>(seeds), n, length, seed, replay,
                       static_cast<int64_t*>(trace));
  else
    hipLaunchKernelGGL((random_walk_kernel<int32_t>), grid, dim3(kThreads), 0, st, indptr,
                       static_cast<const int32_t*>(indices), num_nodes,
                       static_cast<const int32_t*>(seeds), n, length, seed, replay,
                       static_cast<int32_t*>(trace));
  return check_launch("random_walk");
}

int gs_metapath_walk(const int64_t* const* all_indptr, const void* const* all_indices,
                     const int64_t* all_num_nodes, int id_bytes, const int64_t* metapath, int64_t length, const void* seeds,
                     int64_t n, uint64_t seed, const uint32_t* replay, void* trace,
                     void* stream) {
  GS_REQUIRE(n >= 0 && length >= 0, "gs_metapath_walk: negative size");
  GS_REQUIRE(n == 0 || (seeds && trace), "gs_metapath_walk: null pointer");
  GS_REQUIRE(n == 0 || length == 0 || (all_indptr && all_indices && all_num_nodes && metapath),
             "gs_metapath_walk: null relation tables");
  GS_REQUIRE(valid_id_bytes(id_bytes), "gs_metapath_walk: id_bytes must be 4 or 8, got %d", id_bytes);
  if (n == 0) return GS_OK;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const dim3 grid(blocks_for(n, kThreads));
  const bool long_work = length > 0 && n >= (kStreamSteps + length - 1) / length;
  ProfileScope prof("metapath_walk", st);
  auto go = [&](auto kernel, auto id) {
    using IdT = decltype(id);
    hipLaunchKernelGGL(kernel, grid, dim3(kThreads), 0, st, all_indptr,
                       reinterpret_cast<const IdT* const*>(all_indices), all_num_nodes, metapath, length,
                       static_cast<const IdT*>(seeds), n, seed, replay, static_cast<IdT*>(trace));
  };
  if (id_bytes == 8)
    go(long_work ? metapath_walk_kernel<int64_t, true> : metapath_walk_kernel<int64_t, false>, int64_t());
  else
    go(long_work ? metapath_walk_kernel<int32_t, true> : metapath_walk_kernel<int32_t, false>, int32_t());
  return check_launch("metapath_walk");
}

}  // extern "C"
