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
// 66 M times in 47 M steps.  A third of those are the offsets', which is why long walks pack
// them first.  With few it is latency: 256 threads per workgroup, no
// LDS, ~24 VGPRs, as many waves as there are.  One Philox block feeds four steps.
#include "gs_common.hpp"

namespace gs {
namespace {

constexpr int kThreads = 256;

// Neighbour arrays from this size on are read as streams (the line is the first to leave the
// L2): hardly one of their lines is met again, and the offsets, which are, stay longer.
// Arrays that the L2s and the memory-side cache hold in good part lose by it, and so do all with a
// packed table of the offsets (below), which stays without it: 1 M walkers, 80 steps, 4 M nodes of 50
// edges 1237 us plain, 1455 as a stream.  Without a table, 38 steps, three graphs
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

// The neighbour that draw x takes of `deg` ones from `start` on; -1: there are none.
template <typename IdT>
__device__ __forceinline__ int64_t neighbour(const IdT* __restrict__ indices, int64_t start,
                                             int64_t deg, uint32_t x, bool stream) {
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

// A node outside [0, num_nodes) has no neighbours (the walker dies there), so a
// stray seed can never turn into a wild read.
template <typename IdT>
__device__ __forceinline__ int64_t step_from(const int64_t* __restrict__ indptr,
                                             const IdT* __restrict__ indices, int64_t num_nodes,
                                             int64_t curr, uint32_t x, bool stream) {
  if (static_cast<uint64_t>(curr) >= static_cast<uint64_t>(num_nodes)) return -1;
  const int64_t start = indptr[curr];
  return neighbour(indices, start, indptr[curr + 1] - start, x, stream);
}

// The offsets of kRecordNodes nodes in 16 bytes: the first node's start in 32 bits, then every node's
// end as its distance from that start, in 16 bits each and in order.  Where that cannot be said (a
// hub among the nodes), the first distance is larger than the last and the offsets themselves are
// read instead.  A step reads a record at once, and what the L2s (4 MB a die) have to hold of the offsets
// is a third: 1 M walkers, 80 steps, 4 M nodes of 50 edges 1428 -> 1237 us with the making of the table
// (12).  60 nodes to a line of 128 bytes, start and two ends read apart, were a fifth smaller and no
// better: 1 M nodes 1132 us against 1166, but 200 k walkers 266 against 263, 4 M nodes of 8 edges 673
// against 668.
constexpr int kRecordNodes = 6;

// Whether a table of the offsets is made in front of a walk: where they outgrow an L2 by far or by a little, the
// walkers fill the chip (fewer wait for the longer step instead: 50 k walkers, 80 steps 126 -> 135 us) and the steps earn
// the table back.  Offsets as they are / table, us, 20 to 50 edges a node, walkers x steps:
//                  300 k x 10   300 k x 20   300 k x 80    1 M x 4      1 M x 10     1 M x 80
//   131 k nodes     43/46        78/80       254/250       57/57       133/129      846/801
//   500 k           55/54       101/98       360/340       77/72       176/163     1207/1124
//     2 M           54/54        94/90       304/274       80/74       171/154     1024/897
//     8 M           59/72        99/114      313/314       88/96       180/183     1021/952
//    16 M           63/87       113/132      369/365       91/113      195/206     1194/1108
bool packed_pays(int64_t num_nodes, int64_t nnz, int64_t n, int64_t length) {
  return num_nodes >= (int64_t(1) << 18) && num_nodes < (int64_t(1) << 32) && nnz < (int64_t(1) << 32) &&
         n >= (int64_t(1) << 18) && length > 0 &&
         n >= ((int64_t(1) << 21) + num_nodes * 3 / 2 + length - 1) / length;
}
size_t table_bytes(int64_t num_nodes) {
  return padded(static_cast<size_t>((num_nodes + kRecordNodes - 1) / kRecordNodes) * sizeof(uint4));
}

__global__ void __launch_bounds__(kThreads)
pack_offsets_kernel(const int64_t* __restrict__ indptr, int64_t num_nodes, int64_t records,
                    uint4* __restrict__ table) {
  const int64_t r = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
  if (r >= records) return;
  int64_t at[kRecordNodes + 1];
#pragma unroll
  for (int k = 0; k <= kRecordNodes; ++k) {
    const int64_t v = r * kRecordNodes + k;
    at[k] = indptr[v < num_nodes ? v : num_nodes];
  }
  bool fits = static_cast<uint64_t>(at[0]) < (1ull << 32) &&
              static_cast<uint64_t>(at[kRecordNodes] - at[0]) < (1ull << 16);
  uint32_t end[kRecordNodes];
#pragma unroll
  for (int k = 0; k < kRecordNodes; ++k) {
    fits &= at[k + 1] >= at[k];
    end[k] = static_cast<uint32_t>(at[k + 1] - at[0]);
  }
  table[r] = fits ? make_uint4(static_cast<uint32_t>(at[0]), end[1] << 16 | end[0],
                               end[3] << 16 | end[2], end[5] << 16 | end[4])
                  : make_uint4(0u, 1u, 0u, 0u);
}

// PACKED: the offsets come from `table`, made for this call from indptr
template <typename IdT, bool PACKED>
__global__ void __launch_bounds__(kThreads)
random_walk_kernel(const int64_t* __restrict__ indptr, const uint4* __restrict__ table,
                   const IdT* __restrict__ indices,
                   int64_t num_nodes, const IdT* __restrict__ seeds, int64_t n, int64_t length, uint64_t seed,
                   const uint32_t* __restrict__ replay, IdT* __restrict__ trace) {
  const int64_t w = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
  if (w >= n) return;
  int64_t curr = static_cast<int64_t>(seeds[w]);
  trace[w] = static_cast<IdT>(curr);
  const bool stream = !PACKED && indptr[num_nodes] >= kStreamBytes / static_cast<int64_t>(sizeof(IdT));
  U4 x;
  for (int64_t t = 0; t < length; ++t) {
    if (!replay && (t & 3) == 0)
      x = draw_block(seed, kTagWalk, static_cast<uint64_t>(w), static_cast<uint64_t>(t >> 2));
    int64_t pick = -1;
    if (curr >= 0) {
      const uint32_t xv = replay ? replay[t * n + w] : x.v[t & 3];
      if (!PACKED) {
        pick = step_from(indptr, indices, num_nodes, curr, xv, stream);
      } else if (curr < num_nodes) {
        const uint32_t v = static_cast<uint32_t>(curr), record = v / kRecordNodes;
        const uint32_t j = v - record * kRecordNodes, half = j >> 1;
        const uint4 r = table[record];
        const uint32_t here = half == 0 ? r.y : half == 1 ? r.z : r.w;
        const uint32_t left = half == 0 ? 0u : half == 1 ? r.y : r.z;
        const uint32_t begin = j & 1 ? here & 0xFFFFu : left >> 16;
        const uint32_t end = j & 1 ? here >> 16 : here & 0xFFFFu;
        int64_t start = static_cast<int64_t>(r.x) + begin;
        int64_t deg = static_cast<int64_t>(end - begin);
        if ((r.y & 0xFFFFu) > r.w >> 16) {
          start = indptr[curr];
          deg = indptr[curr + 1] - start;
        }
        pick = neighbour(indices, start, deg, xv, false);
      }
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

size_t gs_random_walk_workspace_bytes(int64_t num_nodes, int64_t nnz, int64_t n, int64_t length) {
  return packed_pays(num_nodes, nnz, n, length) ? table_bytes(num_nodes) : 0;
}

int gs_random_walk_workspace(const int64_t* indptr, int64_t num_nodes, const void* indices, int id_bytes,
                             const void* seeds, int64_t n, int64_t length, uint64_t seed,
                             const uint32_t* replay, void* trace, void* workspace,
                             size_t workspace_bytes, void* stream) {
  GS_REQUIRE(n >= 0 && length >= 0 && num_nodes >= 0, "gs_random_walk: negative size");
  GS_REQUIRE(n == 0 || (indptr && seeds && trace), "gs_random_walk: null pointer");
  GS_REQUIRE(valid_id_bytes(id_bytes), "gs_random_walk: id_bytes must be 4 or 8, got %d", id_bytes);
  if (n == 0) return GS_OK;
  hipStream_t st = static_cast<hipStream_t>(stream);
  uint4* table = nullptr;
  const int64_t records = (num_nodes + kRecordNodes - 1) / kRecordNodes;
  if (workspace_bytes > 0 && num_nodes > 0) {
    GS_REQUIRE(num_nodes < (int64_t(1) << 32), "gs_random_walk: too many nodes for a table of offsets");
    Carver ws(workspace, workspace_bytes);
    table = ws.take<uint4>(static_cast<size_t>(records));
    if (!ws.ok) {
      set_error_text("gs_random_walk: workspace needs %zu bytes, 256-byte aligned",
                     table_bytes(num_nodes));
      return GS_ERR_WORKSPACE;
    }
  }
  const dim3 grid(blocks_for(n, kThreads));
  ProfileScope prof("random_walk", st);
  if (table)
    hipLaunchKernelGGL(pack_offsets_kernel, dim3(blocks_for(records, kThreads)), dim3(kThreads), 0, st,
                       indptr, num_nodes, records, table);
  auto go = [&](auto kernel, auto id) {
    using IdT = decltype(id);
    hipLaunchKernelGGL(kernel, grid, dim3(kThreads), 0, st, indptr, table,
                       static_cast<const IdT*>(indices), num_nodes, static_cast<const IdT*>(seeds), n,
                       length, seed, replay, static_cast<IdT*>(trace));
  };
  if (id_bytes == 8)
    go(table ? random_walk_kernel<int64_t, true> : random_walk_kernel<int64_t, false>, int64_t());
  else
    go(table ? random_walk_kernel<int32_t, true> : random_walk_kernel<int32_t, false>, int32_t());
  return check_launch("random_walk");
}

int gs_random_walk(const int64_t* indptr, int64_t num_nodes, const void* indices, int id_bytes,
                   const void* seeds, int64_t n, int64_t length, uint64_t seed, const uint32_t* replay,
                   void* trace, void* stream) {
  return gs_random_walk_workspace(indptr, num_nodes, indices, id_bytes, seeds, n, length, seed, replay,
                                  trace, nullptr, 0, stream);
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
