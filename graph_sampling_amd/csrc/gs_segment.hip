// Segment (SpMV-style) reductions over edge data on gfx950.
//
// Replaces impl::CSCSumCUDA, impl::COOSumCUDA, impl::CSCNormalizeCUDA
// (reference src/cuda/graph_ops.cu:92,122,184) and impl::fusion::COOEDivUSum
// (src/cuda/fusion/edge_map_reduce.cu:10).
//
// The reference gives every segment to one thread (graph_ops.cu:16-39), which
// stalls a whole wave on a power-law hub.  Here the edges are cut into tiles of 4096,
// one workgroup each.  The tile's data go to LDS in one coalesced sweep and are not read
// again: segments of at most 16 edges are added up there by a lane each, in edge order
// (bit-identical to a sequential sum), up to 128 edges by 16 lanes, longer ones by a
// wave; a normalise divides in place and stores the tile.  A segment that crosses a tile
// border leaves a piece in either tile (one of at most 16 edges belongs to the tile it
// starts in, whole); the pieces are added up in tile order, and the edges of crossing
// segments, about a third of them on a power-law graph, are all that a normalise reads a
// second time.  A 300 000-edge hub is 75 workgroups' work, and the order of the additions
// is fixed by the edges' layout alone, so results repeat from run to run.
//
// Tiles, marks and pieces count from the first offset, so a range of a larger matrix's columns,
// offsets and data as they stand there, costs what its own edges cost.
//
// A workgroup learns its segments from the offsets, 64 at a time in each wave, from the one
// that holds its first edge on; with few edges per segment (a slice's rows among all rows:
// millions of empty segments) from one int per edge that a pass over the offsets has left at
// every segment's first edge.
//
// 124 M edges in 2.45 M columns (half of them of at most 16 edges, 19 % of the edges in columns
// longer than a tile), as streams (kStreamEdges), kernels of one of each in turn: sum 116 us (4.7 TB/s; the bytes
// bound it: tiles 105 of it), normalise 236 us (4.3 TB/s over the bytes it needs, 5.0 with the second reading: tiles
// 151, the crossing segments 79; each tile's chain of LDS steps hides behind the other tiles of its
// CU); the calls 348-353 (plainly 380-390).  A lane per short column, a scan per 1024-edge chunk for the
// others and a divide pass over all edges, each reading its edges for itself, took 214 and 380.  Tiles of 8192 edges:
// 156 and 324, against 144 and 308 as the tiles of 4096 were then, plainly.  Workgroups that stay for two or four
// tiles, the next one's data on their way while one is added up: 64 registers are too few for that, and at 96 both
// calls took 449 us against 357.
#include <limits>
#include "gs_common.hpp"

namespace gs {
namespace {

constexpr int kThreads = 256;
constexpr int64_t kLaneMaxLen = 16;

constexpr int kLaneEdges = 4;        // of one 16-byte read
constexpr int kTileItems = 16;          // of a thread in the passes before and behind the tiles
constexpr int kTile = kThreads * kTileItems;
constexpr int kGroup = 16;              // lanes that add up a segment of 17 .. kGroupMaxLen edges
constexpr int kGroupMaxLen = 128;

struct Tiles {
  int* head;      // [tiles + 1] segment of the tile's first edge; behind the last: of the last edge
  int* outgoing;  // [tiles] long segment that starts here and goes on after the tile, or -1
  float* carry;   // [tiles][2] piece of the incoming long segment, piece of the outgoing one
  int* inner;     // [tiles] normalise: first | end << 16 of the edges that are done
  int* mark;      // [edges] kMarks: the segment that starts at the edge, or -1
};

// The edges of the offsets.  The caller's count is an upper bound; there is workspace for that many.
struct Edges {
  int64_t first, end;
  __device__ __forceinline__ Edges(const int64_t* __restrict__ indptr, int64_t num_seg, int64_t nnz)
      : first(indptr[0]), end(indptr[num_seg]) {
    if (end - first > nnz) end = first + nnz;
  }
  // Edges of the tile that begins at p0 < end.  (The empty statement holds the number apart from
  // comparisons of it with a whole tile: where the compiler folds such a one into the minimum's, it
  // loses the instruction that hands the result to the selection, and every tile counts as whole.)
  __device__ __forceinline__ int in_tile(int64_t p0) const {
    int n = static_cast<int>(end - p0 < kTile ? end - p0 : kTile);
    asm volatile("" : "+s"(n));
    return n;
  }
};

// How a workgroup learns its segments.
enum Walk {
  kSearch,  // it searches the offsets for the tile's first and last, and leaves the first in head[]
  kHeads,   // head[] is there (tile_heads_kernel)
  kMarks    // head[] and mark[] are
};

__global__ void __launch_bounds__(kThreads) clear_marks_kernel(int* mark, int64_t n) {
  const int64_t i0 = static_cast<int64_t>(blockIdx.x) * kTile + threadIdx.x;
#pragma unroll
  for (int k = 0; k < kTileItems; ++k)
    if (i0 + k * kThreads < n) mark[i0 + k * kThreads] = -1;
}

// head[] of every tile that begins inside a segment; mark[]; a sum's empty segments
template <bool SUM, bool MARK, typename IdT>
__global__ void __launch_bounds__(kThreads)
tile_heads_kernel(const int64_t* __restrict__ indptr, const IdT* __restrict__ nmap, int64_t num_seg,
                  int64_t nnz, float* __restrict__ out, Tiles tl) {
  const int64_t s = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
  const Edges edges(indptr, num_seg, nnz);
  int64_t t0 = 0, t1 = -1;
  if (s < num_seg) {
    const int64_t begin = indptr[s], end = indptr[s + 1];
    if (end > begin) {
      const int64_t stop = end < edges.end ? end : edges.end;
      t0 = (begin - edges.first + kTile - 1) / kTile;
      t1 = (stop - edges.first - 1) / kTile;
      if (begin < stop) {
        if (stop == edges.end) tl.head[t1 + 1] = static_cast<int>(s);
        if (MARK) tl.mark[begin - edges.first] = static_cast<int>(s);
      } else if (SUM) {  // (behind the last edge that counts)
        out[nmap ? static_cast<int64_t>(nmap[s]) : s] = 0.0f;
      }
    } else if (SUM) {
      out[nmap ? static_cast<int64_t>(nmap[s]) : s] = 0.0f;
    }
  }
  const bool wide = t1 - t0 >= kWave;
  if (!wide)
    for (int64_t t = t0; t <= t1; ++t) tl.head[t] = static_cast<int>(s);
  unsigned long long todo = __ballot(wide);
  const int lane = threadIdx.x & (kWave - 1);
  while (todo) {
    const int src = __ffsll(static_cast<long long>(todo)) - 1;
    todo &= todo - 1;
    const int64_t w0 = __shfl(t0, src, kWave), w1 = __shfl(t1, src, kWave);
    const int64_t ws = __shfl(s, src, kWave);
    for (int64_t t = w0 + lane; t <= w1; t += kWave) tl.head[t] = static_cast<int>(ws);
  }
}

// first and last tile of segment g, which has edges
__device__ __forceinline__ void tiles_of(const int64_t* __restrict__ indptr, int64_t g,
                                         const Edges& edges, int64_t* from, int64_t* to) {
  const int64_t end = indptr[g + 1] < edges.end ? indptr[g + 1] : edges.end;
  *from = (indptr[g] - edges.first) / kTile;
  *to = (end - edges.first - 1) / kTile;
}

// sum over the 16 lanes of a row, in every lane
__device__ __forceinline__ float row_sum(float x) {
  x += lane_move<0x128>(x);
  x += lane_move<0x124>(x);
  x += lane_move<0x122>(x);
  return x + lane_move<0x121>(x);
}

using F4 = float __attribute__((ext_vector_type(4)));

// Source: where a tile's data come from.
enum Source {
  kPlain,     // data[edge], 16-byte aligned
  kStreamed,  // the same, of at least kStreamEdges edges (a sum: and kStreamSumBytes)
  kLoose,     // data[edge]
  kMapped     // data[emap[edge]]
};

// From here on data and results (8 bytes an edge) are more than the 256 MB that the memory-side
// cache holds, and reads and writes past it that say so are the faster ones: a bare read of 496 MB 6.5 TB/s
// against 5.9, sum and normalise of 124 M edges 390 -> 357 us, of 60 M 245 -> 229, of 40 M 150 -> 142.
// Shorter arrays gain less or nothing (16 M edges 118 -> 114), and what reads a result soon
// after finds it in the cache no more (normalise, then the sum of its result: 16 M edges 84 -> 85.5,
// 32 M the same, 60 M 218 -> 212).
constexpr int64_t kStreamEdges = int64_t(1) << 25;
// A sum leaves its data where they were: from so many bytes of data, offsets and sums on, 4 an edge and 12 a segment.
// The same array summed again and again / three in turn, plain -> as a stream, us: 34 M edges, 80 k segments 32.3 ->
// 33.7 / 33.6 -> 33.4, 40 M, 5 M segments (220 MB) 133.6 -> 138.9 / 138.2 -> 138.2, 62.5 M, 1.2 M segments (265 MB)
// 65.0 -> 70.7 / 65.4 -> 66.9, 64 M, 0.13 M segments (258 MB) 51.1 -> 54.4 / 54.2 -> 53.8; 64 M, 8 M segments (352 MB)
// 148.5 -> 139.2 / 148.0 -> 139.0, 100 M, 10 M segments 229.5 -> 204.9 / 229.7 -> 204.2.
constexpr int64_t kStreamSumBytes = int64_t(1) << 28;

template <Source SOURCE>
__device__ __forceinline__ F4 read_four(const float* at) {
  const F4* p = reinterpret_cast<const F4*>(at);
  return SOURCE == kStreamed ? __builtin_nontemporal_load(p) : *p;
}
template <Source SOURCE>
__device__ __forceinline__ void write_four(float* at, F4 v) {
  F4* p = reinterpret_cast<F4*>(at);
  if (SOURCE == kStreamed) __builtin_nontemporal_store(v, p);
  else *p = v;
}

// One tile.  Once the data are in LDS (the first barrier) the waves go their own ways: each takes
// an equal share of the segments that start in the tile (with marks: those that start in its share
// of the edges), the first one the incoming segment as well, 64 at a time -- the short ones a
// lane each, what is longer from a list in LDS of the wave's own, four at a time or one by one.
// With lists and flags shared by the workgroup and a barrier after every step a tile took 12 us
// where it takes 7, which is what held the chip back; with the segments dealt out by
// quarters of the edges, one tile of 16 k segments kept a wave busy for 80 us at the end.
// Its 64 segments after 64 are a wave's serial chain, the longest where columns are many and short
// (a tile of 16 k of them, most empty), so how many waves share a tile goes by what there is
// to wait for it (tile_threads).
template <bool NORMALIZE, Source SOURCE, Walk WALK, int THREADS, typename IdT>
__global__ void __launch_bounds__(THREADS, WALK == kMarks || SOURCE == kMapped ? 4 : 8)
segment_tiles_kernel(const int64_t* __restrict__ indptr, const int64_t* __restrict__ emap,
                     const IdT* __restrict__ nmap, const float* __restrict__ data,
                     int64_t num_seg, int64_t nnz, int powk, float* __restrict__ out, Tiles tl) {
  constexpr bool EMAP = SOURCE == kMapped, PLAIN = SOURCE == kPlain || SOURCE == kStreamed;
  constexpr int kWaves = THREADS / kWave, kItems = kTile / THREADS;
  __shared__ __attribute__((aligned(16))) float s_v[kTile];
  __shared__ uint32_t s_list[kWaves][kWave];
  __shared__ int64_t s_head[2];
  __shared__ int s_first, s_end, s_out;  // edges in front of `first`, from `end` on: of crossing segments
  // (the last tile first: where columns are numbered with the busy ones in front, the tiles of
  // thousands of columns, which take several times as long, come last, and the chip would wait for
  // the last of them: 144 -> 128 us)
  const int64_t t = gridDim.x - 1 - blockIdx.x;
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
  // (what the chain of dependent reads starts with goes out first; the data wait for the first and
  // the last offset, since an array may end where the offsets do: sum and normalise of 124 M
  // edges 391 us with that wait, 389 without)
  int left_head = 0, left_tail = 0;
  if (WALK != kSearch) {
    left_head = tl.head[t];
    if (WALK == kHeads) left_tail = tl.head[t + 1];
  }
  const Edges edges(indptr, num_seg, nnz);
  // (both are asked for before the workgroup knows whether it has edges)
  if (WALK != kSearch) asm volatile("" : "+s"(left_head), "+s"(left_tail));
  int64_t head = left_head, tail = left_tail;  // segments of the tile's first edge and of the one behind its last
  const int64_t p0 = edges.first + t * kTile;
  if (p0 >= edges.end) return;
  const int n = edges.in_tile(p0);
  const int64_t p1 = p0 + n;
  const bool vec = PLAIN && n == kTile && (reinterpret_cast<uintptr_t>(data + p0) & 15u) == 0;
  F4 q[kItems / kLaneEdges];
  if (vec) {
#pragma unroll
    for (int k = 0; k < kItems / kLaneEdges; ++k)
      q[k] = read_four<SOURCE>(data + p0 + (k * THREADS + tid) * kLaneEdges);
  } else if constexpr (PLAIN) {  // (the last tile, or a first offset that is no multiple of 4)
#pragma unroll
    for (int k = 0; k < kItems / kLaneEdges; ++k)
#pragma unroll
      for (int u = 0; u < kLaneEdges; ++u) {
        const int i = (k * THREADS + tid) * kLaneEdges + u;
        q[k][u] = data[p0 + (i < n ? i : n - 1)];
      }
  }

  int64_t where[EMAP ? kItems : 1];
  float x[kItems];
  if constexpr (!PLAIN) {
    if constexpr (EMAP) {
#pragma unroll
      for (int k = 0; k < kItems; ++k) {
        const int i = k * THREADS + tid;
        where[k] = emap[p0 + (i < n ? i : n - 1)];
      }
    }
#pragma unroll
    for (int k = 0; k < kItems; ++k) {
      const int i = k * THREADS + tid;
      x[k] = data[EMAP ? where[EMAP ? k : 0] : p0 + (i < n ? i : n - 1)];
    }
  }
  if (WALK == kSearch) {
    if (wave < 2) {
      const int64_t r = wave_upper_bound(indptr, num_seg + 1, wave == 0 ? p0 : p1 - 1) - 1;
      if (lane == 0) s_head[wave] = r;
      if (tid == 0) tl.head[t] = static_cast<int>(r);
    }
    __syncthreads();
    head = s_head[0];
    tail = s_head[1];
  }
  // this wave's segments, and the offsets of the next 256 of them, four sets of 64 (the ends of a
  // set are the next one's beginnings; of the last, an entry of its own)
  const int64_t share = (tail - head + kWaves) / kWaves;
  const int64_t seg0 = head + wave * share;
  const int64_t seg1 = seg0 + share < tail + 1 ? seg0 + share : tail + 1;
  constexpr int kSets = 4;
  int64_t starts[kSets + 1];
  auto offsets = [&](int64_t first) {
#pragma unroll
    for (int u = 0; u <= kSets; ++u) {
      const int64_t r = first + u * kWave + (u < kSets ? lane : 0);
      starts[u] = indptr[r < seg1 ? r : seg1];
    }
  };
  if (WALK != kMarks && seg0 < seg1) offsets(seg0);
  if (tid == 0) {
    s_first = 0;
    s_end = n;
    s_out = -1;
  }
  // x^powk of a thread's edges, one loop for all of them (the products are powk_f's)
  if constexpr (PLAIN) {
    F4 p[kItems / kLaneEdges];
#pragma unroll
    for (int k = 0; k < kItems / kLaneEdges; ++k) p[k] = q[k];
    if (!NORMALIZE)
      for (int i = 1; i < powk; ++i) {
#pragma unroll
        for (int k = 0; k < kItems / kLaneEdges; ++k) p[k] *= q[k];
      }
#pragma unroll
    for (int k = 0; k < kItems / kLaneEdges; ++k)
      *reinterpret_cast<F4*>(s_v + (k * THREADS + tid) * kLaneEdges) = p[k];
  } else {
    float p[kItems];
#pragma unroll
    for (int k = 0; k < kItems; ++k) p[k] = x[k];
    if (!NORMALIZE)
      for (int i = 1; i < powk; ++i) {
#pragma unroll
        for (int k = 0; k < kItems; ++k) p[k] *= x[k];
      }
#pragma unroll
    for (int k = 0; k < kItems; ++k) s_v[k * THREADS + tid] = p[k];
  }
  __syncthreads();

  auto put = [&](int64_t seg, float total) {
    out[nmap ? static_cast<int64_t>(nmap[seg]) : seg] = total;
  };
  // A segment of at most 16 edges, one lane; what of it lies in the next tile included, which
  // leaves it alone.
  auto short_one = [&](int64_t seg, int64_t begin, int64_t end) {
    const int at = static_cast<int>(begin - p0);
    const int stop = static_cast<int>((end < p1 ? end : p1) - p0);
    float acc = 0.0f;
    for (int j = at; j < stop; j += 4) {  // (four reads, then four additions in edge order)
      float v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) v[u] = s_v[j + u < kTile ? j + u : kTile - 1];
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (j + u < stop) acc += v[u];
    }
    for (int64_t e = p1; e < end; ++e) {
      const float v = data[EMAP ? emap[e] : e];
      acc += NORMALIZE ? v : powk_f(v, powk);
    }
    if (NORMALIZE) {
      for (int j = at; j < stop; ++j) s_v[j] = s_v[j] / acc;
      for (int64_t e = p1; e < end; ++e) {
        const int64_t d = EMAP ? emap[e] : e;
        out[d] = data[d] / acc;
      }
    } else {
      put(seg, acc);
    }
  };
  // Up to 64 segments, one a lane (seg < 0: none): the lane's starts in the wave's share, or is the
  // incoming one.
  // Without marks, lane l's is segment base + l.
  auto round = [&](int64_t base, int64_t seg, int64_t begin, int64_t end) {
    const bool here = seg >= 0;
    const bool incoming = here && begin < p0;
    const bool is_long = here && end - begin > kLaneMaxLen;
    const int at = static_cast<int>((incoming ? p0 : begin) - p0);
    const int stop = static_cast<int>((end < p1 ? end : p1) - p0);
    const int len = stop - at;
    if (incoming) s_first = stop;
    const bool outgoing = is_long && !incoming && end > p1;
    if (outgoing) {
      s_end = at;
      s_out = static_cast<int>(seg);
    }
    if (here && !is_long && !incoming) short_one(seg, begin, end);
    // where a long segment's sum goes: 0 its own place, 1 the incoming piece's, 2 the outgoing one's
    const int kind = incoming ? 1 : (outgoing ? 2 : 0);
    auto finish = [&](int k, int64_t s, float total) {
      if (k == 1) tl.carry[2 * t] = total;
      else if (k == 2) tl.carry[2 * t + 1] = total;
      else if (!NORMALIZE) put(s, total);
    };
    const bool few = is_long && len <= kGroupMaxLen;
    const unsigned long long list = __ballot(few);
    if (list) {
      const int count = __popcll(list);
      // {first edge: 12 bits, edges less one: 7, lane: 6, kind: 2}
      if (few)
        s_list[wave][__popcll(list & ((1ull << lane) - 1ull))] =
            static_cast<uint32_t>(at) | static_cast<uint32_t>(len - 1) << 12 |
            static_cast<uint32_t>(lane) << 19 | static_cast<uint32_t>(kind) << 25;
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      for (int i0 = 0; i0 < count; i0 += kWave / kGroup) {
        const int i = i0 + lane / kGroup, j0 = lane & (kGroup - 1);
        const bool live = i < count;
        const uint32_t w = s_list[wave][live ? i : 0];
        const int left = live ? static_cast<int>((w >> 12) & 0x7F) + 1 - j0 : 0;
        const int from = left > 0 ? static_cast<int>(w & 0xFFF) + j0 : 0;
        constexpr int kEach = kGroupMaxLen / kGroup;
        float v[kEach];
#pragma unroll
        for (int u = 0; u < kEach; ++u) v[u] = s_v[from + (u * kGroup < left ? u * kGroup : 0)];
        float acc = 0.0f;
#pragma unroll
        for (int u = 0; u < kEach; ++u)
          if (u * kGroup < left) acc += v[u];
        const float total = row_sum(acc);
        const int src = static_cast<int>((w >> 19) & 63), k = static_cast<int>(w >> 25);
        const int64_t s = WALK == kMarks ? __shfl(seg, src, kWave) : base + src;
        if (live && j0 == 0) finish(k, s, total);
        if (NORMALIZE && k == 0) {
#pragma unroll
          for (int u = 0; u < kEach; ++u)
            if (u * kGroup < left) s_v[from + u * kGroup] = v[u] / total;
        }
      }
      __builtin_amdgcn_wave_barrier();
    }
    for (unsigned long long todo = __ballot(is_long && !few); todo; todo &= todo - 1) {
      const int src = __ffsll(static_cast<long long>(todo)) - 1;
      const int from = __builtin_amdgcn_readlane(at, src), size = __builtin_amdgcn_readlane(len, src);
      const int k = __builtin_amdgcn_readlane(kind, src);
      constexpr int kEach = 8;
      float total = 0.0f;
      for (int j = lane; j < size; j += kEach * kWave) {
        float v[kEach];
#pragma unroll
        for (int u = 0; u < kEach; ++u) v[u] = s_v[from + (j + u * kWave < size ? j + u * kWave : j)];
#pragma unroll
        for (int u = 1; u < kEach; ++u)
          if (j + u * kWave >= size) v[u] = 0.0f;
        total += ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
      }
      total = row_sum(total);
      total = (__builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, total), 0)) +
               __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, total), 16))) +
              (__builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, total), 32)) +
               __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, total), 48)));
      if (lane == src) finish(k, seg, total);
      if (NORMALIZE && k == 0)
        for (int j = lane; j < size; j += kWave) s_v[from + j] = s_v[from + j] / total;
    }
  };

  constexpr int kShare = kTile / kWaves;
  const int64_t q0 = p0 + wave * kShare;
  if (WALK == kMarks ? q0 < p1 : seg0 < seg1) {
    if (WALK == kMarks) {
      int seg[kShare / kWave];
      int64_t end[kShare / kWave];
#pragma unroll
      for (int k = 0; k < kShare / kWave; ++k) {
        const int64_t p = q0 + k * kWave + lane;
        seg[k] = p < p1 ? tl.mark[p - edges.first] : -1;
      }
      int64_t begin_in = 0;
      bool incoming = false;
      if (wave == 0) {  // the tile's incoming segment, when no segment starts at its first edge
        begin_in = indptr[head];
        incoming = lane == 0 && begin_in < p0;
        if (incoming) seg[0] = static_cast<int>(head);
      }
#pragma unroll
      for (int k = 0; k < kShare / kWave; ++k) end[k] = indptr[seg[k] >= 0 ? seg[k] + 1 : 0];
#pragma unroll 1
      for (int k = 0; k < kShare / kWave; ++k) {
        int s = seg[0];
        int64_t e = end[0];
#pragma unroll
        for (int u = 1; u < kShare / kWave; ++u)
          if (u == k) s = seg[u], e = end[u];
        if (__ballot(s >= 0) == 0ull) continue;
        round(0, s, k == 0 && incoming ? begin_in : q0 + k * kWave + lane, e);
      }
    } else {
      for (int64_t r0 = seg0;;) {
        bool any = false;
#pragma unroll 1
        for (int u = 0; u < kSets && r0 + u * kWave < seg1; ++u) {
          int64_t begin = starts[0], next = starts[1];
#pragma unroll
          for (int v = 1; v < kSets; ++v)
            if (u == v) begin = starts[v], next = starts[v + 1];
          int64_t end = __shfl_down(begin, 1, kWave);
          next = __shfl(next, 0, kWave);
          if (lane == kWave - 1) end = next;
          // (the segment behind the tile's last edge may start there)
          const int64_t r = r0 + u * kWave + lane;
          const bool mine = end > begin && begin < p1;
          if (__ballot(mine)) {
            any = true;
            round(r - lane, mine ? r : -1, begin, end);
          }
        }
        const int64_t behind = __shfl(starts[kSets], 0, kWave);
        r0 += kSets * kWave;
        if (r0 >= seg1) break;
        // after nothing but empty segments: on to the one that holds the next edge
        if (!any) {
          r0 = wave_upper_bound(indptr, num_seg + 1, behind) - 1;
          if (r0 >= seg1) break;
        }
        offsets(r0);
      }
    }
  }
  __syncthreads();
  if (tid == 0) tl.outgoing[t] = s_out;
  if constexpr (NORMALIZE) {
    const int first = s_first, stop = s_end > first ? s_end : first;
    if (tid == 0) tl.inner[t] = first | stop << 16;
    if constexpr (EMAP) {
#pragma unroll
      for (int k = 0; k < kItems; ++k) {
        const int i = k * THREADS + tid;
        if (i >= first && i < stop) out[where[k]] = s_v[i];
      }
    } else if (vec && (reinterpret_cast<uintptr_t>(out + p0) & 15u) == 0) {
#pragma unroll
      for (int k = 0; k < kItems / kLaneEdges; ++k) {
        const int i = (k * THREADS + tid) * kLaneEdges;
        const F4 v = *reinterpret_cast<const F4*>(s_v + i);
        if (i >= first && i + 3 < stop) {
          write_four<SOURCE>(out + p0 + i, v);
        } else {
          if (i >= first && i < stop) out[p0 + i] = v.x;
          if (i + 1 >= first && i + 1 < stop) out[p0 + i + 1] = v.y;
          if (i + 2 >= first && i + 2 < stop) out[p0 + i + 2] = v.z;
          if (i + 3 >= first && i + 3 < stop) out[p0 + i + 3] = v.w;
        }
      }
    } else {
#pragma unroll
      for (int k = 0; k < kItems; ++k) {
        const int i = k * THREADS + tid;
        if (i >= first && i < stop) out[p0 + i] = s_v[i];
      }
    }
  }
}

// Sum of the pieces of a long segment behind its first tile, by a whole workgroup; in every thread.
// s_part: a float per wave.
__device__ __forceinline__ float sum_pieces(const Tiles& tl, int64_t from, int64_t to, float* s_part) {
  constexpr int kEach = 8;  // reads of a thread in flight
  float part = 0.0f;
  for (int64_t k0 = from + 1 + threadIdx.x; k0 <= to; k0 += kEach * kThreads) {
    float v[kEach];
#pragma unroll
    for (int u = 0; u < kEach; ++u) v[u] = tl.carry[2 * (k0 + u * kThreads <= to ? k0 + u * kThreads : to)];
#pragma unroll
    for (int u = 0; u < kEach; ++u)
      if (k0 + u * kThreads <= to) part += v[u];
  }
#pragma unroll
  for (int d = kWave / 2; d > 0; d >>= 1) part += __shfl_xor(part, d, kWave);
  if ((threadIdx.x & (kWave - 1)) == 0) s_part[threadIdx.x / kWave] = part;
  __syncthreads();
  float total = 0.0f;
#pragma unroll
  for (int w = 0; w < kThreads / kWave; ++w) total += s_part[w];
  __syncthreads();
  return total;
}

// Normalise, launches of more than kHubLaunch tiles: the sum of a segment of more than kHubTiles of
// them goes to its outgoing piece's place once, where otherwise each of its tiles adds up all the
// pieces for itself, a square of reads (one segment of 130 M edges: 691 us with it, of 140 M 342
// without).  The launch costs a graph without such a segment 7 us, 264 -> 269 for 124 M edges,
// hence not for fewer tiles.  One segment of so many at most starts in a workgroup's tiles.
constexpr int64_t kHubTiles = 1024;
constexpr int64_t kHubLaunch = 32768;

__global__ void __launch_bounds__(kThreads)
hub_totals_kernel(const int64_t* __restrict__ indptr, int64_t num_seg, int64_t nnz, Tiles tl) {
  __shared__ int64_t s_from, s_to;
  __shared__ float s_part[kThreads / kWave];
  const Edges edges(indptr, num_seg, nnz);
  if (threadIdx.x == 0) s_to = -1;
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kHubTiles / kThreads; ++k) {
    const int64_t t = static_cast<int64_t>(blockIdx.x) * kHubTiles + k * kThreads + threadIdx.x;
    const int g = edges.first + t * kTile < edges.end ? tl.outgoing[t] : -1;
    if (g < 0) continue;
    int64_t from, to;
    tiles_of(indptr, g, edges, &from, &to);
    if (to - from > kHubTiles) {
      s_from = from;
      s_to = to;
    }
  }
  __syncthreads();
  if (s_to < 0) return;
  const float total = sum_pieces(tl, s_from, s_to, s_part);
  if (threadIdx.x == 0) tl.carry[2 * s_from + 1] += total;
}

// The edges of segments that cross tile borders: what lies in front of a tile's inner edges
// belongs to the incoming segment, what lies behind to the outgoing one.  Each workgroup adds
// up the pieces of its two segments for itself, a wave each or, of segments over more than 64
// tiles, the whole workgroup (one segment of 32 M edges: 191 -> 85 us, of 100 M 1321 -> 458);
// `hubs`: the totals of those over more than kHubTiles are there.
template <Source SOURCE>
__global__ void __launch_bounds__(kThreads)
crossing_divide_kernel(const int64_t* __restrict__ indptr, const int64_t* __restrict__ emap,
                       const float* __restrict__ data, int64_t num_seg, int64_t nnz,
                       float* __restrict__ out, Tiles tl, bool hubs) {
  constexpr bool EMAP = SOURCE == kMapped;
  __shared__ float s_total[2];
  __shared__ int s_wide[2];  // whether the segment spans more than 64 tiles
  __shared__ int64_t s_tiles[2][2];
  __shared__ float s_part[kThreads / kWave];
  const int64_t t = blockIdx.x;
  const Edges edges(indptr, num_seg, nnz);
  const int64_t p0 = edges.first + t * kTile;
  int inner = tl.inner[t], g_in = tl.head[t], g_out = tl.outgoing[t];
  asm volatile("" : "+s"(inner), "+s"(g_in), "+s"(g_out));  // (asked for in front of the branch)
  if (p0 >= edges.end) return;
  const int n = edges.in_tile(p0);
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
  int first = inner & 0xFFFF;
  const int stop = inner >> 16;
  if (first > 0 && indptr[g_in + 1] - indptr[g_in] <= kLaneMaxLen) first = 0;  // (done where it starts)
  if (first == 0 && stop == n) return;
  const bool vec = !EMAP && n == kTile &&
                   ((reinterpret_cast<uintptr_t>(data + p0) | reinterpret_cast<uintptr_t>(out + p0)) & 15u) == 0;
  F4 v[kTileItems / 4];
  if (vec) {
#pragma unroll
    for (int k = 0; k < kTileItems / 4; ++k) {
      const int i = k * (4 * kThreads) + 4 * tid;
      v[k] = 0.0f;
      if (i < first || i + 3 >= stop) v[k] = read_four<SOURCE>(data + p0 + i);
    }
  }
  if (wave < 2) {
    const int g = wave == 0 ? (first > 0 ? g_in : -1) : g_out;
    int64_t from = 0, to = 0;
    if (g >= 0) {
      tiles_of(indptr, g, edges, &from, &to);
      if (to - from <= kWave) {
        float part = from + 1 + lane <= to ? tl.carry[2 * (from + 1 + lane)] : 0.0f;
#pragma unroll
        for (int d = kWave / 2; d > 0; d >>= 1) part += __shfl_xor(part, d, kWave);
        if (lane == 0) s_total[wave] = tl.carry[2 * from + 1] + part;
      }
    }
    if (lane == 0) {
      s_wide[wave] = to - from > kWave;
      s_tiles[wave][0] = from;
      s_tiles[wave][1] = to;
    }
  }
  __syncthreads();
  if (s_wide[0] | s_wide[1]) {  // (the same for the whole workgroup)
    for (int r = 0; r < 2; ++r) {
      if (!s_wide[r]) continue;
      const int64_t from = s_tiles[r][0], to = s_tiles[r][1];
      const float rest = hubs && to - from > kHubTiles ? 0.0f : sum_pieces(tl, from, to, s_part);
      if (tid == 0) s_total[r] = tl.carry[2 * from + 1] + rest;
    }
    __syncthreads();
  }
  const float before = s_total[0], behind = s_total[1];
  if (vec) {
#pragma unroll
    for (int k = 0; k < kTileItems / 4; ++k) {
      const int i = k * (4 * kThreads) + 4 * tid;
      if (i + 3 < first || i >= stop) {
        const float d = i >= stop ? behind : before;
        write_four<SOURCE>(out + p0 + i, F4{v[k].x / d, v[k].y / d, v[k].z / d, v[k].w / d});
      } else if (i < first || i + 3 >= stop) {
        const float w[4] = {v[k].x, v[k].y, v[k].z, v[k].w};
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          if (i + u < first) out[p0 + i + u] = w[u] / before;
          else if (i + u >= stop) out[p0 + i + u] = w[u] / behind;
        }
      }
    }
    return;
  }
  for (int i = tid; i < n; i += kThreads)
    if (i < first || i >= stop) {
      const int64_t d = EMAP ? emap[p0 + i] : p0 + i;
      out[d] = data[d] / (i < first ? before : behind);
    }
}

constexpr int64_t kCarryAlone = 16;  // pieces a single lane adds up by itself

// One lane per tile: a tile that holds the head of a long segment going on after it adds
// up the pieces, in tile order.  A segment that goes on over more than 16 tiles (a hub
// column) is added up by the whole wave instead of one lane walking the pieces.
template <typename IdT>
__global__ void __launch_bounds__(kThreads)
carry_kernel(const int64_t* __restrict__ indptr, const IdT* __restrict__ nmap, int64_t num_seg,
             int64_t nnz, float* __restrict__ sums, Tiles tl) {
  const Edges edges(indptr, num_seg, nnz);
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t t = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
  int g = -1;
  int64_t from = 0, last = 0;  // tiles the segment starts in and reaches
  if (edges.first + t * kTile < edges.end) {
    g = tl.outgoing[t];
    if (g >= 0) tiles_of(indptr, g, edges, &from, &last);
  }
  const bool wide = g >= 0 && last - t > kCarryAlone;
  if (g >= 0 && !wide) {
    float total = tl.carry[2 * t + 1];
    for (int64_t k = t + 1; k <= last; ++k) total += tl.carry[2 * k];
    sums[nmap ? static_cast<int64_t>(nmap[g]) : g] = total;
  }
  unsigned long long todo = __ballot(wide);
  while (todo) {
    const int l = __ffsll(static_cast<long long>(todo)) - 1;
    todo &= todo - 1;
    const int64_t next = __shfl(t, l, kWave) + 1;
    const int64_t to = __shfl(last, l, kWave);
    float part = 0.0f;
    for (int64_t k = next + lane; k <= to; k += kWave) part += tl.carry[2 * k];
#pragma unroll
    for (int d = kWave / 2; d > 0; d >>= 1) part += __shfl_xor(part, d, kWave);
    if (lane == l) sums[nmap ? static_cast<int64_t>(nmap[g]) : g] = tl.carry[2 * t + 1] + part;
  }
}

inline Source source_of(const int64_t* emap, const float* data, bool streams) {
  if (emap) return kMapped;
  if ((reinterpret_cast<uintptr_t>(data) & 15u) != 0) return kLoose;
  return streams ? kStreamed : kPlain;
}

inline int64_t num_tiles(int64_t nnz) { return nnz <= 0 ? 1 : (nnz + kTile - 1) / kTile; }

// The marks cost 12 bytes per edge; walking the offsets costs a workgroup a round of 256 per
// 256 segments of its tile, and from eight rounds a tile on that is the longer way.  Of few segments no wave has
// more than one round, and clearing and setting marks are two launches: 1 k columns of 1 k edges normalised, 14 us of
// kernels, 6.5 so.
constexpr int64_t kMarkSegments = 4096;
inline bool use_marks(int64_t num_seg, int64_t nnz) { return num_seg > kMarkSegments && 2 * num_seg > nnz; }
constexpr int64_t kSearchTiles = 512;  // up to here a normalise's workgroups look for their first segment

bool carve_tiles(void* workspace, size_t bytes, int64_t num_seg, int64_t nnz, Tiles* tl) {
  Carver ws(workspace, bytes);
  const size_t tiles = static_cast<size_t>(num_tiles(nnz));
  tl->head = ws.take<int>(tiles + 1);
  tl->outgoing = ws.take<int>(tiles);
  tl->carry = ws.take<float>(2 * tiles);
  tl->inner = ws.take<int>(tiles);
  tl->mark = use_marks(num_seg, nnz) ? ws.take<int>(static_cast<size_t>(nnz > 0 ? nnz : 1)) : nullptr;
  return ws.ok;
}

size_t segment_workspace_bytes(int64_t num_seg, int64_t nnz) {
  const size_t tiles = static_cast<size_t>(num_tiles(nnz));
  return padded((tiles + 1) * 4) + 2 * padded(tiles * 4) + padded(tiles * 8) +
         (use_marks(num_seg, nnz) ? padded(static_cast<size_t>(nnz > 0 ? nnz : 1) * 4) : 0);
}

// Threads of a tile's workgroup.  A launch of few tiles ends with its longest one, and more waves
// shorten that; one of many tiles is held up by every wave's share of the common steps.  In us,
// sum / normalise of R-MAT graphs, by 256, 512 and 1024 threads:
//   262 k edges, 33 k columns    23 / 40    17 / 25    16 / 21
//   1.0 M edges, 131 k columns   34 / 54    22 / 33    17 / 25
//   8 M edges, 1 M columns       60 / 94    38 / 62    32 / 48
//   8 M edges, 250 k columns     27 / 47    21 / 35    28 / 48
//   12 M edges, 1.5 M columns    71 / 99    46 / 64    45 / 76
//   20 M edges, 1.2 M columns    52 / 78    42 / 70    60 / 107
//   40 M edges, 2.45 M columns   78 / 117   71 / 135  104 / 208
// 256 alone fell behind a lane per short column and passes of their own for the long ones where
// columns have few edges (8 M edges, 1 M columns: 43 / 56).
enum Width { kWidest = 1024, kMiddle = 512, kNarrow = 256 };
inline Width tile_threads(int64_t num_seg, int64_t nnz) {
  const int64_t tiles = num_tiles(nnz);
  if (tiles <= kSearchTiles || (tiles <= 2048 && 16 * num_seg > nnz)) return kWidest;
  return tiles <= 6144 || use_marks(num_seg, nnz) ? kMiddle : kNarrow;
}

// what the tiles' workgroups find in head[] and mark[]
template <bool SUM, typename IdT>
void launch_heads(const int64_t* indptr, const IdT* nmap, int64_t num_seg, int64_t nnz, float* out,
                  const Tiles& tl, hipStream_t st) {
  const dim3 grid(blocks_for(num_seg, kThreads));
  if (!tl.mark) {
    hipLaunchKernelGGL((tile_heads_kernel<SUM, false, IdT>), grid, dim3(kThreads), 0, st, indptr,
                       nmap, num_seg, nnz, out, tl);
    return;
  }
  hipLaunchKernelGGL(clear_marks_kernel, dim3(blocks_for(nnz, kTile)), dim3(kThreads), 0, st, tl.mark,
                     nnz);
  hipLaunchKernelGGL((tile_heads_kernel<SUM, true, IdT>), grid, dim3(kThreads), 0, st, indptr, nmap,
                     num_seg, nnz, out, tl);
}

template <typename IdT>
int segment_sum_impl(const int64_t* indptr, const int64_t* emap, const void* nmap,
                     const float* data, int64_t num_seg, int64_t nnz, int powk, float* out,
                     const Tiles& tl, hipStream_t st) {
  const IdT* nm = static_cast<const IdT*>(nmap);
  const int64_t tiles = num_tiles(nnz);
  launch_heads<true>(indptr, nm, num_seg, nnz, out, tl, st);
  const Width width = tile_threads(num_seg, nnz);
  // (so many edges that they are streamed are more than 6144 tiles)
  static_assert(kStreamEdges / kTile > 6144, "tile_threads: marks and kMiddle, or kNarrow");
  auto pick = [&](auto source) {
    constexpr Source S = decltype(source)::value;
    if constexpr (S == kStreamed)
      return tl.mark ? segment_tiles_kernel<false, S, kMarks, kMiddle, IdT>
                     : segment_tiles_kernel<false, S, kHeads, kNarrow, IdT>;
    else if (tl.mark)
      return width == kWidest ? segment_tiles_kernel<false, S, kMarks, kWidest, IdT>
                              : segment_tiles_kernel<false, S, kMarks, kMiddle, IdT>;
    return width == kWidest   ? segment_tiles_kernel<false, S, kHeads, kWidest, IdT>
           : width == kMiddle ? segment_tiles_kernel<false, S, kHeads, kMiddle, IdT>
                              : segment_tiles_kernel<false, S, kHeads, kNarrow, IdT>;
  };
  const Source source =
      source_of(emap, data, nnz >= kStreamEdges && 4 * nnz + 12 * num_seg >= kStreamSumBytes);
  auto* kernel = source == kMapped  ? pick(std::integral_constant<Source, kMapped>{})
                 : source == kLoose ? pick(std::integral_constant<Source, kLoose>{})
                 : source == kStreamed ? pick(std::integral_constant<Source, kStreamed>{})
                                    : pick(std::integral_constant<Source, kPlain>{});
  hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(tiles)), dim3(width), 0, st, indptr, emap, nm,
                     data, num_seg, nnz, powk, out, tl);
  if (tiles > 1)
    hipLaunchKernelGGL((carry_kernel<IdT>), dim3(blocks_for(tiles, kThreads)), dim3(kThreads), 0, st,
                       indptr, nm, num_seg, nnz, out, tl);
  return check_launch("segment_sum");
}

template <Source SOURCE>
void launch_normalize(Walk walk, const int64_t* indptr, const int64_t* emap, const float* data,
                      int64_t num_seg, int64_t nnz, float* out, const Tiles& tl, hipStream_t st) {
  const int64_t* no_map = nullptr;
  const int64_t tiles = num_tiles(nnz);
  const Width width = tile_threads(num_seg, nnz);
  auto* kernel = [&] {
    if constexpr (SOURCE == kStreamed)
      return walk == kMarks ? segment_tiles_kernel<true, SOURCE, kMarks, kMiddle, int64_t>
                            : segment_tiles_kernel<true, SOURCE, kHeads, kNarrow, int64_t>;
    else
      return walk == kSearch ? segment_tiles_kernel<true, SOURCE, kSearch, kWidest, int64_t>
             : walk == kMarks
                 ? (width == kWidest ? segment_tiles_kernel<true, SOURCE, kMarks, kWidest, int64_t>
                                     : segment_tiles_kernel<true, SOURCE, kMarks, kMiddle, int64_t>)
             : width == kWidest ? segment_tiles_kernel<true, SOURCE, kHeads, kWidest, int64_t>
             : width == kMiddle ? segment_tiles_kernel<true, SOURCE, kHeads, kMiddle, int64_t>
                                : segment_tiles_kernel<true, SOURCE, kHeads, kNarrow, int64_t>;
  }();
  hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(tiles)), dim3(width), 0, st, indptr, emap,
                     no_map, data, num_seg, nnz, 1, out, tl);
  const bool hubs = tiles > kHubLaunch;
  if (hubs)
    hipLaunchKernelGGL(hub_totals_kernel, dim3(blocks_for(tiles, kHubTiles)), dim3(kThreads), 0, st,
                       indptr, num_seg, nnz, tl);
  if (tiles > 1)
    hipLaunchKernelGGL((crossing_divide_kernel<SOURCE>),
                       dim3(static_cast<unsigned>(tiles)), dim3(kThreads), 0, st, indptr, emap, data,
                       num_seg, nnz, out, tl, hubs);
}

int segment_normalize_impl(const int64_t* indptr, const int64_t* emap, const float* data,
                           int64_t num_seg, int64_t nnz, float* out, const Tiles& tl,
                           hipStream_t st) {
  // (few tiles: a launch costs more than the search)
  const Walk walk = tl.mark ? kMarks : (num_tiles(nnz) > kSearchTiles ? kHeads : kSearch);
  if (walk != kSearch)
    launch_heads<false>(indptr, static_cast<const int64_t*>(nullptr), num_seg, nnz, out, tl, st);
  const Source source = source_of(emap, data, nnz >= kStreamEdges);
  auto* launch = source == kMapped  ? launch_normalize<kMapped>
                 : source == kLoose ? launch_normalize<kLoose>
                 : source == kStreamed ? launch_normalize<kStreamed>
                                       : launch_normalize<kPlain>;
  launch(walk, indptr, emap, data, num_seg, nnz, out, tl, st);
  return check_launch("segment_normalize");
}

// Sums by an arbitrary key (COO targets).  The reference adds every edge to its target with a
// global atomic (graph_ops.cu:45-64, edge_map_reduce.cu:15-23); on a power-law graph thousands
// of those hit the same address -- a hub row, or the one column a run of a column-sorted COO
// belongs to -- and queue up at the memory side (tens of ns each).  Here a workgroup first
// gathers its 2048 edges in an LDS table keyed by target (LDS atomics), then issues one global
// add per distinct target: a 300 000-edge hub costs 150 global adds instead of 300 000.  The
// adds are the hardware's fp32 adds, not the compare-and-swap loop a plain atomicAdd(float*)
// compiles to here.
constexpr int kAggEdges = 8;  // edges per thread

// Few edges are spread over more workgroups, two a thread: the launch is then a handful of trips
// to memory and an LDS table to clear, which a shorter tile has less of.  Every target of a tile costs
// an addition to memory, though, and those to one target queue up, so beyond 8192 edges short tiles
// are for eight targets an edge and more.  The launch alone in us, two / eight a thread, targets
// skewed (a sixth to a third of the edges on one) and uniform:
//            100 targets          20 k               2.45 M
//    5 k    5.1/5.3  5.1/4.9    4.5/7.2  4.0/8.9    4.3/10.2 5.0/10.1
//    8 k    6.9/5.3  7.0/4.9    5.9/7.2  4.0/9.0    4.9/10.0 5.0/10.1
//   22 k   15.0/7.7 15.5/7.4   11.6/8.9  4.6/10.2   8.6/10.1 5.5/11.8
//   30 k   19.9/9.2 20.7/8.8   15.3/10.2 5.0/9.8   10.5/12.3 6.0/11.2
// e_div_u_sum adds up by the column of a slice's edges, which come column by column: a tile has few
// of them (512 columns, 2 k to 30 k edges: 3.1-3.6/6.7-8.1; columns in random order, 1000 skewed
// ones, 20 k edges: 13/9).
constexpr int kAggFewEdges = 2;
constexpr int64_t kAggFew = int64_t(1) << 15;
constexpr int64_t kAggFewAny = int64_t(1) << 13;
constexpr int64_t kAggFewTargets = 8;  // an edge

template <int EDGES>
struct KeyedSums {
  static constexpr int kSlots = 2 * kThreads * EDGES;  // load <= 1/2
  long long key[kSlots];
  double sum[kSlots];  // (64 additions to 32-bit floats in LDS take 81 ns here, to 64-bit ones 8)
};

template <int EDGES>
__device__ __forceinline__ void keyed_clear(KeyedSums<EDGES>& t) {
  for (int i = threadIdx.x; i < t.kSlots; i += kThreads) {
    t.key[i] = -1;
    t.sum[i] = 0.0;
  }
  __syncthreads();
}

// (a negative key is no target: it is left out here, as -1 would add to a slot that stays empty for
// the next key to take)
template <int EDGES>
__device__ __forceinline__ void keyed_add(KeyedSums<EDGES>& t, long long key, float v) {
  if (key < 0) return;
  unsigned int h = static_cast<unsigned int>((static_cast<unsigned long long>(key) *
                                              0x9E3779B97F4A7C15ull) >> 40) & (t.kSlots - 1);
  while (true) {
    const long long seen = static_cast<long long>(
        atomicCAS(reinterpret_cast<unsigned long long*>(&t.key[h]), ~0ull,
                  static_cast<unsigned long long>(key)));
    if (seen == -1 || seen == key) break;
    h = (h + 1) & (t.kSlots - 1);
  }
  unsafeAtomicAdd(&t.sum[h], static_cast<double>(v));
}

// (a key of bound or more is left out)
template <int EDGES>
__device__ __forceinline__ void keyed_flush(KeyedSums<EDGES>& t, float* __restrict__ out,
                                            long long bound = 0x7FFFFFFFFFFFFFFFll) {
  __syncthreads();
  for (int i = threadIdx.x; i < t.kSlots; i += kThreads)
    if (t.key[i] >= 0 && t.key[i] < bound) unsafeAtomicAdd(out + t.key[i], static_cast<float>(t.sum[i]));
}

// out[target[e]] += f(data[emap ? emap[e] : e])   (graph_ops.cu:45-64)
// (a thread's reads go out together, clamped to the last edge, before its first addition: one
// edge at a time every addition waits for its own trips to memory)
template <typename IdT, int EDGES>
__global__ void __launch_bounds__(kThreads)
coo_sum_kernel(const IdT* __restrict__ target, const int64_t* __restrict__ emap,
               const float* __restrict__ data, int64_t E, int powk, float* __restrict__ out,
               long long bound) {
  __shared__ KeyedSums<EDGES> table;
  const int64_t base = static_cast<int64_t>(blockIdx.x) * (kThreads * EDGES) + threadIdx.x;
  IdT to[EDGES];
  int64_t at[EDGES];
  float v[EDGES];
#pragma unroll
  for (int k = 0; k < EDGES; ++k) {
    const int64_t e = base + static_cast<int64_t>(k) * kThreads;
    at[k] = e < E ? e : E - 1;
    to[k] = target[at[k]];
  }
  if (emap) {
#pragma unroll
    for (int k = 0; k < EDGES; ++k) at[k] = emap[at[k]];
  }
#pragma unroll
  for (int k = 0; k < EDGES; ++k) v[k] = data[at[k]];
  keyed_clear(table);
#pragma unroll
  for (int k = 0; k < EDGES; ++k) {
    if (base + static_cast<int64_t>(k) * kThreads < E)
      keyed_add(table, static_cast<long long>(to[k]), powk_f(v[k], powk));
  }
  keyed_flush(table, out, bound);
}

// edge_map_reduce.cu:15-23
template <typename IdT, int EDGES>
__global__ void __launch_bounds__(kThreads)
e_div_u_sum_kernel(const IdT* __restrict__ row, const IdT* __restrict__ col,
                   const float* __restrict__ data, const float* __restrict__ divisor, int64_t E,
                   float* __restrict__ out_data, float* __restrict__ out_sum) {
  __shared__ KeyedSums<EDGES> table;
  const int64_t base = static_cast<int64_t>(blockIdx.x) * (kThreads * EDGES) + threadIdx.x;
  IdT from[EDGES], to[EDGES];
  float v[EDGES], d[EDGES];
#pragma unroll
  for (int k = 0; k < EDGES; ++k) {
    const int64_t e = base + static_cast<int64_t>(k) * kThreads;
    const int64_t at = e < E ? e : E - 1;
    from[k] = row[at];
    to[k] = col[at];
    v[k] = data[at];
  }
#pragma unroll
  for (int k = 0; k < EDGES; ++k) d[k] = divisor[from[k]];
  keyed_clear(table);
#pragma unroll
  for (int k = 0; k < EDGES; ++k) {
    const int64_t e = base + static_cast<int64_t>(k) * kThreads;
    if (e < E) {
      v[k] /= d[k];
      out_data[e] = v[k];
      keyed_add(table, static_cast<long long>(to[k]), v[k]);
    }
  }
  keyed_flush(table, out_sum);
}

}  // namespace
}  // namespace gs

using namespace gs;

extern "C" {

size_t gs_segment_workspace_bytes(int64_t num_segments, int64_t nnz) {
  return segment_workspace_bytes(num_segments, nnz);
}

int gs_segment_sum(const int64_t* indptr, const int64_t* e_ids, const void* n_ids, int id_bytes,
                   const float* data, int64_t num_segments, int64_t nnz, int64_t powk, float* out,
                   void* workspace, size_t workspace_bytes, void* stream) {
  GS_REQUIRE(num_segments >= 0 && nnz >= 0 && powk >= 1,
             "gs_segment_sum: negative size or powk < 1");
  GS_REQUIRE(num_segments == 0 || (indptr && out && (nnz == 0 || data)),
             "gs_segment_sum: null pointer");
  GS_REQUIRE(!n_ids || valid_id_bytes(id_bytes), "gs_segment_sum: id_bytes must be 4 or 8, got %d",
             id_bytes);
  GS_REQUIRE(num_segments < (int64_t(1) << 31), "gs_segment_sum: more than 2^31 segments");
  if (num_segments == 0) return GS_OK;
  Tiles tl;
  if (!carve_tiles(workspace, workspace_bytes, num_segments, nnz, &tl)) {
    set_error_text("gs_segment_sum: workspace needs %zu bytes, 256-byte aligned",
                   gs_segment_workspace_bytes(num_segments, nnz));
    return GS_ERR_WORKSPACE;
  }
  auto* impl = n_ids && id_bytes == 4 ? segment_sum_impl<int32_t> : segment_sum_impl<int64_t>;
  return impl(indptr, e_ids, n_ids, data, num_segments, nnz, static_cast<int>(powk), out, tl,
              static_cast<hipStream_t>(stream));
}

int gs_coo_sum(const void* target, int id_bytes, const int64_t* e_ids, const float* data, int64_t E,
               int64_t powk, float* out, void* stream) {
  return gs::coo_sum_bounded(target, id_bytes, e_ids, data, E, powk,
                             std::numeric_limits<int64_t>::max(), out, stream);
}

}  // extern "C"

// gs_coo_sum with targets outside [0, num_targets) left out (gs_coo_sum_binned's other path)
int gs::coo_sum_bounded(const void* target, int id_bytes, const int64_t* e_ids, const float* data,
                        int64_t E, int64_t powk, int64_t num_targets, float* out, void* stream) {
  GS_REQUIRE(E >= 0 && powk >= 1, "gs_coo_sum: negative size or powk < 1");
  GS_REQUIRE(E == 0 || (target && data && out), "gs_coo_sum: null pointer");
  GS_REQUIRE(valid_id_bytes(id_bytes), "gs_coo_sum: id_bytes must be 4 or 8, got %d", id_bytes);
  if (E == 0) return GS_OK;
  const bool many_targets = num_targets != std::numeric_limits<int64_t>::max() && num_targets >= kAggFewTargets * E;
  const bool few = E <= kAggFewAny || (E < kAggFew && many_targets);
  const dim3 grid(blocks_for(E, kThreads * (few ? kAggFewEdges : kAggEdges)));
  hipStream_t st = static_cast<hipStream_t>(stream);
  auto launch = [&](auto* kernel, const auto* to) {
    hipLaunchKernelGGL(kernel, grid, dim3(kThreads), 0, st, to, e_ids, data, E,
                       static_cast<int>(powk), out, static_cast<long long>(num_targets));
  };
  if (id_bytes == 8)
    launch(few ? coo_sum_kernel<int64_t, kAggFewEdges> : coo_sum_kernel<int64_t, kAggEdges>,
           static_cast<const int64_t*>(target));
  else
    launch(few ? coo_sum_kernel<int32_t, kAggFewEdges> : coo_sum_kernel<int32_t, kAggEdges>,
           static_cast<const int32_t*>(target));
  return check_launch("coo_sum");
}

extern "C" {


int gs_segment_normalize(const int64_t* indptr, const int64_t* e_ids, const float* data,
                         int64_t num_segments, int64_t nnz, float* out, void* workspace,
                         size_t workspace_bytes, void* stream) {
  GS_REQUIRE(num_segments >= 0 && nnz >= 0 && num_segments < (int64_t(1) << 31),
             "gs_segment_normalize: negative size or more than 2^31 segments");
  GS_REQUIRE(num_segments == 0 || nnz == 0 || (indptr && data && out),
             "gs_segment_normalize: null pointer");
  if (num_segments == 0 || nnz == 0) return GS_OK;
  Tiles tl;
  if (!carve_tiles(workspace, workspace_bytes, num_segments, nnz, &tl)) {
    set_error_text("gs_segment_normalize: workspace needs %zu bytes, 256-byte aligned",
                   gs_segment_workspace_bytes(num_segments, nnz));
    return GS_ERR_WORKSPACE;
  }
  return segment_normalize_impl(indptr, e_ids, data, num_segments, nnz, out, tl,
                                static_cast<hipStream_t>(stream));
}

int gs_e_div_u_sum(const void* row, const void* col, int id_bytes, const float* data,
                   const float* divisor, int64_t E, float* out_data, float* out_sum,
                   void* stream) {
  GS_REQUIRE(E >= 0, "gs_e_div_u_sum: negative size");
  GS_REQUIRE(E == 0 || (row && col && data && divisor && out_data && out_sum),
             "gs_e_div_u_sum: null pointer");
  GS_REQUIRE(valid_id_bytes(id_bytes), "gs_e_div_u_sum: id_bytes must be 4 or 8, got %d", id_bytes);
  if (E == 0) return GS_OK;
  const bool few = E < kAggFew;
  const dim3 grid(blocks_for(E, kThreads * (few ? kAggFewEdges : kAggEdges)));
  hipStream_t st = static_cast<hipStream_t>(stream);
  auto launch = [&](auto* kernel, const auto* from, const auto* to) {
    hipLaunchKernelGGL(kernel, grid, dim3(kThreads), 0, st, from, to, data, divisor, E, out_data,
                       out_sum);
  };
  if (id_bytes == 8)
    launch(few ? e_div_u_sum_kernel<int64_t, kAggFewEdges> : e_div_u_sum_kernel<int64_t, kAggEdges>,
           static_cast<const int64_t*>(row), static_cast<const int64_t*>(col));
  else
    launch(few ? e_div_u_sum_kernel<int32_t, kAggFewEdges> : e_div_u_sum_kernel<int32_t, kAggEdges>,
           static_cast<const int32_t*>(row), static_cast<const int32_t*>(col));
  return check_launch("e_div_u_sum");
}

}  // extern "C"
