// Induced-subgraph slicing of a small node set with long columns on gfx950: what GraphSAINT-style
// samplers ask for (a few thousand visited nodes of a power-law graph, whose columns hold
// millions of edges).
//
// Same result as the general column + row slice (gs_rowslice.hip; reference
// src/cuda/fusion/column_row_slicing.cu:102-211), renamed rows and, in the same pass, the kept
// edges' data.  What differs is where the id set lives: every compute unit keeps an exact copy of
// it in LDS.
//
// A workgroup builds the set once; from then on its waves go their own ways, with no barrier
// between them: each owns a run of consecutive 512-position tiles of the virtual column slice,
// all runs of equal length and as many waves as the chip holds at once.  Per tile:
//   * position -> column from 64 staged offsets of the wave's own, bounded to the columns that 64
//     positions touch (a tile inside one column: one look at the offsets, one address);
//   * the ids of the NEXT tile are asked for before this tile's marks leave, since the few waves
//     beside the set have little else to hide that latency behind;
//   * kept edges leave one bit each and, packed to the front of the tile's range of a scratch
//     array, their new row number in 2 bytes, and beside it their datum or, with long columns, every
//     64 positions where they are in the parent (marks_read_data).
// A scan of the tile counts and one copy kernel put the pieces together; of long columns the copy reads
// the kept edges' data from the parent.  (With the tiles shared by the waves of a workgroup, offsets and counts through LDS and two barriers a tile, the marks
// took 293 us where a wave's own tiles took 225, before they were streamed.)
//
// Two forms of the set.  BitmapSet, for graphs whose numbers of nodes fit (about 600 k): a bit
// per node, the set bits before each 32-bit word, and the place of every set bit's id: three
// LDS reads per edge with no loop and no branch.  BucketSet for any ids: a 16-byte read of a
// four-slot bucket; a slot holds 18 hash bits and the id's place, a match is confirmed against
// the id itself (in LDS too up to 8192 ids), and a bucket with a free slot ends the search.
// Its loop over buckets and slots is what bounds it (a kernel of this kind that shared its tiles
// among the waves took 419 us with it where it took 293 with the bitmap).
//
// What bounds the bitmap form: nothing alone.  450 MB are 94 us at the rate of a copy, the vector ALUs are busy for
// 50 us and the LDS for 35 (46 before the bitmap's rows were turned, `slot`), and the four waves a SIMD that the
// set leaves room for overlap them in part: six and eight waves, fewer instructions and ids out of an L2 each change
// 130 us by less than 15.  7263 nodes whose columns hold 50.8 M edges, 22.0 M kept, 64-bit ids
// and weights: 130 us for the marks and 114 us for the copy (517 MB, 4.5 TB/s), where a filter and a table in the
// L2s, parent positions carried along and a gather of the data behind took 546 + 226 + 104.
#include "gs_common.hpp"

namespace gs {
namespace {

constexpr int kPer = 8;                   // positions a lane holds
constexpr int kTileShift = 9;
constexpr int kTile = kPer * kWave;       // positions of a wave's tile
constexpr int kWindow = 64;               // columns whose offsets a wave stages at a time
constexpr int kPlaceBits = 14;
constexpr int kMaxIds = (1 << kPlaceBits) - 1;  // (the last place with all tag bits set is "free")
constexpr int kStagedIds = 8192;          // ids up to which the ids themselves are in LDS as well
constexpr uint32_t kFree = ~0u;
constexpr size_t kLdsBytes = 160 * 1024;  // of a compute unit
constexpr int kUnits = 256;               // compute units
constexpr int64_t kLongColumns = 512;     // positions a column from which the copy reads the data (marks_read_data)
constexpr int64_t kMostBits = 8 * static_cast<int64_t>(kLdsBytes);

struct InducedMarks {
  unsigned long long* mask;  // one bit per position
  int32_t* word_rank;        // kept positions of the tile before each 64-position word
  int64_t* tile_counts;
  int64_t* tile_base;        // exclusive scan of tile_counts
  uint16_t* packed;          // new row numbers (places, 14 bits) of the kept edges, at the front of the tile's range
  int64_t* word_at;          // with data that the copy reads: where a word's edges are in the parent (WordAt)
  float* packed_data;        // with data that the marks read: the kept edges', beside packed
  int* outside;              // set when an id lies beyond the bitmap: the call has to be repeated
  LookbackState lb;          // of the scan of the tile counts; the marks clear it
  int64_t lb_tiles;
  int64_t n;
  int64_t tiles;
};

// Where the edges of 64 consecutive positions are in the parent: the place of the first when they are one
// column's, else the columns of the first and of the last.
struct WordAt {
  __device__ static __forceinline__ int64_t columns(int64_t first, int64_t last) {
    return INT64_MIN | (last - first) << 32 | first;
  }
  __device__ static __forceinline__ bool one(int64_t at) { return at >= 0; }
  __device__ static __forceinline__ int64_t first(int64_t at) { return at & 0xFFFFFFFF; }
  __device__ static __forceinline__ int64_t more(int64_t at) { return at >> 32 & 0x7FFFFFFF; }
};

// use(j, id) for this thread's share of the ids, eight of them asked for together: one trip to memory
// for eight is what building the set waits for.
template <int BLOCK, typename IdT, typename Use>
__device__ __forceinline__ void each_set_id(const IdT* __restrict__ ids, int n, Use use) {
  constexpr int kTogether = 8;
  for (int j0 = threadIdx.x; j0 < n; j0 += BLOCK * kTogether) {
    IdT id[kTogether];
#pragma unroll
    for (int u = 0; u < kTogether; ++u) id[u] = ids[j0 + u * BLOCK < n ? j0 + u * BLOCK : n - 1];
#pragma unroll
    for (int u = 0; u < kTogether; ++u)
      if (j0 + u * BLOCK < n) use(j0 + u * BLOCK, id[u]);
  }
}

// A bit per node number below `bound`, and a clear one for all others.
template <typename IdT>
struct BitmapSet {
  uint32_t* bits;
  uint16_t* before;  // set bits before each word
  uint32_t* place;   // two to a word: nothing, then the place of the id of every set bit
  uint32_t bound;

  // Words of the bitmap, in rows of 64.  A power-of-two-skewed graph (R-MAT's low ids are its hubs) has most of
  // its ids in words whose numbers share the lower bits, which are the LDS bank: of the cycles that look-ups kept
  // the LDS busy, three in four were conflicts.  Every row is turned by its own number.
  __host__ __device__ static __forceinline__ uint32_t slots(uint32_t bound) { return (bound / 32 + 64) & ~63u; }
  __device__ static __forceinline__ uint32_t slot(uint32_t id) {
    const uint32_t word = id >> 5;
    return (word & ~63u) | ((word + (word >> 6) * 37u) & 63u);
  }
  static size_t lds_bytes(int64_t bound, int64_t n_ids) {
    if (bound > kMostBits) return SIZE_MAX / 4;
    const size_t words = slots(static_cast<uint32_t>(bound));
    return (words * 4 + 15) / 16 * 16 + (words * 2 + 15) / 16 * 16 +
           (static_cast<size_t>(n_ids + 1) * 2 + 15) / 16 * 16;
  }
  __device__ __forceinline__ char* carve(char* lds, int64_t bound_, int n_ids) {
    const size_t words = slots(static_cast<uint32_t>(bound_));
    bound = static_cast<uint32_t>(bound_);
    bits = reinterpret_cast<uint32_t*>(lds);
    lds += (words * 4 + 15) / 16 * 16;
    before = reinterpret_cast<uint16_t*>(lds);
    lds += (words * 2 + 15) / 16 * 16;
    place = reinterpret_cast<uint32_t*>(lds);
    return lds + (static_cast<size_t>(n_ids + 1) * 2 + 15) / 16 * 16;
  }
  __device__ __forceinline__ uint32_t rank(uint32_t id) const {
    return before[slot(id)] + __popc(bits[slot(id)] & ((1u << (id & 31)) - 1u));
  }
  // every lane of the workgroup; s_scan: BLOCK / 64 + 1 words
  template <int BLOCK>
  __device__ __forceinline__ void build(const IdT* __restrict__ ids, int n_ids, int64_t* s_scan,
                                        int* outside) {
    const int words = static_cast<int>(slots(bound));
    for (int j = threadIdx.x; j < words; j += BLOCK) bits[j] = 0;
    for (int j = threadIdx.x; j < n_ids / 2 + 1; j += BLOCK) place[j] = 0;
    if (blockIdx.x == 0 && threadIdx.x == 0) *outside = 0;
    __syncthreads();
    each_set_id<BLOCK>(ids, n_ids, [&](int, IdT i) {
      const uint64_t id = static_cast<uint64_t>(static_cast<int64_t>(i));
      if (id < bound)
        atomicOr(&bits[slot(static_cast<uint32_t>(id))], 1u << (id & 31));
      else if (blockIdx.x == 0)
        *outside = 1;
    });
    __syncthreads();
    const int each = (words + BLOCK - 1) / BLOCK;
    const int first = threadIdx.x * each;
    int mine = 0;
    for (int j = first; j < first + each && j < words; ++j) mine += __popc(bits[j]);
    int64_t total;
    int run = static_cast<int>(block_exclusive_scan<BLOCK>(mine, &total, s_scan));
    for (int j = first; j < first + each && j < words; ++j) {
      before[j] = static_cast<uint16_t>(run);
      run += __popc(bits[j]);
    }
    __syncthreads();
    each_set_id<BLOCK>(ids, n_ids, [&](int j, IdT i) {
      const uint64_t id = static_cast<uint64_t>(static_cast<int64_t>(i));
      if (id >= bound) return;
      const uint32_t r = rank(static_cast<uint32_t>(id)) + 1;
      const int shift = (r & 1) * 16;
      uint32_t was = place[r >> 1];
      // the same id twice: its last place counts
      while (((was >> shift) & 0xFFFFu) < static_cast<uint32_t>(j)) {
        const uint32_t now = (was & ~(0xFFFFu << shift)) | (static_cast<uint32_t>(j) << shift);
        const uint32_t seen = atomicCAS(&place[r >> 1], was, now);
        if (seen == was) break;
        was = seen;
      }
    });
    __syncthreads();
  }
  // in[k]: id[k] is in the set; val[k] its place then (something otherwise).  The bit moved to the
  // top is the sign, and what is below it are the set bits before it: nine vector instructions an edge.
  __device__ __forceinline__ void lookup(const IdT (&id)[kPer], int (&val)[kPer], bool (&in)[kPer]) const {
    uint32_t at[kPer], w[kPer], r[kPer];
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      const uint32_t low = static_cast<uint32_t>(id[k]);
      at[k] = low < bound ? low : bound;
    }
    if (sizeof(IdT) == 8) {
      uint32_t high = 0;
#pragma unroll
      for (int k = 0; k < kPer; ++k) high |= static_cast<uint32_t>(static_cast<uint64_t>(id[k]) >> 32);
      if (__ballot(high != 0)) {
#pragma unroll
        for (int k = 0; k < kPer; ++k)
          if (static_cast<uint64_t>(id[k]) >> 32) at[k] = bound;
      }
    }
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      w[k] = bits[slot(at[k])];
      r[k] = before[slot(at[k])];
    }
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      const uint32_t top = w[k] << (~at[k] & 31);
      in[k] = static_cast<int>(top) < 0;
      r[k] += __popc(top);
    }
    const uint16_t* half = reinterpret_cast<const uint16_t*>(place);
#pragma unroll
    for (int k = 0; k < kPer; ++k) val[k] = half[r[k]];
  }
};

// Four-slot buckets of hashed ids: 4096 of them up to 8192 ids, 8192 beyond.
template <typename IdT, bool STAGED>
struct BucketSet {
  static constexpr int kBucketBits = STAGED ? 12 : 13;
  static constexpr int kBuckets = 1 << kBucketBits;
  uint4* bucket;
  IdT* s_ids;       // STAGED: the ids in LDS
  const IdT* ids;

  static size_t lds_bytes(int64_t, int64_t n_ids) {
    return static_cast<size_t>(kBuckets) * 16 +
           (STAGED ? (static_cast<size_t>(n_ids) * sizeof(IdT) + 15) / 16 * 16 : 0);
  }
  __device__ __forceinline__ char* carve(char* lds, int64_t, int n_ids) {
    bucket = reinterpret_cast<uint4*>(lds);
    lds += static_cast<size_t>(kBuckets) * 16;
    s_ids = reinterpret_cast<IdT*>(lds);
    return STAGED ? lds + (static_cast<size_t>(n_ids) * sizeof(IdT) + 15) / 16 * 16 : lds;
  }
  __device__ static __forceinline__ uint32_t mix(int64_t id) {
    return (static_cast<uint32_t>(id) ^ (static_cast<uint32_t>(id >> 32) * 0x85EBCA6Bu)) * 0x9E3779B1u;
  }
  __device__ static __forceinline__ uint32_t mix(int32_t id) {
    return static_cast<uint32_t>(id) * 0x9E3779B1u;
  }
  __device__ static __forceinline__ uint32_t home(uint32_t h) { return h >> (32 - kBucketBits); }
  __device__ static __forceinline__ uint32_t tag(uint32_t h) { return h << kPlaceBits; }  // in place
  __device__ __forceinline__ IdT id_at(uint32_t p) const { return STAGED ? s_ids[p] : ids[p]; }

  template <int BLOCK>
  __device__ __forceinline__ void build(const IdT* __restrict__ list, int n_ids, int64_t*,
                                        int* outside) {
    ids = list;
    if (blockIdx.x == 0 && threadIdx.x == 0) *outside = 0;
    for (int j = threadIdx.x; j < kBuckets; j += BLOCK)
      bucket[j] = make_uint4(kFree, kFree, kFree, kFree);
    if (STAGED) each_set_id<BLOCK>(list, n_ids, [&](int j, IdT id) { s_ids[j] = id; });
    __syncthreads();
    uint32_t* slot = reinterpret_cast<uint32_t*>(bucket);
    for (int j = threadIdx.x; j < n_ids; j += BLOCK) {
      const IdT id = id_at(j);
      const uint32_t h = mix(id);
      const uint32_t word = tag(h) | static_cast<uint32_t>(j);
      uint32_t at = home(h) * 4;
      while (true) {  // (more slots than ids: a free one comes)
        const uint32_t was = atomicCAS(&slot[at], kFree, word);
        if (was == kFree) break;
        if ((was ^ word) >> kPlaceBits == 0 && id_at(was & kMaxIds) == id) {
          atomicMax(&slot[at], word);  // the same id twice: its last place counts
          break;
        }
        at = (at + 1) & (kBuckets * 4 - 1);
      }
    }
    __syncthreads();
  }
  __device__ __forceinline__ void lookup(const IdT (&id)[kPer], int (&val)[kPer], bool (&in)[kPer]) const {
#pragma unroll
    for (int half = 0; half < kPer; half += 4) {
      uint4 b[4];
      uint32_t h[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        h[k] = mix(id[half + k]);
        b[k] = bucket[home(h[k])];
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        uint32_t at = home(h[k]);
        const uint32_t mine = tag(h[k]);
        int found = -1;
        while (true) {
          // (a free slot has all tag bits set and the one place no id has)
          const uint32_t w[4] = {b[k].x, b[k].y, b[k].z, b[k].w};
          uint32_t hit = kFree;
          int hits = 0;
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const bool same = (w[q] ^ mine) >> kPlaceBits == 0 && w[q] != kFree;
            hit = same ? w[q] : hit;
            hits += same;
          }
          if (hits) {
            if (id_at(hit & kMaxIds) == id[half + k]) {
              found = static_cast<int>(hit & kMaxIds);
            } else if (hits > 1) {
              for (int q = 0; q < 4; ++q)
                if ((w[q] ^ mine) >> kPlaceBits == 0 && w[q] != kFree &&
                    id_at(w[q] & kMaxIds) == id[half + k])
                  found = static_cast<int>(w[q] & kMaxIds);
            }
          }
          if (found >= 0 || w[3] == kFree) break;  // (slots fill in order)
          at = (at + 1) & (kBuckets - 1);
          b[k] = bucket[at];
        }
        val[half + k] = found;
        in[half + k] = found >= 0;
      }
    }
  }
};

// first r of [lo, hi] with off[r + 1] > p (offsets in order; there is one)
__device__ __forceinline__ int row_of(const int64_t* off, int lo, int hi, int64_t p) {
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (off[mid + 1] > p) hi = mid; else lo = mid + 1;
  }
  return lo;
}

// What a kept edge brings along: nothing, data[position], data[e_ids[position]]; for the copy, what lies packed beside
// its row number; for the marks, nothing but where its data are.
enum Data { kNoData, kByPosition, kByEdgeId, kPacked, kPlaces };

constexpr int kWavesPerSimd = 4;  // what the set leaves room for

template <typename IdT, typename Set, int BLOCK, Data DATA, bool STREAM>
__global__ void __launch_bounds__(BLOCK, kWavesPerSimd)
induced_mark_kernel(const int64_t* __restrict__ indptr, int64_t num_cols,
                    const IdT* __restrict__ indices, const IdT* __restrict__ cols, int64_t S,
                    const int64_t* __restrict__ sub_indptr, int64_t D, const IdT* __restrict__ ids,
                    int n_ids, int64_t bound, const float* __restrict__ data,
                    const int64_t* __restrict__ e_ids, InducedMarks m) {
  constexpr bool PLACES = DATA == kPlaces;
  __shared__ int64_t s_offsets[BLOCK / kWave][kWindow + 1];
  __shared__ int64_t s_starts[BLOCK / kWave][kWindow];  // start of the column minus its offset
  __shared__ int64_t s_scan[BLOCK / kWave + 1];
  extern __shared__ __align__(16) char lds[];
  Set set;
  set.carve(lds, bound, n_ids);
  set.template build<BLOCK>(ids, n_ids, s_scan, m.outside);

  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);  // (a scalar, and so is all that follows from it)
  constexpr int kStep = BLOCK / kWave;  // the waves of a workgroup take turns along its run
  const int64_t tile0 = m.tiles * blockIdx.x / gridDim.x + wave;
  const int64_t tile1 = m.tiles * (blockIdx.x + 1) / gridDim.x;
  if (blockIdx.x == 0) {  // (the launch behind this one uses it, under epoch 1)
    if (threadIdx.x == 0) *m.lb.error = 0u;
    for (int64_t j = threadIdx.x; j < m.lb_tiles; j += BLOCK) m.lb.status[j] = 0ull;
  }
  if (tile0 >= tile1) return;  // (no barrier from here on)

  int64_t* off = s_offsets[wave];
  int64_t* start = s_starts[wave];
  int64_t window = 0;  // first column of the window
  int row = 0;         // column of the window that holds the last position looked at
  // that column's end, and its start minus its offset (uniform: kept out of the lanes' registers,
  // so that 64 positions inside one column cost two additions)
  int64_t row_end = 0, row_start = 0;
  auto uniform = [](int64_t v) -> int64_t {
    const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<int>(v));
    const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<int>(v >> 32));
    return static_cast<int64_t>((static_cast<uint64_t>(hi) << 32) | lo);
  };
  // lane r: column first + r
  auto stage = [&](int64_t first) {
    window = first;
    row = 0;
    const int64_t r = first + lane;
    const int64_t at = sub_indptr[r < S ? r : S];
    const int64_t c = static_cast<int64_t>(cols[r < S ? r : S - 1]);
    start[lane] = (r < S && c >= 0 && c < num_cols ? indptr[c] : 0) - at;
    off[lane] = r <= S ? at : INT64_MAX;
    if (lane == 0) off[kWindow] = first + kWindow <= S ? sub_indptr[first + kWindow] : INT64_MAX;
    // (LDS operations of one wave keep their order; only the compiler has to be told)
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };

  // the column of position q, where a tile begins: its place in the window from one look at all offsets
  auto settle = [&](int64_t q) {
    if (off[kWindow] <= q) stage(wave_upper_bound(sub_indptr, S + 1, q) - 1);
    row = __popcll(__ballot(off[lane + 1] <= q));
    row_end = uniform(off[row + 1]);
    row_start = uniform(start[row]);
  };

  // where the 64 positions from q on lie in the parent (q never decreases); word_at: the same as a WordAt
  auto locate = [&](int64_t q, int64_t& word_at) -> int64_t {
    const int64_t last = (q + kWave < D ? q + kWave : D) - 1;
    int64_t p = q + lane;
    p = p < last ? p : last;
    word_at = row_start + q;
    if (last < row_end) return row_start + p;
    if (off[kWindow] <= last) {
      // the window ends among them: the next one starts at the column of the first
      if (off[kWindow] > q) {
        stage(window + row_of(off, row, kWindow - 1, q));
      } else {
        stage(wave_upper_bound(sub_indptr, S + 1, q) - 1);
      }
    }
    if (off[kWindow] <= last) {
      // more columns in 64 positions than a window holds: search the offsets themselves
      row_end = 0;
      int64_t lo = window, hi = S - 1;
      while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if (sub_indptr[mid + 1] > p) hi = mid; else lo = mid + 1;
      }
      if (PLACES) word_at = WordAt::columns(__shfl(lo, 0, kWave), __shfl(lo, kWave - 1, kWave));
      return indptr[static_cast<int64_t>(cols[lo])] + p - sub_indptr[lo];
    }
    if (off[row + 1] <= q) row = row_of(off, row + 1, kWindow - 1, q);
    row_end = uniform(off[row + 1]);
    row_start = uniform(start[row]);
    word_at = row_start + q;
    if (last < row_end) return row_start + p;
    const int r = row_of(off, row, kWindow - 1, p);
    if (PLACES) word_at = WordAt::columns(window + row, window + __builtin_amdgcn_readlane(r, kWave - 1));
    return start[r] + p;
  };

  // (STREAM: beyond the caches' size what a call reads is gone from them before anyone reads it again)
  auto once = [](const auto* p) { return STREAM ? __builtin_nontemporal_load(p) : *p; };
  IdT id[kPer];
  int64_t next_at = 0, my_at = 0;  // lane k: of word k of the tile asked for and of this one
  // (the data of all: 64 neighbours share their lines with the kept ones among them)
  float next_w[DATA == kByPosition ? kPer : 1], w[DATA == kByPosition || DATA == kByEdgeId ? kPer : 1];
  int64_t e[DATA == kByEdgeId ? kPer : 1];
  auto fetch = [&](int64_t t) {
    const int64_t q0 = t * kTile;
    if (q0 >= row_end) settle(q0);
    if (q0 + kTile <= row_end) {  // inside one column: one address
      const IdT* from = indices + row_start + q0 + lane;
#pragma unroll
      for (int k = 0; k < kPer; ++k) id[k] = once(from + k * kWave);
      if constexpr (DATA == kByPosition) {
#pragma unroll
        for (int k = 0; k < kPer; ++k) next_w[k] = once(data + row_start + q0 + lane + k * kWave);
      }
      if constexpr (DATA == kByEdgeId) {
#pragma unroll
        for (int k = 0; k < kPer; ++k) e[k] = once(e_ids + row_start + q0 + lane + k * kWave);
      }
      if (PLACES) next_at = row_start + q0 + lane * kWave;
      return;
    }
    int64_t at[kPer];
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      const int64_t q = q0 + k * kWave;
      int64_t word_at;
      at[k] = locate(q < D ? q : D - 1, word_at);
      if (PLACES && lane == k) next_at = word_at;
    }
#pragma unroll
    for (int k = 0; k < kPer; ++k) id[k] = once(indices + at[k]);
    if constexpr (DATA == kByPosition) {
#pragma unroll
      for (int k = 0; k < kPer; ++k) next_w[k] = once(data + at[k]);
    }
    if constexpr (DATA == kByEdgeId) {
#pragma unroll
      for (int k = 0; k < kPer; ++k) e[k] = once(e_ids + at[k]);
    }
  };

  stage(wave_upper_bound(sub_indptr, S + 1, tile0 * kTile) - 1);
  fetch(tile0);
  for (int64_t t = tile0; t < tile1; t += kStep) {
    const int64_t p0 = t * kTile;
    int val[kPer];
    bool in[kPer];
    set.lookup(id, val, in);
    my_at = next_at;
    if (p0 + kTile > D) {
#pragma unroll
      for (int k = 0; k < kPer; ++k)
        if (p0 + k * kWave + lane >= D) in[k] = false;
    }
    if constexpr (DATA == kByPosition) {
#pragma unroll
      for (int k = 0; k < kPer; ++k) w[k] = next_w[k];
    }
    if constexpr (DATA == kByEdgeId) {
#pragma unroll
      for (int k = 0; k < kPer; ++k) w[k] = in[k] ? data[e[k]] : 0.0f;
    }
    if (t + kStep < tile1) fetch(t + kStep);
    int before = 0, my_before = 0;
    unsigned long long my_word = 0;
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      const unsigned long long kept = __ballot(in[k]);
      if (lane == k) {
        my_word = kept;
        my_before = before;
      }
      const int rank = before + __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(kept >> 32),
                                                          __builtin_amdgcn_mbcnt_lo(
                                                              static_cast<uint32_t>(kept), 0));
      before += __popcll(kept);
      if (in[k]) {
        m.packed[p0 + rank] = static_cast<uint16_t>(val[k]);
        if constexpr (DATA == kByPosition || DATA == kByEdgeId) m.packed_data[p0 + rank] = w[k];
      }
    }
    if (lane < kPer && p0 + lane * kWave < D) {
      m.mask[(p0 >> 6) + lane] = my_word;
      m.word_rank[(p0 >> 6) + lane] = my_before;
      if (PLACES) m.word_at[(p0 >> 6) + lane] = my_at;
    }
    if (lane == 0) m.tile_counts[t] = before;
  }
}

struct TileCount {
  const int64_t* p;
  __device__ __forceinline__ int64_t operator()(int64_t i) const { return p[i]; }
};

__global__ void __launch_bounds__(256)
induced_indptr_kernel(const int64_t* __restrict__ sub_indptr, int64_t S, InducedMarks m,
                      int64_t* __restrict__ out_indptr) {
  const int64_t r = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (r > S) return;
  const int64_t i = sub_indptr[r];
  if (i >= m.n) {
    out_indptr[r] = m.tile_base[m.tiles];  // (-1 when an id lay outside)
    return;
  }
  const int64_t w = i >> 6;
  const unsigned long long below = m.mask[w] & ((1ull << (i & 63)) - 1ull);
  out_indptr[r] = m.tile_base[i >> kTileShift] + m.word_rank[w] + __popcll(below);
}

// Every tile's kept edges from the front of its range to their place in the result, a wave at a
// time: eight times 64, all reads before the stores.  The data come from the parent, word by word.
constexpr int kCopyTiles = 4;  // of a workgroup, one for every wave
// Up to so many kept edges of a tile are a lane each, whatever their words: 40 M positions in columns of 600, 32-bit ids,
// 4 and 8 % kept, word by word 202 and 219 us, so 191 and 204 (192, three of a lane: the same).
constexpr int kFewKept = kWave;

template <typename IdT, Data DATA, bool STREAM>
__global__ void __launch_bounds__(256)
induced_compact_kernel(InducedMarks m, const int64_t* __restrict__ indptr, const IdT* __restrict__ cols,
                       const int64_t* __restrict__ sub_indptr, const float* __restrict__ data,
                       const int64_t* __restrict__ e_ids, IdT* __restrict__ out_indices,
                       float* __restrict__ out_data) {
  constexpr bool kParent = DATA == kByPosition || DATA == kByEdgeId;
  // kept positions of a tile's words of several columns (or of all), and above them the places of their data in the tile
  __shared__ uint32_t s_kept[kParent ? kCopyTiles : 1][kTile];
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);  // (a scalar, and so are all addresses' bases)
  const int64_t t = static_cast<int64_t>(blockIdx.x) * kCopyTiles + wave;
  if (t >= m.tiles) return;
  const int64_t base = m.tile_base[t];
  const int count = static_cast<int>(m.tile_base[t + 1] - base);
  unsigned long long my_word = 0;  // lane k: word k of the tile
  int my_rank = 0;
  int64_t my_at = 0;
  if (kParent && lane < kPer && t * kTile + lane * kWave < m.n) {
    my_word = m.mask[t * kPer + lane];
    my_rank = m.word_rank[t * kPer + lane];
    my_at = m.word_at[t * kPer + lane];
  }
  if (count == 0) return;
  auto once = [](const auto* p) { return STREAM ? __builtin_nontemporal_load(p) : *p; };
  uint16_t v[kPer];
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int r = k * kWave + lane;
    v[k] = m.packed[t * kTile + (r < count ? r : count - 1)];
  }
  auto put_indices = [&] {
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      const int r = k * kWave + lane;
      if (r < count) {
        if (STREAM)
          __builtin_nontemporal_store(static_cast<IdT>(v[k]), out_indices + base + r);
        else
          out_indices[base + r] = static_cast<IdT>(v[k]);
      }
    }
  };
  auto put_datum = [&](float datum, int r) {
    if (STREAM)
      __builtin_nontemporal_store(datum, out_data + base + r);
    else
      out_data[base + r] = datum;
  };
  auto of = [](uint64_t u, int k) {  // lane k's
    return static_cast<uint64_t>(static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(u >> 32), k))) << 32 |
           static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(u), k));
  };
  auto set_before = [](uint64_t word) {
    return static_cast<int>(__builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(word >> 32),
                                                      __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(word), 0)));
  };
  if constexpr (kParent) {
    const bool of_several = my_word && !WordAt::one(my_at);
    const uint64_t several_words = __ballot(of_several);
    const bool few = count <= kFewKept;
    if (several_words || few) {
      // Kept edge by kept edge, so that a column is looked for where an edge is kept, and three of a lane's together, so
      // that they are the same few trips.
      int most = of_several ? static_cast<int>(WordAt::more(my_at)) : 0;
#pragma unroll
      for (int d = 1; d < kPer; d <<= 1) {
        const int other = __shfl_xor(most, d, kWave);
        most = most > other ? most : other;
      }
      most = __builtin_amdgcn_readfirstlane(most);
      uint32_t* kept_at = s_kept[wave];
      int listed = 0;
#pragma unroll
      for (int k = 0; k < kPer; ++k) {
        if (!few && !(several_words >> k & 1u)) continue;
        const uint64_t word = of(my_word, k);
        const int before = set_before(word);
        if (word >> lane & 1u)
          kept_at[listed + before] =
              static_cast<uint32_t>(__builtin_amdgcn_readlane(my_rank, k) + before) << 16 | (k * kWave + lane);
        listed += __popcll(word);
      }
      __builtin_amdgcn_wave_barrier();
      auto some = [&](int r0, auto how_many) {
        constexpr int N = decltype(how_many)::value;
        int64_t at[N], end[N], start[N];
        int lo[N], hi[N], r[N];
        bool one[N];
#pragma unroll
        for (int u = 0; u < N; ++u) {
          const int j = r0 + u * kWave + lane;
          const uint32_t kept_one = kept_at[j < listed ? j : listed - 1];
          const int p = static_cast<int>(kept_one & 0xFFFFu);
          const int64_t where = __shfl(my_at, p / kWave, kWave);
          r[u] = static_cast<int>(kept_one >> 16);
          at[u] = t * kTile + p;
          one[u] = WordAt::one(where);
          lo[u] = static_cast<int>(WordAt::first(where));
          hi[u] = lo[u] + static_cast<int>(WordAt::more(where));
          if (one[u]) {
            at[u] = where + (p & (kWave - 1));
            lo[u] = hi[u] = 0;
          }
        }
        if (several_words) {
          for (int left = most; left; left >>= 1) {
#pragma unroll
            for (int u = 0; u < N; ++u) end[u] = sub_indptr[lo[u] + ((hi[u] - lo[u]) >> 1) + 1];
#pragma unroll
            for (int u = 0; u < N; ++u) {
              const int mid = lo[u] + ((hi[u] - lo[u]) >> 1);
              if (lo[u] < hi[u]) {
                if (end[u] > at[u]) hi[u] = mid; else lo[u] = mid + 1;
              }
            }
          }
#pragma unroll
          for (int u = 0; u < N; ++u) {
            start[u] = static_cast<int64_t>(cols[lo[u]]);
            end[u] = sub_indptr[lo[u]];
          }
#pragma unroll
          for (int u = 0; u < N; ++u) start[u] = indptr[one[u] ? 0 : start[u]];
#pragma unroll
          for (int u = 0; u < N; ++u)
            if (!one[u]) at[u] += start[u] - end[u];
        }
        if constexpr (DATA == kByEdgeId) {
#pragma unroll
          for (int u = 0; u < N; ++u) at[u] = once(e_ids + at[u]);
        }
        float datum[N];
#pragma unroll
        for (int u = 0; u < N; ++u) datum[u] = once(data + at[u]);
#pragma unroll
        for (int u = 0; u < N; ++u)
          if (r0 + u * kWave + lane < listed) put_datum(datum[u], r[u]);
      };
      if (listed <= kWave) {
        some(0, std::integral_constant<int, 1>());
      } else {
        for (int r0 = 0; r0 < listed; r0 += 3 * kWave) some(r0, std::integral_constant<int, 3>());
      }
      if (listed == count) {
        put_indices();
        return;
      }
      if (of_several) my_word = 0;  // (the others' edges below)
    }
  }
  bool kept[kParent ? kPer : 1];
  int rank[kParent ? kPer : 1];
  float x[DATA == kNoData ? 1 : kPer];
  if constexpr (DATA == kPacked) {
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      const int r = k * kWave + lane;
      x[k] = m.packed_data[t * kTile + (r < count ? r : count - 1)];
    }
  }
  if constexpr (kParent) {
    int64_t at[kPer];
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      const uint64_t word = of(my_word, k);
      const int64_t where = static_cast<int64_t>(of(static_cast<uint64_t>(my_at), k));
      kept[k] = word >> lane & 1u;
      rank[k] = __builtin_amdgcn_readlane(my_rank, k) + set_before(word);
      // (lanes whose edge is left out read with the word's first kept one, a word without any the first datum: behind
      // the last position there is no edge)
      const int place = kept[k] ? lane : (word ? __builtin_ctzll(word) : 0);
      at[k] = word ? where + place : 0;
    }
    if constexpr (DATA == kByEdgeId) {
#pragma unroll
      for (int k = 0; k < kPer; ++k) at[k] = once(e_ids + at[k]);
    }
#pragma unroll
    for (int k = 0; k < kPer; ++k) x[k] = once(data + at[k]);
  }
  put_indices();
  if constexpr (DATA == kPacked) {
#pragma unroll
    for (int k = 0; k < kPer; ++k)
      if (k * kWave + lane < count) put_datum(x[k], k * kWave + lane);
  }
  if constexpr (kParent) {
#pragma unroll
    for (int k = 0; k < kPer; ++k)
      if (kept[k]) put_datum(x[k], rank[k]);
  }
}

// Whether the marks read the data and pack them beside the row numbers, or the copy reads the kept edges' from the
// parent.  The first is 8 bytes more of every kept edge, the second a wave's trips to memory one behind the other, and to
// the offsets too where columns are short.  The whole call, the marks / the copy, us, 40 M positions, 32-bit ids, 8000 of
// 1 M nodes in the set, 4 % kept by chance, and 64-bit ids of 0.4 M, 10, 50 and 90 % kept:
//   positions / columns  64 431/455, 360/401, 415/500, 487/573    130 357/380, 267/297, 329/375, 403/436
//                       300 328/351, 221/235, 279/299, 355/345    600 284/304, 200/210, 264/267, 336/313
//                      4000 238/252, 177/178, 239/241, 312/287    and 500 of 0.2 M nodes, 139/122
// and 7263 nodes with columns of 7000, 50.8 M, 43 % kept: 185 + 85 / 130 + 114 us (1142 / 967 MB).
inline bool marks_read_data(int64_t S, int64_t D) { return D < kLongColumns * S; }

// in_marks: with data, who reads them
size_t induced_bytes(int64_t D, bool with_data, bool in_marks) {
  if (D < 1) D = 1;
  const size_t words = static_cast<size_t>(D / kWave + 1), n = static_cast<size_t>(D);
  const int64_t tiles = ((D - 1) >> kTileShift) + 1;
  return padded(words * 8) + padded(words * 4) + padded(static_cast<size_t>(tiles + 1) * 8) +
         padded(static_cast<size_t>(tiles + 2) * 8) + lookback_state_bytes(scan_num_tiles(tiles)) + 256 +
         padded(n * 2) + (with_data ? (in_marks ? padded(n * 4) : padded(words * 8)) : 0);
}

bool carve_induced(void* workspace, size_t bytes, int64_t D, bool with_data, bool in_marks, InducedMarks* m) {
  Carver ws(workspace, bytes);
  const size_t words = static_cast<size_t>(D / kWave + 1);
  const size_t most = static_cast<size_t>(((D - 1) >> kTileShift) + 1);
  m->n = D;
  m->tiles = static_cast<int64_t>(most);
  m->mask = ws.take<unsigned long long>(words);
  m->word_rank = ws.take<int32_t>(words);
  m->tile_counts = ws.take<int64_t>(most + 1);
  m->tile_base = ws.take<int64_t>(most + 2);
  m->lb_tiles = scan_num_tiles(m->tiles);
  m->lb = carve_lookback(ws, m->lb_tiles, 1u);
  m->outside = ws.take<int>(1);
  m->packed = ws.take<uint16_t>(static_cast<size_t>(D));
  m->word_at = with_data && !in_marks ? ws.take<int64_t>(words) : nullptr;
  m->packed_data = with_data && in_marks ? ws.take<float>(static_cast<size_t>(D)) : nullptr;
  return ws.ok;
}

struct MarkCall {
  const int64_t* indptr;
  int64_t num_cols;
  const void *indices, *cols;
  int64_t S;
  const int64_t* sub_indptr;
  int64_t D;
  const void* ids;
  int64_t n_ids, bound;
  const float* data;
  const int64_t* e_ids;
  bool in_marks;
};

// Whether the ids and data of D positions are more than the 256 MB that the memory-side cache holds.
// The whole call (walk, unique nodes and subgraph), plain / streamed, with the data read by the marks: 50.8 M positions
// with 64-bit ids and data (610 MB) 398-412 / 383-394 us;
// graphs of 100 M edges, 1.5 M nodes and of 50 M, 0.2 M, a few hundred seeds, 32-bit ids 217 / 216, 157 / 159.
inline bool streams(int64_t D, size_t id_bytes, bool with_data) {
  return D * static_cast<int64_t>(id_bytes + (with_data ? 4 : 0)) >= int64_t(1) << 28;
}

template <typename IdT, typename Set, int BLOCK, Data DATA>
int launch_mark(const MarkCall& c, int per_unit, const InducedMarks& m, hipStream_t st) {
  auto* kernel = streams(c.D, sizeof(IdT), DATA != kNoData) ? induced_mark_kernel<IdT, Set, BLOCK, DATA, true>
                                                            : induced_mark_kernel<IdT, Set, BLOCK, DATA, false>;
  const size_t bytes = Set::lds_bytes(c.bound, c.n_ids);
  // (per call: the attribute belongs to the device the call runs on)
  if (hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                          hipFuncAttributeMaxDynamicSharedMemorySize,
                          static_cast<int>(bytes)) != hipSuccess) {
    set_error_text("gs_induced_slice_mark: %s", hipGetErrorString(hipGetLastError()));
    return GS_ERR_LAUNCH;
  }
  const int64_t runs = (m.tiles + BLOCK / kWave - 1) / (BLOCK / kWave), most = int64_t(kUnits) * per_unit;
  hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(runs < most ? runs : most)),
                     dim3(BLOCK), bytes, st, c.indptr, c.num_cols, static_cast<const IdT*>(c.indices),
                     static_cast<const IdT*>(c.cols), c.S, c.sub_indptr, c.D,
                     static_cast<const IdT*>(c.ids), static_cast<int>(c.n_ids), c.bound, c.data,
                     c.e_ids, m);
  return check_launch("induced_slice_mark");
}

template <typename IdT, typename Set, int BLOCK>
int launch_mark(const MarkCall& c, int per_unit, const InducedMarks& m, hipStream_t st) {
  if (!c.data) return launch_mark<IdT, Set, BLOCK, kNoData>(c, per_unit, m, st);
  if (!c.in_marks) return launch_mark<IdT, Set, BLOCK, kPlaces>(c, per_unit, m, st);
  if (!c.e_ids) return launch_mark<IdT, Set, BLOCK, kByPosition>(c, per_unit, m, st);
  return launch_mark<IdT, Set, BLOCK, kByEdgeId>(c, per_unit, m, st);
}

// LDS that the kernel declares itself
constexpr size_t fixed_lds(int block) {
  return static_cast<size_t>(block / kWave) * ((2 * kWindow + 1) * 8 + 8) + 256;
}

// Which form of the set: the bitmap when it fits, as two workgroups of 512 lanes a compute unit
// when two of them fit, as one of 1024 lanes otherwise; else the buckets.
template <typename IdT>
int pick_mark(const MarkCall& c, const InducedMarks& m, hipStream_t st) {
  const size_t bitmap = BitmapSet<IdT>::lds_bytes(c.bound, c.n_ids);
  if (2 * (bitmap + fixed_lds(512)) <= kLdsBytes)
    return launch_mark<IdT, BitmapSet<IdT>, 512>(c, 2, m, st);
  if (bitmap + fixed_lds(1024) <= kLdsBytes)
    return launch_mark<IdT, BitmapSet<IdT>, 1024>(c, 1, m, st);
  static_assert(size_t(1 << 13) * 16 + fixed_lds(1024) <= kLdsBytes, "buckets");
  if (c.n_ids <= kStagedIds) return launch_mark<IdT, BucketSet<IdT, true>, 1024>(c, 1, m, st);
  return launch_mark<IdT, BucketSet<IdT, false>, 1024>(c, 1, m, st);
}

template <typename IdT>
void launch_compact(int64_t D, const InducedMarks& m, const int64_t* indptr, const void* cols,
                    const int64_t* sub_indptr, const float* data, const int64_t* e_ids, IdT* out_indices,
                    float* out_data, hipStream_t st) {
  const bool packed = !data && out_data;
  const bool past = streams(D, sizeof(IdT), data || packed);
  auto* kernel = packed   ? (past ? induced_compact_kernel<IdT, kPacked, true> : induced_compact_kernel<IdT, kPacked, false>)
                 : !data  ? (past ? induced_compact_kernel<IdT, kNoData, true> : induced_compact_kernel<IdT, kNoData, false>)
                 : !e_ids ? (past ? induced_compact_kernel<IdT, kByPosition, true>
                                  : induced_compact_kernel<IdT, kByPosition, false>)
                          : (past ? induced_compact_kernel<IdT, kByEdgeId, true>
                                  : induced_compact_kernel<IdT, kByEdgeId, false>);
  hipLaunchKernelGGL(kernel, dim3(blocks_for(m.tiles, kCopyTiles)), dim3(256), 0, st, m, indptr,
                     static_cast<const IdT*>(cols), sub_indptr, data, e_ids, out_indices, out_data);
}

}  // namespace
}  // namespace gs

using namespace gs;

extern "C" {

// An id set that fits one compute unit's LDS; enough positions for every compute unit to earn the
// building of its copy of the set back; columns that are not all short (the positions of a tile are
// resolved among a handful of staged offsets).  The whole call in us, general slice / this one, 64-bit
// ids, 8000 of them, of graphs of 200 k nodes (a bit per node) and 1 M (buckets), with the edges' data:
//   positions / columns      16       32       64       256           16       32       64       256
//   1 M positions         74/58    77/56    69/52    65/45         76/72    72/72    71/65    66/57
//   2 M                   82/63    79/62    76/58    72/49         82/76    81/71    78/68    75/64
//   8 M                  159/116  157/112  154/93   151/70        163/150  158/152  154/131  145/101
// and of 1000 ids, 1 M and 8 M, 72/52 159/109, 68/51 154/105, 71/46 151/86, 63/40 147/62; 72/54 160/116, 69/53 149/107,
// 68/48 145/88, 67/40 124/66: nothing is lost with either form on this side of the lines.  nnz does not matter.
int gs_induced_slice_applies(int64_t num_row_ids, int64_t S, int64_t D, int64_t) {
  return num_row_ids > 0 && num_row_ids <= kMaxIds && S > 0 && S < (int64_t(1) << 31) && D >= (int64_t(1) << 20) && D >= 16 * S;
}

size_t gs_induced_slice_notify_workspace_bytes(int64_t S, int64_t D, int with_data) {
  return induced_bytes(D, with_data != 0, marks_read_data(S, D));
}

size_t gs_induced_slice_workspace_bytes(int64_t D, int with_data) { return induced_bytes(D, with_data != 0, true); }

static int induced_mark(const int64_t* indptr, int64_t num_cols, const void* indices, int64_t nnz, int64_t num_rows,
                        int id_bytes, const void* column_ids, int64_t S, const int64_t* sub_indptr, int64_t D,
                        const void* row_ids, int64_t num_row_ids, const float* edge_data, const int64_t* edge_ids,
                        bool in_marks, int64_t* out_indptr, gs_mailbox* mailbox, int64_t ticket, void* workspace,
                        size_t workspace_bytes, void* stream) {
  GS_REQUIRE(gs_induced_slice_applies(num_row_ids, S, D, nnz) && num_rows >= 0,
             "gs_induced_slice_mark: sizes beyond gs_induced_slice_applies");
  GS_REQUIRE(indptr && indices && column_ids && sub_indptr && row_ids && out_indptr,
             "gs_induced_slice_mark: null pointer");
  GS_REQUIRE(valid_id_bytes(id_bytes), "gs_induced_slice_mark: id_bytes must be 4 or 8, got %d",
             id_bytes);
  InducedMarks m;
  if (!carve_induced(workspace, workspace_bytes, D, edge_data != nullptr, in_marks, &m)) {
    set_error_text("gs_induced_slice_mark: workspace needs %zu bytes, 256-byte aligned",
                   induced_bytes(D, edge_data != nullptr, in_marks));
    return GS_ERR_WORKSPACE;
  }
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int64_t bound = num_rows > 0 ? num_rows : int64_t(1) << 40;  // (no bound given: no bitmap)
  const MarkCall c{indptr, num_cols, indices, column_ids, S, sub_indptr, D, row_ids, num_row_ids,
                   bound, edge_data, edge_ids, in_marks};
  GS_RETURN_IF_ERROR(id_bytes == 8 ? pick_mark<int64_t>(c, m, st) : pick_mark<int32_t>(c, m, st));
  TileCount f{m.tile_counts};
  GS_RETURN_IF_ERROR(chained_scan(f, m.tiles, m.tile_base, m.lb, st, mailbox, ticket, m.outside));
  hipLaunchKernelGGL(induced_indptr_kernel, dim3(blocks_for(S + 1, 256)), dim3(256), 0, st,
                     sub_indptr, S, m, out_indptr);
  return check_launch("induced_slice_mark");
}

int gs_induced_slice_mark(const int64_t* indptr, int64_t num_cols, const void* indices, int64_t nnz,
                          int64_t num_rows, int id_bytes, const void* column_ids, int64_t S,
                          const int64_t* sub_indptr, int64_t D, const void* row_ids,
                          int64_t num_row_ids, const float* edge_data, const int64_t* edge_ids,
                          int64_t* out_indptr, void* workspace, size_t workspace_bytes,
                          void* stream) {
  return induced_mark(indptr, num_cols, indices, nnz, num_rows, id_bytes, column_ids, S, sub_indptr, D, row_ids,
                      num_row_ids, edge_data, edge_ids, true, out_indptr, nullptr, 0, workspace, workspace_bytes, stream);
}

int gs_induced_slice_mark_notify(const int64_t* indptr, int64_t num_cols, const void* indices, int64_t nnz,
                                 int64_t num_rows, int id_bytes, const void* column_ids, int64_t S,
                                 const int64_t* sub_indptr, int64_t D, const void* row_ids,
                                 int64_t num_row_ids, const float* edge_data, const int64_t* edge_ids,
                                 int64_t* out_indptr, gs_mailbox* mailbox, int64_t ticket, void* workspace,
                                 size_t workspace_bytes, void* stream) {
  return induced_mark(indptr, num_cols, indices, nnz, num_rows, id_bytes, column_ids, S, sub_indptr, D, row_ids,
                      num_row_ids, edge_data, edge_ids, marks_read_data(S, D), out_indptr, mailbox, ticket, workspace,
                      workspace_bytes, stream);
}

static int induced_compact(const int64_t* indptr, int id_bytes, const void* column_ids, const int64_t* sub_indptr,
                           int64_t D, const float* edge_data, const int64_t* edge_ids, bool in_marks, void* out_indices,
                           float* out_data, void* workspace, size_t workspace_bytes, void* stream) {
  GS_REQUIRE(valid_id_bytes(id_bytes), "gs_induced_slice_compact: id_bytes must be 4 or 8, got %d",
             id_bytes);
  InducedMarks m;
  if (!carve_induced(workspace, workspace_bytes, D, out_data != nullptr, in_marks, &m)) {
    set_error_text("gs_induced_slice_compact: pass the workspace given to gs_induced_slice_mark");
    return GS_ERR_WORKSPACE;
  }
  if (in_marks) edge_data = nullptr;  // (they lie packed)
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (id_bytes == 8)
    launch_compact(D, m, indptr, column_ids, sub_indptr, edge_data, edge_ids,
                   static_cast<int64_t*>(out_indices), out_data, st);
  else
    launch_compact(D, m, indptr, column_ids, sub_indptr, edge_data, edge_ids,
                   static_cast<int32_t*>(out_indices), out_data, st);
  return check_launch("induced_slice_compact");
}

int gs_induced_slice_compact(int64_t D, int id_bytes, void* out_indices, float* out_data,
                             void* workspace, size_t workspace_bytes, void* stream) {
  GS_REQUIRE(D > 0 && out_indices, "gs_induced_slice_compact: bad argument");
  return induced_compact(nullptr, id_bytes, nullptr, nullptr, D, nullptr, nullptr, true, out_indices, out_data,
                         workspace, workspace_bytes, stream);
}

int gs_induced_slice_compact_parent(const int64_t* indptr, int id_bytes, const void* column_ids, int64_t S,
                                    const int64_t* sub_indptr, int64_t D, const float* edge_data,
                                    const int64_t* edge_ids, void* out_indices, float* out_data,
                                    void* workspace, size_t workspace_bytes, void* stream) {
  GS_REQUIRE(D > 0 && out_indices && indptr && column_ids && sub_indptr, "gs_induced_slice_compact: bad argument");
  GS_REQUIRE(!edge_data == !out_data, "gs_induced_slice_compact: data without a place for them, or the other way round");
  return induced_compact(indptr, id_bytes, column_ids, sub_indptr, D, edge_data, edge_ids, marks_read_data(S, D),
                         out_indices, out_data, workspace, workspace_bytes, stream);
}

}  // extern "C"
