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
//     positions touch (with long columns: no search at all);
//   * the ids (and data) of the NEXT tile are asked for before this tile's are looked up, since
//     the few waves beside the set have little else to hide that latency behind;
//   * kept edges leave one bit each and, packed to the front of the tile's range of a scratch
//     array, their new row number in 2 bytes and their datum.
// A scan of the tile counts and one copy kernel put the pieces together.  (With the tiles shared
// by the waves of a workgroup, offsets and counts through LDS and two barriers a tile, the marks
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
// What bounds the bitmap form: the LDS look-ups and the vector ALUs beside 750 MB in 184 us in the case below,
// 4.1 TB/s (reads that are truly a tile ahead: 183); more waves than the set leaves room for would be needed to
// overlap the two better.  7263 nodes whose columns hold 50.8 M edges, 22.0 M kept, 64-bit ids
// and weights: 184 us for the marks and 71-84 us for the copy (new row numbers in 4 bytes and nothing
// streamed: 225 + 70), where a filter and a table in the
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

struct InducedMarks {
  unsigned long long* mask;  // one bit per position
  int32_t* word_rank;        // kept positions of the tile before each 64-position word
  int64_t* tile_counts;
  int64_t* tile_base;        // exclusive scan of tile_counts
  uint16_t* packed;          // new row numbers (places, 14 bits) of the kept edges, at the front of the tile's range
  float* packed_data;        // their data (null: none)
  int* outside;              // set when an id lies beyond the bitmap: the call has to be repeated
  int64_t n;
  int64_t tiles;
};

// A bit per node number below `bound`.
template <typename IdT>
struct BitmapSet {
  uint32_t* bits;
  uint16_t* before;  // set bits before each word
  uint32_t* place;   // two to a word: place of the id of every set bit
  uint32_t bound;

  static size_t lds_bytes(int64_t bound, int64_t n_ids) {
    const size_t words = static_cast<size_t>(bound + 31) / 32;
    return (words * 4 + 15) / 16 * 16 + (words * 2 + 15) / 16 * 16 +
           (static_cast<size_t>(n_ids) * 2 + 15) / 16 * 16;
  }
  __device__ __forceinline__ char* carve(char* lds, int64_t bound_, int n_ids) {
    const size_t words = static_cast<size_t>(bound_ + 31) / 32;
    bound = static_cast<uint32_t>(bound_);
    bits = reinterpret_cast<uint32_t*>(lds);
    lds += (words * 4 + 15) / 16 * 16;
    before = reinterpret_cast<uint16_t*>(lds);
    lds += (words * 2 + 15) / 16 * 16;
    place = reinterpret_cast<uint32_t*>(lds);
    return lds + (static_cast<size_t>(n_ids) * 2 + 15) / 16 * 16;
  }
  __device__ __forceinline__ uint32_t rank(uint32_t id) const {
    return before[id >> 5] + __popc(bits[id >> 5] & ((1u << (id & 31)) - 1u));
  }
  // every lane of the workgroup; s_scan: BLOCK / 64 + 1 words
  template <int BLOCK>
  __device__ __forceinline__ void build(const IdT* __restrict__ ids, int n_ids, int64_t* s_scan,
                                        int* outside) {
    const int words = static_cast<int>((bound + 31) / 32);
    for (int j = threadIdx.x; j < words; j += BLOCK) bits[j] = 0;
    for (int j = threadIdx.x; j < (n_ids + 1) / 2; j += BLOCK) place[j] = 0;
    if (blockIdx.x == 0 && threadIdx.x == 0) *outside = 0;
    __syncthreads();
    for (int j = threadIdx.x; j < n_ids; j += BLOCK) {
      const uint64_t id = static_cast<uint64_t>(static_cast<int64_t>(ids[j]));
      if (id < bound)
        atomicOr(&bits[id >> 5], 1u << (id & 31));
      else if (blockIdx.x == 0)
        *outside = 1;
    }
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
    for (int j = threadIdx.x; j < n_ids; j += BLOCK) {
      const uint64_t id = static_cast<uint64_t>(static_cast<int64_t>(ids[j]));
      if (id >= bound) continue;
      const uint32_t r = rank(static_cast<uint32_t>(id));
      const int shift = (r & 1) * 16;
      uint32_t was = place[r >> 1];
      // the same id twice: its last place counts
      while (((was >> shift) & 0xFFFFu) < static_cast<uint32_t>(j)) {
        const uint32_t now = (was & ~(0xFFFFu << shift)) | (static_cast<uint32_t>(j) << shift);
        const uint32_t seen = atomicCAS(&place[r >> 1], was, now);
        if (seen == was) break;
        was = seen;
      }
    }
    __syncthreads();
  }
  // val[k] = place of id[k], -1 when it is not in the set
  __device__ __forceinline__ void lookup(const IdT (&id)[kPer], int (&val)[kPer]) const {
    uint32_t at[kPer], w[kPer];
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      const uint64_t v = static_cast<uint64_t>(static_cast<int64_t>(id[k]));
      at[k] = v < bound ? static_cast<uint32_t>(v) : 0u;
      w[k] = bits[at[k] >> 5];
      if (v >= bound) w[k] = 0;
    }
    uint32_t r[kPer];
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      const uint32_t bit = 1u << (at[k] & 31);
      r[k] = before[at[k] >> 5] + __popc(w[k] & (bit - 1u));
      val[k] = w[k] & bit ? 0 : -1;
      if (val[k]) r[k] = 0;
    }
    const uint16_t* half = reinterpret_cast<const uint16_t*>(place);
#pragma unroll
    for (int k = 0; k < kPer; ++k) val[k] |= half[r[k]];
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
    if (STAGED)
      for (int j = threadIdx.x; j < n_ids; j += BLOCK) s_ids[j] = list[j];
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
  __device__ __forceinline__ void lookup(const IdT (&id)[kPer], int (&val)[kPer]) const {
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

// What a wave's edges bring along: nothing, data[position], or data[e_ids[position]].
enum Data { kNoData, kByPosition, kByEdgeId };

template <typename IdT, typename Set, int BLOCK, Data DATA, bool STREAM>
__global__ void __launch_bounds__(BLOCK, 4)  // (16 waves a compute unit: what the set leaves room for)
induced_mark_kernel(const int64_t* __restrict__ indptr, int64_t num_cols,
                    const IdT* __restrict__ indices, const IdT* __restrict__ cols, int64_t S,
                    const int64_t* __restrict__ sub_indptr, int64_t D, const IdT* __restrict__ ids,
                    int n_ids, int64_t bound, const float* __restrict__ data,
                    const int64_t* __restrict__ e_ids, int64_t tiles_each, InducedMarks m) {
  __shared__ int64_t s_offsets[BLOCK / kWave][kWindow + 1];
  __shared__ int64_t s_starts[BLOCK / kWave][kWindow];  // start of the column minus its offset
  __shared__ int64_t s_scan[BLOCK / kWave + 1];
  extern __shared__ __align__(16) char lds[];
  Set set;
  set.carve(lds, bound, n_ids);
  set.template build<BLOCK>(ids, n_ids, s_scan, m.outside);

  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  constexpr int kStep = BLOCK / kWave;  // the waves of a workgroup take turns along its run
  const int64_t run = static_cast<int64_t>(blockIdx.x) * kStep * tiles_each;
  const int64_t tile0 = run + wave;
  const int64_t tile1 = run + kStep * tiles_each < m.tiles ? run + kStep * tiles_each : m.tiles;
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

  // where the 64 positions from q on lie in the parent (q never decreases)
  auto locate = [&](int64_t q) -> int64_t {
    const int64_t last = (q + kWave < D ? q + kWave : D) - 1;
    int64_t p = q + lane;
    p = p < last ? p : last;
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
      return indptr[static_cast<int64_t>(cols[lo])] + p - sub_indptr[lo];
    }
    if (off[row + 1] <= q) row = row_of(off, row + 1, kWindow - 1, q);
    row_end = uniform(off[row + 1]);
    row_start = uniform(start[row]);
    if (last < row_end) return row_start + p;
    const int r = row_of(off, row, kWindow - 1, p);
    return start[r] + p;
  };

  struct Held {
    IdT id[kPer];
    float w[DATA == kByPosition ? kPer : 1];
    int64_t e[DATA == kByEdgeId ? kPer : 1];
  };
  // (STREAM: beyond the caches' size what a call reads is gone from them before anyone reads it again)
  auto once = [](const auto* p) { return STREAM ? __builtin_nontemporal_load(p) : *p; };
  auto fetch = [&](int64_t t, Held& h) {
    int64_t at[kPer];
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      const int64_t q = t * kTile + k * kWave;
      at[k] = locate(q < D ? q : D - 1);
    }
#pragma unroll
    for (int k = 0; k < kPer; ++k) h.id[k] = once(indices + at[k]);
    // (the data of all: 64 neighbours share their lines with the kept ones among them)
    if constexpr (DATA == kByPosition) {
#pragma unroll
      for (int k = 0; k < kPer; ++k) h.w[k] = once(data + at[k]);
    }
    if constexpr (DATA == kByEdgeId) {
#pragma unroll
      for (int k = 0; k < kPer; ++k) h.e[k] = once(e_ids + at[k]);
    }
  };

  Held now, next;
  stage(wave_upper_bound(sub_indptr, S + 1, tile0 * kTile) - 1);
  fetch(tile0, now);
  for (int64_t t = tile0; t < tile1; t += kStep) {
    if (t + kStep < tile1) fetch(t + kStep, next);
    const int64_t p0 = t * kTile;
    int val[kPer];
    set.lookup(now.id, val);
    if (p0 + kTile > D) {
#pragma unroll
      for (int k = 0; k < kPer; ++k)
        if (p0 + k * kWave + lane >= D) val[k] = -1;
    }
    float w[DATA == kNoData ? 1 : kPer];
    if constexpr (DATA == kByEdgeId) {
#pragma unroll
      for (int k = 0; k < kPer; ++k) w[k] = val[k] >= 0 ? data[now.e[k]] : 0.0f;
    }
    int before = 0, my_before = 0;
    unsigned long long my_word = 0;
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      const unsigned long long kept = __ballot(val[k] >= 0);
      if (lane == k) {
        my_word = kept;
        my_before = before;
      }
      const int rank = before + __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(kept >> 32),
                                                          __builtin_amdgcn_mbcnt_lo(
                                                              static_cast<uint32_t>(kept), 0));
      before += __popcll(kept);
      if (val[k] >= 0) {
        m.packed[p0 + rank] = static_cast<uint16_t>(val[k]);
        if constexpr (DATA == kByPosition) m.packed_data[p0 + rank] = now.w[k];
        if constexpr (DATA == kByEdgeId) m.packed_data[p0 + rank] = w[k];
      }
    }
    if (lane < kPer && p0 + lane * kWave < D) {
      m.mask[(p0 >> 6) + lane] = my_word;
      m.word_rank[(p0 >> 6) + lane] = my_before;
    }
    if (lane == 0) m.tile_counts[t] = before;
    now = next;
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
    out_indptr[r] = r == S && *m.outside ? int64_t(-1) : m.tile_base[m.tiles];
    return;
  }
  const int64_t w = i >> 6;
  const unsigned long long below = m.mask[w] & ((1ull << (i & 63)) - 1ull);
  out_indptr[r] = m.tile_base[i >> kTileShift] + m.word_rank[w] + __popcll(below);
}

// Every tile's kept edges from the front of its range to their place in the result, a wave at a
// time: eight times 64, all reads before the stores.
constexpr int kCopyTiles = 4;  // of a workgroup, one for every wave

template <typename IdT, bool STREAM>
__global__ void __launch_bounds__(256)
induced_compact_kernel(InducedMarks m, IdT* __restrict__ out_indices, float* __restrict__ out_data) {
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  const int64_t t = static_cast<int64_t>(blockIdx.x) * kCopyTiles + wave;
  if (t >= m.tiles) return;
  const int64_t base = m.tile_base[t];
  const int count = static_cast<int>(m.tile_base[t + 1] - base);
  if (count == 0) return;
  uint16_t v[kPer];
  float x[kPer];
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int r = k * kWave + lane;
    v[k] = m.packed[t * kTile + (r < count ? r : count - 1)];
  }
  if (out_data) {
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      const int r = k * kWave + lane;
      x[k] = m.packed_data[t * kTile + (r < count ? r : count - 1)];
    }
  }
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int r = k * kWave + lane;
    if (r < count) {
      if (STREAM) {
        __builtin_nontemporal_store(static_cast<IdT>(v[k]), out_indices + base + r);
        if (out_data) __builtin_nontemporal_store(x[k], out_data + base + r);
      } else {
        out_indices[base + r] = static_cast<IdT>(v[k]);
        if (out_data) out_data[base + r] = x[k];
      }
    }
  }
}

bool carve_induced(void* workspace, size_t bytes, int64_t D, bool with_data, InducedMarks* m,
                   int64_t** scan_tiles) {
  Carver ws(workspace, bytes);
  const size_t words = static_cast<size_t>(D / kWave + 1);
  const size_t most = static_cast<size_t>(((D - 1) >> kTileShift) + 1);
  m->n = D;
  m->tiles = static_cast<int64_t>(most);
  m->mask = ws.take<unsigned long long>(words);
  m->word_rank = ws.take<int32_t>(words);
  m->tile_counts = ws.take<int64_t>(most + 1);
  m->tile_base = ws.take<int64_t>(most + 2);
  *scan_tiles = ws.take<int64_t>(static_cast<size_t>(scan_num_tiles(m->tiles) + 1));
  m->outside = ws.take<int>(1);
  m->packed = ws.take<uint16_t>(static_cast<size_t>(D));
  m->packed_data = with_data ? ws.take<float>(static_cast<size_t>(D)) : nullptr;
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
};

// Whether the ids and data of D positions are more than the 256 MB that the memory-side cache holds.
// The whole call (walk, unique nodes and subgraph), plain / streamed: 50.8 M positions with 64-bit ids and data (610 MB)
// 398-412 / 383-394 us (marks 216 / 185, copy 67 / 84: who stores past the cache leaves it to the other);
// graphs of 100 M edges, 1.5 M nodes and of 50 M, 0.2 M, a few hundred seeds, 32-bit ids 217 / 216, 157 / 159.
inline bool streams(int64_t D, size_t id_bytes, bool with_data) {
  return D * static_cast<int64_t>(id_bytes + (with_data ? 4 : 0)) >= int64_t(1) << 28;
}

template <typename IdT, typename Set, int BLOCK, Data DATA>
int launch_mark(const MarkCall& c, int per_unit, const InducedMarks& m, hipStream_t st) {
  auto* kernel = streams(c.D, sizeof(IdT), DATA != kNoData)
                     ? induced_mark_kernel<IdT, Set, BLOCK, DATA, true>
                     : induced_mark_kernel<IdT, Set, BLOCK, DATA, false>;
  const size_t bytes = Set::lds_bytes(c.bound, c.n_ids);
  // (per call: the attribute belongs to the device the call runs on)
  if (hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                          hipFuncAttributeMaxDynamicSharedMemorySize,
                          static_cast<int>(bytes)) != hipSuccess) {
    set_error_text("gs_induced_slice_mark: %s", hipGetErrorString(hipGetLastError()));
    return GS_ERR_LAUNCH;
  }
  const int64_t waves = static_cast<int64_t>(kUnits) * per_unit * (BLOCK / kWave);
  const int64_t each = (m.tiles + waves - 1) / waves;
  hipLaunchKernelGGL(kernel, dim3(blocks_for(m.tiles, static_cast<int>(each * (BLOCK / kWave)))),
                     dim3(BLOCK), bytes, st, c.indptr, c.num_cols, static_cast<const IdT*>(c.indices),
                     static_cast<const IdT*>(c.cols), c.S, c.sub_indptr, c.D,
                     static_cast<const IdT*>(c.ids), static_cast<int>(c.n_ids), c.bound, c.data,
                     c.e_ids, each, m);
  return check_launch("induced_slice_mark");
}

template <typename IdT, typename Set, int BLOCK>
int launch_mark(const MarkCall& c, int per_unit, const InducedMarks& m, hipStream_t st) {
  if (!c.data) return launch_mark<IdT, Set, BLOCK, kNoData>(c, per_unit, m, st);
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

}  // namespace
}  // namespace gs

using namespace gs;

extern "C" {

// An id set that fits one compute unit's LDS; enough positions for every compute unit to earn the
// building of its copy of the set back; columns that are not all short (the positions of a tile are
// resolved among a handful of staged offsets).  The whole call in us, general slice / this one, 64-bit
// ids, of graphs of 200 k nodes (a bit per node) and 1 M (buckets), with the edges' data:
//   8000 ids, 0.5 M / 1 M / 2 M positions   78/68 80/69 86/75    78/85 81/79 87/83
//   1000 ids, 0.25 M / 1 M positions        67/49 70/50          75/52 68/51
//   positions / columns 4, 8, 12, 16, 32    94/89 94/94 97/96 98/92 93/91    93/93 89/88 88/85 87/89 87/82
// so the lines lie where nothing is lost with either form.  nnz does not matter.
int gs_induced_slice_applies(int64_t num_row_ids, int64_t S, int64_t D, int64_t) {
  return num_row_ids > 0 && num_row_ids <= kMaxIds && S > 0 && D >= (int64_t(1) << 20) && D >= 16 * S;
}

size_t gs_induced_slice_workspace_bytes(int64_t D, int with_data) {
  if (D < 1) D = 1;
  const size_t words = static_cast<size_t>(D / kWave + 1), n = static_cast<size_t>(D);
  const int64_t tiles = ((D - 1) >> kTileShift) + 1;
  return padded(words * 8) + padded(words * 4) + padded(static_cast<size_t>(tiles + 1) * 8) +
         padded(static_cast<size_t>(tiles + 2) * 8) + scan_workspace_bytes(tiles) + 256 +
         padded(n * 2) + (with_data ? padded(n * 4) : 0);
}

int gs_induced_slice_mark(const int64_t* indptr, int64_t num_cols, const void* indices, int64_t nnz,
                          int64_t num_rows, int id_bytes, const void* column_ids, int64_t S,
                          const int64_t* sub_indptr, int64_t D, const void* row_ids,
                          int64_t num_row_ids, const float* edge_data, const int64_t* edge_ids,
                          int64_t* out_indptr, void* workspace, size_t workspace_bytes,
                          void* stream) {
  GS_REQUIRE(gs_induced_slice_applies(num_row_ids, S, D, nnz) && num_rows >= 0,
             "gs_induced_slice_mark: sizes beyond gs_induced_slice_applies");
  GS_REQUIRE(indptr && indices && column_ids && sub_indptr && row_ids && out_indptr,
             "gs_induced_slice_mark: null pointer");
  GS_REQUIRE(valid_id_bytes(id_bytes), "gs_induced_slice_mark: id_bytes must be 4 or 8, got %d",
             id_bytes);
  InducedMarks m;
  int64_t* scan_tiles;
  if (!carve_induced(workspace, workspace_bytes, D, edge_data != nullptr, &m, &scan_tiles)) {
    set_error_text("gs_induced_slice_mark: workspace needs %zu bytes, 256-byte aligned",
                   gs_induced_slice_workspace_bytes(D, edge_data != nullptr));
    return GS_ERR_WORKSPACE;
  }
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int64_t bound = num_rows > 0 ? num_rows : int64_t(1) << 40;  // (no bound given: no bitmap)
  const MarkCall c{indptr, num_cols, indices, column_ids, S, sub_indptr, D, row_ids, num_row_ids,
                   bound, edge_data, edge_ids};
  GS_RETURN_IF_ERROR(id_bytes == 8 ? pick_mark<int64_t>(c, m, st) : pick_mark<int32_t>(c, m, st));
  TileCount f{m.tile_counts};
  GS_RETURN_IF_ERROR(exclusive_scan(f, m.tiles, m.tile_base, scan_tiles, st));
  hipLaunchKernelGGL(induced_indptr_kernel, dim3(blocks_for(S + 1, 256)), dim3(256), 0, st,
                     sub_indptr, S, m, out_indptr);
  return check_launch("induced_slice_mark");
}

int gs_induced_slice_compact(int64_t D, int id_bytes, void* out_indices, float* out_data,
                             void* workspace, size_t workspace_bytes, void* stream) {
  GS_REQUIRE(D > 0 && out_indices, "gs_induced_slice_compact: bad argument");
  GS_REQUIRE(valid_id_bytes(id_bytes), "gs_induced_slice_compact: id_bytes must be 4 or 8, got %d",
             id_bytes);
  InducedMarks m;
  int64_t* scan_tiles;
  if (!carve_induced(workspace, workspace_bytes, D, out_data != nullptr, &m, &scan_tiles)) {
    set_error_text("gs_induced_slice_compact: pass the workspace given to gs_induced_slice_mark");
    return GS_ERR_WORKSPACE;
  }
  hipStream_t st = static_cast<hipStream_t>(stream);
  const dim3 grid(blocks_for(m.tiles, kCopyTiles));
  const bool stream_out = streams(D, static_cast<size_t>(id_bytes), out_data != nullptr);
  auto go = [&](auto* kernel, auto* indices) {
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, st, m, indices, out_data);
  };
  if (id_bytes == 8)
    go(stream_out ? induced_compact_kernel<int64_t, true> : induced_compact_kernel<int64_t, false>,
       static_cast<int64_t*>(out_indices));
  else
    go(stream_out ? induced_compact_kernel<int32_t, true> : induced_compact_kernel<int32_t, false>,
       static_cast<int32_t*>(out_indices));
  return check_launch("induced_slice_compact");
}

}  // extern "C"
