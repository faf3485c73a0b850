// The tail of a layer-wise (LADIES / FastGCN style) sampler on a column slice held as a COO:
// the node set, the rows of the slice that belong to it, and the block's values in the order
// the reference's operator chain leaves them in
//   nodes = unique(cat(seeds, picked));  sub = U[nodes, :].divide(prob[nodes], axis=1)
//   (examples/ladies/ladies_raw.py:15-22: a CSR of all of U, src/graph.cc:258-283, its row
//   slice, a division by row, then a CSC of the result for normalize(axis=0) and the block,
//   src/graph.cc:585-644, 782-839)
// without the sorts of all of U: the edges are tested against the sorted node set (held in
// LDS), and only the kept ones are sorted, once, by (column, new row).
#include "gs_common.hpp"

namespace gs {
namespace {

// ---------------------------------------------------------------- node set ----
constexpr int kUnionThreads = 1024;

// out = the distinct values of a and b in increasing order (what torch.unique gives for ids,
// which are not negative), *count = how many: one workgroup, bitonic sort of
// kUnionThreads * PER >= na + nb keys.  A thread holds PER consecutive keys in registers: pairs
// up to PER / 2 apart are compared there, those of one wave by a lane exchange, and only the
// ones of different waves (10 of the 55 to 91 steps) meet in LDS behind a barrier.  A chain of
// short dependent steps is all this launch is: with every step through LDS and a barrier it took
// 17 us for 1024 keys, now 6, and 10 for 1383.
template <typename KeyT>
__device__ __forceinline__ void order_pair(KeyT& x, KeyT& y, bool ascending) {
  const KeyT lo = x < y ? x : y, hi = x < y ? y : x;
  x = ascending ? lo : hi;
  y = ascending ? hi : lo;
}

// sorts the keys (~0: none) of the workgroup and writes the distinct ones
template <typename IdT, typename KeyT, int PER>
__device__ __forceinline__ void sort_and_write(KeyT (&key)[PER], KeyT* s_keys, int64_t* s_scan,
                                               IdT* __restrict__ out, int64_t* __restrict__ count) {
  constexpr KeyT kNoKey = ~KeyT(0);
  constexpr int kSlots = kUnionThreads * PER;
  const int t = threadIdx.x;
  for (int k = 2; k <= kSlots; k <<= 1) {
    int j = k >> 1;
    // partners in other waves: j / PER >= 64 threads away
    for (; j >= kWave * PER; j >>= 1) {
#pragma unroll
      for (int r = 0; r < PER; ++r) s_keys[r * kUnionThreads + t] = key[r];
      __syncthreads();
      const int other = t ^ (j / PER);
      const bool keep_low = ((t * PER & k) == 0) == (t < other);
#pragma unroll
      for (int r = 0; r < PER; ++r) {
        const KeyT y = s_keys[r * kUnionThreads + other];
        key[r] = (y < key[r]) == keep_low ? y : key[r];
      }
      __syncthreads();
    }
    for (; j >= PER; j >>= 1) {  // partners in other lanes of this wave
      const bool keep_low = ((t * PER & k) == 0) == ((t & (j / PER)) == 0);
#pragma unroll
      for (int r = 0; r < PER; ++r) {
        const KeyT y = __shfl_xor(key[r], j / PER, kWave);
        key[r] = (y < key[r]) == keep_low ? y : key[r];
      }
    }
    // partners of the thread's own: distance and direction are known to the compiler
#pragma unroll
    for (int d = PER / 2; d > 0; d >>= 1) {
      if (d <= j) {
#pragma unroll
        for (int r = 0; r < PER; ++r)
          if ((r & d) == 0) order_pair(key[r], key[r | d], ((t * PER + r) & k) == 0);
      }
    }
  }
  // the last key of the thread before tells whether this thread's first is a new one
  s_keys[t] = key[PER - 1];
  __syncthreads();
  KeyT before = t > 0 ? s_keys[t - 1] : kNoKey;
  bool fresh[PER];
  int64_t mine = 0;
#pragma unroll
  for (int r = 0; r < PER; ++r) {
    fresh[r] = key[r] != kNoKey && key[r] != before;
    before = key[r];
    mine += fresh[r];
  }
  int64_t total;
  int64_t at = block_exclusive_scan<kUnionThreads>(mine, &total, s_scan);
#pragma unroll
  for (int r = 0; r < PER; ++r)
    if (fresh[r]) out[at++] = static_cast<IdT>(key[r]);
  if (t == 0) *count = total;
}

template <typename IdT, int PER>
__global__ void __launch_bounds__(kUnionThreads)
sorted_union_kernel(const IdT* __restrict__ a, int64_t na, const IdT* __restrict__ b, int64_t nb,
                    IdT* __restrict__ out, int64_t* __restrict__ count) {
  using KeyT = typename std::make_unsigned<IdT>::type;
  extern __shared__ unsigned long long s_raw[];  // key r of thread t at r * kUnionThreads + t
  __shared__ int64_t s_scan[kUnionThreads / kWave + 1];
  const int t = threadIdx.x;
  KeyT key[PER];
  bool wide = false;
#pragma unroll
  for (int r = 0; r < PER; ++r) {
    const int64_t i = static_cast<int64_t>(r) * kUnionThreads + t;  // (any key may start anywhere)
    key[r] = ~KeyT(0);  // sorts behind every id
    if (i < na)
      key[r] = static_cast<KeyT>(a[i]);
    else if (i < na + nb)
      key[r] = static_cast<KeyT>(b[i - na]);
    wide |= i < na + nb && key[r] >= 0xFFFFFFFFull;
  }
  if constexpr (sizeof(KeyT) == 8) {
    // ids of any graph below 2^32 nodes: half the lane moves and half the LDS traffic (3000 keys 27 -> 18 us)
    if (!__syncthreads_or(wide)) {
      uint32_t narrow[PER];
#pragma unroll
      for (int r = 0; r < PER; ++r) narrow[r] = static_cast<uint32_t>(key[r]);
      sort_and_write(narrow, reinterpret_cast<uint32_t*>(s_raw), s_scan, out, count);
      return;
    }
  }
  sort_and_write(key, reinterpret_cast<KeyT*>(s_raw), s_scan, out, count);
}

// ------------------------------------------------------------- row filter ----
constexpr int kPickThreads = 256;
constexpr int kPickItems = 16;
constexpr int kPickTile = kPickThreads * kPickItems;
constexpr int kPickPosBits = 12;  // of a position inside a tile
static_assert(kPickTile == 1 << kPickPosBits, "a tile's positions fill the field");

// Where node `i` of 2^bits sorted nodes stands in their search tree (children of k at 2k and
// 2k + 1, the last node apart at 0): the levels' nodes lie side by side, so that the lanes of a
// wave read neighbouring words at every step -- in the sorted array itself the candidates of a
// step are a power of two apart and fall on one bank.
__device__ __forceinline__ int tree_place(int i, int bits) {
  const int up = __ffs(i + 1) - 1;  // levels above the leaves
  return up == bits ? 0 : (1 << (bits - 1 - up)) + ((i + 1) >> (up + 1));
}

// Pass one: which edges' rows are among the nodes (looked up in a search tree in LDS).  The kept
// ones leave as place among the nodes << 12 | position in the tile, packed at the front of the
// tile's range of `packed`, in the order of the edges; tile_counts[tile] = how many.  A wave takes
// 1024 consecutive edges, 16 a lane, whose reads go out together and whose searches run side by
// side: one after another each was a chain of ten dependent LDS reads
// (2 M edges, 1 k nodes: 31 -> 12 us; 22 k edges: 20 -> 8 us).  (An open-addressing table over
// the node set in LDS, built by every workgroup for itself, was no faster than those searches.)
template <typename IdT>
__global__ void __launch_bounds__(kPickThreads)
pick_count_kernel(const IdT* __restrict__ row, int64_t E, const IdT* __restrict__ nodes,
                  const int64_t* __restrict__ num_nodes, int max_nodes, int tree_bits,
                  int* __restrict__ packed, int64_t* __restrict__ tile_counts) {
  using KeyT = typename std::make_unsigned<IdT>::type;
  extern __shared__ unsigned long long s_raw[];
  KeyT* s_tree = reinterpret_cast<KeyT*>(s_raw);
  __shared__ int s_waves[kPickThreads / kWave];
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  const int64_t tile = static_cast<int64_t>(blockIdx.x) * kPickTile;
  const int first = wave * kPickItems * kWave + lane;
  IdT rows[kPickItems];
#pragma unroll
  for (int u = 0; u < kPickItems; ++u) {
    const int64_t e = tile + first + u * kWave;
    rows[u] = row[e < E ? e : E - 1];
  }
  const int64_t n64 = *num_nodes;
  const int n = static_cast<int>(n64 < max_nodes ? n64 : max_nodes);
  const int places = 1 << tree_bits;
  for (int i = threadIdx.x; i < places; i += kPickThreads)
    s_tree[tree_place(i, tree_bits)] = i < n ? static_cast<KeyT>(nodes[i]) : ~KeyT(0);
  __syncthreads();
  int at[kPickItems];
  KeyT found[kPickItems];
  const KeyT last = s_tree[0];
#pragma unroll
  for (int u = 0; u < kPickItems; ++u) at[u] = 1, found[u] = last;
  for (int step = 0; step < tree_bits; ++step) {
#pragma unroll
    for (int u = 0; u < kPickItems; ++u) {
      const KeyT node = s_tree[at[u]];
      const bool below = node < static_cast<KeyT>(rows[u]);
      found[u] = below ? found[u] : node;  // the smallest node not below the row
      at[u] = 2 * at[u] + below;
    }
  }
  int kept[kPickItems];
  int mine = 0;  // of the wave
  unsigned int mask = 0;
#pragma unroll
  for (int u = 0; u < kPickItems; ++u) {
    at[u] -= places;  // how many nodes are below the row
    const bool keep = found[u] == static_cast<KeyT>(rows[u]) && at[u] < n &&
                      tile + first + u * kWave < E;
    const unsigned long long lanes = __ballot(keep);
    kept[u] = mine + __popcll(lanes & ((1ull << lane) - 1ull));
    mine += __popcll(lanes);
    mask |= static_cast<unsigned int>(keep) << u;
  }
  if (lane == 0) s_waves[wave] = mine;
  __syncthreads();
  int before = 0, total = 0;
#pragma unroll
  for (int w = 0; w < kPickThreads / kWave; ++w) {
    before += w < wave ? s_waves[w] : 0;
    total += s_waves[w];
  }
#pragma unroll
  for (int u = 0; u < kPickItems; ++u)
    if ((mask >> u) & 1u)
      packed[tile + before + kept[u]] = (at[u] << kPickPosBits) | (first + u * kWave);
  if (threadIdx.x == 0) tile_counts[blockIdx.x] = total;
}

// Pass two: the kept edges, in edge order, as key = column << node_bits | place and their
// position in the COO.  A tile's first output place is the sum of the counts of the tiles before
// it: added up by the tile itself (SELF_PREFIX) or left by a scan of the counts.
template <typename IdT, bool SELF_PREFIX>
__global__ void __launch_bounds__(kPickThreads)
pick_fill_kernel(const int* __restrict__ packed, const IdT* __restrict__ col, int node_bits,
                 const int64_t* __restrict__ tile_counts, const int64_t* __restrict__ tile_offsets,
                 int64_t num_tiles, const int64_t* __restrict__ num_nodes,
                 IdT* __restrict__ kept_key, IdT* __restrict__ kept_pos,
                 int64_t* __restrict__ totals, gs_mailbox* box, int64_t ticket) {
  __shared__ int64_t s_scan[kPickThreads / kWave + 1];
  const int64_t tile = blockIdx.x;
  const int count = static_cast<int>(tile_counts[tile]);
  int64_t out;
  if (SELF_PREFIX) {
    int64_t part = 0;
    for (int64_t t = threadIdx.x; t < tile; t += kPickThreads) part += tile_counts[t];
    block_exclusive_scan<kPickThreads>(part, &out, s_scan);
  } else {
    out = tile_offsets[tile];
  }
  if (tile == num_tiles - 1 && threadIdx.x == 0) {
    totals[0] = *num_nodes;
    totals[1] = out + count;
    post_mailbox(box, out + count, ticket);
  }
  for (int k = threadIdx.x; k < count; k += kPickThreads) {
    const int word = packed[tile * kPickTile + k];
    const int64_t e = tile * kPickTile + (word & (kPickTile - 1));
    kept_key[out + k] =
        static_cast<IdT>((static_cast<int64_t>(col[e]) << node_bits) | (word >> kPickPosBits));
    kept_pos[out + k] = static_cast<IdT>(e);
  }
}

struct LoadCounts {
  const int64_t* p;
  __device__ __forceinline__ int64_t operator()(int64_t i) const { return p[i]; }
};

// ------------------------------------------------------------ block values ----
// offsets of the columns from the kept edges' keys (which come by column): the thread of a
// column's first edge writes the offsets of that column and of the empty ones before it, the
// last edge's thread those of the columns behind
template <typename IdT>
__global__ void __launch_bounds__(256)
column_offsets_kernel(const IdT* __restrict__ kept_key, int64_t kept, int node_bits,
                      int64_t num_cols, int64_t* __restrict__ out_indptr) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (kept == 0) {
    for (int64_t c = i; c <= num_cols; c += static_cast<int64_t>(gridDim.x) * 256) out_indptr[c] = 0;
    return;
  }
  if (i >= kept) return;
  const int64_t c = static_cast<int64_t>(kept_key[i]) >> node_bits;
  const int64_t before = i > 0 ? static_cast<int64_t>(kept_key[i - 1]) >> node_bits : -1;
  for (int64_t k = before + 1; k <= c && k <= num_cols; ++k) out_indptr[k] = i;
  if (i == kept - 1)
    for (int64_t k = c + 1; k <= num_cols; ++k) out_indptr[k] = kept;
}

// The kept edges of every column in the order of (new row, position) -- the order of a stable
// sort of all kept edges by key, which for a few tens of thousands of edges is three radix passes
// of two launches each -- and their values data / divisor[row].  Two kinds of workgroups in one
// launch, both bound by the dependent trips to memory of one workgroup (position, row, divisor):
//  * columns of up to kShortColumn kept edges (nearly all) by edge: a thread counts the edges of
//    its column that come before its own, among keys that the workgroup has staged in LDS (read
//    from memory one after another they were most of 14 us for 871 edges);
//  * the longer ones (hub seeds, parallel edges included) a workgroup each, by a counting sort in
//    LDS, 4096 edges at a time: a wave walks its share 64 edges at a time, a lane finds the lanes
//    that hold the same place with one ballot per key bit, and counts per place in 16-bit
//    counters of the wave's own; an edge's place is the bin's start + the counts of the waves before
//    its own + its rank in its wave.  A column that fits one round of 4096 gets the bins'
//    starts from those counters, a longer one from a histogram of all of it beforehand.
// 512 columns, 871 edges: 14 -> 8 us; 1024 columns, 68 k edges, 82 of them long, up to 3004: 29 ->
// 18 us (from 256 threads a workgroup, the long columns listed by a launch of their own).
constexpr int kShortColumn = 256;
constexpr int kOrderThreads = 1024;
constexpr int kOrderWaves = kOrderThreads / kWave;
constexpr int kColumnPer = 4;  // edges of a thread in a round
constexpr int kColumnStage = kOrderThreads * kColumnPer;
constexpr int kShortStage = kOrderThreads + 2 * (kShortColumn - 1);

// waves that count: as many as leave room for two workgroups a compute unit (one with 8192 places)
inline int order_groups(int node_bits) { return node_bits <= 10 ? 16 : (node_bits == 11 ? 8 : 4); }

template <typename IdT>
__device__ __forceinline__ void order_short_edges(int64_t first, int64_t kept,
                                                  const IdT* __restrict__ kept_key,
                                                  const IdT* __restrict__ kept_pos, int node_bits,
                                                  const int64_t* __restrict__ indptr,
                                                  const IdT* __restrict__ row,
                                                  const float* __restrict__ data,
                                                  const float* __restrict__ divisor,
                                                  IdT* __restrict__ out_row,
                                                  float* __restrict__ out_value, IdT* s_keys) {
  // the keys of every column of up to 256 edges that has one among first .. first + 1023
  const int64_t from = first < kShortColumn - 1 ? 0 : first - (kShortColumn - 1);
  const int64_t to = first + kOrderThreads + kShortColumn - 1 < kept
                         ? first + kOrderThreads + kShortColumn - 1 : kept;
  const int64_t i = first + threadIdx.x;
  const int64_t mine = i < kept ? i : kept - 1;
  const IdT key = kept_key[mine];
  const int64_t e = static_cast<int64_t>(kept_pos[mine]);
  for (int64_t j = from + threadIdx.x; j < to; j += kOrderThreads) s_keys[j - from] = kept_key[j];
  const int64_t column = static_cast<int64_t>(key) >> node_bits;
  const int64_t lo = indptr[column], hi = indptr[column + 1];
  const IdT r = row[e];
  const float w = data ? data[e] : 1.0f;
  const float d = divisor[r];
  __syncthreads();
  if (i >= kept || hi - lo > kShortColumn) return;  // (a long column: its own workgroup's)
  int before = 0;
  const int at = static_cast<int>(i - from), end = static_cast<int>(hi - from);
#pragma unroll 8
  for (int j = static_cast<int>(lo - from); j < end; ++j) {
    const IdT y = s_keys[j];
    before += (y < key) || (y == key && j < at);  // (one column: the keys differ in the place only)
  }
  out_row[lo + before] = r;
  out_value[lo + before] = w / d;
}

template <typename IdT, int GROUPS>
__global__ void __launch_bounds__(kOrderThreads)
order_columns_kernel(const IdT* __restrict__ kept_key, const IdT* __restrict__ kept_pos,
                     int node_bits, const int64_t* __restrict__ indptr,
                     const IdT* __restrict__ row, const float* __restrict__ data,
                     const float* __restrict__ divisor, IdT* __restrict__ out_row,
                     float* __restrict__ out_value, unsigned int long_blocks, int64_t kept) {
  extern __shared__ unsigned long long s_raw[];
  __shared__ int64_t s_scan[kOrderWaves + 1];
  if (blockIdx.x >= long_blocks) {
    order_short_edges(static_cast<int64_t>(blockIdx.x - long_blocks) * kOrderThreads, kept, kept_key,
                      kept_pos, node_bits, indptr, row, data, divisor, out_row, out_value,
                      reinterpret_cast<IdT*>(s_raw));
    return;
  }
  // The launch's first workgroups: number b takes the column of the kept edge b * 257, if it is a
  // long one and that is the first such edge in it (a column of 257 edges or more has one).
  const int64_t probe = static_cast<int64_t>(blockIdx.x) * (kShortColumn + 1);
  const int64_t column = static_cast<int64_t>(kept_key[probe]) >> node_bits;
  const int64_t lo = indptr[column], hi = indptr[column + 1];
  const int64_t len = hi - lo;
  if (len <= kShortColumn || probe - (kShortColumn + 1) >= lo) return;
  const int places = 1 << node_bits;
  const unsigned int mask = static_cast<unsigned int>(places) - 1u;
  unsigned int* s_bin = reinterpret_cast<unsigned int*>(s_raw);
  unsigned int* s_key = s_bin + (places < 4 ? 4 : places);  // (all three 16-byte aligned)
  unsigned short* s_count = reinterpret_cast<unsigned short*>(s_key + kColumnStage);
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  const bool one_round = len <= kColumnStage;
  // exclusive scan of the bins: a thread owns `per` consecutive ones
  const int per = places > kOrderThreads ? places / kOrderThreads : 1;
  auto scan_bins = [&]() {
    const int first = threadIdx.x * per;
    int64_t mine = 0;
    for (int u = 0; u < per; ++u)
      if (first + u < places) mine += s_bin[first + u];
    int64_t total;
    int64_t at = block_exclusive_scan<kOrderThreads>(mine, &total, s_scan);
    for (int u = 0; u < per; ++u) {
      if (first + u < places) {
        const unsigned int n = s_bin[first + u];
        s_bin[first + u] = static_cast<unsigned int>(at);
        at += n;
      }
    }
    __syncthreads();
  };
  if (!one_round) {
    for (int j = threadIdx.x; j < places; j += kOrderThreads) s_bin[j] = 0u;
    __syncthreads();
    for (int64_t j0 = threadIdx.x; j0 < len; j0 += kColumnStage) {
      unsigned int k[kColumnPer];
#pragma unroll
      for (int u = 0; u < kColumnPer; ++u) {
        const int64_t j = j0 + u * kOrderThreads;
        k[u] = static_cast<unsigned int>(kept_key[lo + (j < len ? j : len - 1)]) & mask;
      }
#pragma unroll
      for (int u = 0; u < kColumnPer; ++u)
        if (j0 + u * kOrderThreads < len) atomicAdd(&s_bin[k[u]], 1u);
    }
    __syncthreads();
    scan_bins();
  }
  // without data every value is one; the read then goes to a word that is always there
  const bool has_data = data != nullptr;
  const float* values = has_data ? data : divisor;
  for (int64_t base = 0; base < len; base += kColumnStage) {
    const int n = static_cast<int>(len - base < kColumnStage ? len - base : kColumnStage);
    // everything a thread's edges need from memory is on its way while they are ranked
    unsigned int key[kColumnPer];
    int64_t e[kColumnPer];
    IdT r[kColumnPer];
    float w[kColumnPer], d[kColumnPer];
#pragma unroll
    for (int u = 0; u < kColumnPer; ++u) {
      const int j = static_cast<int>(threadIdx.x) + u * kOrderThreads;
      const int64_t at = lo + base + (j < n ? j : n - 1);
      key[u] = static_cast<unsigned int>(kept_key[at]) & mask;
      e[u] = static_cast<int64_t>(kept_pos[at]);
    }
    for (int j = threadIdx.x; j < GROUPS * places / 8; j += kOrderThreads)
      reinterpret_cast<uint4*>(s_count)[j] = make_uint4(0u, 0u, 0u, 0u);
#pragma unroll
    for (int u = 0; u < kColumnPer; ++u) {
      const int j = static_cast<int>(threadIdx.x) + u * kOrderThreads;
      if (j < n) s_key[j] = key[u];
    }
#pragma unroll
    for (int u = 0; u < kColumnPer; ++u) r[u] = row[e[u]];
#pragma unroll
    for (int u = 0; u < kColumnPer; ++u) w[u] = values[has_data ? e[u] : 0];
#pragma unroll
    for (int u = 0; u < kColumnPer; ++u) d[u] = divisor[r[u]];
    __syncthreads();
    const int share = ((n + GROUPS * kWave - 1) / (GROUPS * kWave)) * kWave;  // edges of a wave
    if (wave < GROUPS) {
      const int end = (wave + 1) * share < n ? (wave + 1) * share : n;
      unsigned short* mine = s_count + wave * places;
      for (int c = wave * share; c < end; c += kWave) {
        const bool valid = c + lane < end;
        const unsigned int k = valid ? s_key[c + lane] : 0u;
        unsigned long long peers = __ballot(valid);
        for (int b = 0; b < node_bits; ++b) {
          const bool bit = (k >> b) & 1u;
          const unsigned long long with_bit = __ballot(valid && bit);
          peers &= bit ? with_bit : ~with_bit;
        }
        if (valid) {
          const unsigned int ahead = __popcll(peers & ((1ull << lane) - 1ull));
          const unsigned int start = mine[k];
          s_key[c + lane] = start + ahead;  // the edge's rank in its wave's share
          if (lane == 63 - __clzll(peers))
            mine[k] = static_cast<unsigned short>(start + __popcll(peers));
        }
      }
    }
    __syncthreads();
    if (one_round) {
      for (int k = threadIdx.x; k < places; k += kOrderThreads) {
        unsigned int total = 0u;
#pragma unroll
        for (int g = 0; g < GROUPS; ++g) total += s_count[g * places + k];
        s_bin[k] = total;
      }
      __syncthreads();
      scan_bins();
    }
#pragma unroll
    for (int u = 0; u < kColumnPer; ++u) {
      const int j = static_cast<int>(threadIdx.x) + u * kOrderThreads;
      if (j < n) {
        unsigned int place = s_bin[key[u]] + s_key[j];
        const int mine = j / share;
        for (int g = 0; g < mine; ++g) place += s_count[g * places + key[u]];
        out_row[lo + place] = r[u];
        out_value[lo + place] = (has_data ? w[u] : 1.0f) / d[u];
      }
    }
    if (one_round) return;
    __syncthreads();
    for (int k = threadIdx.x; k < places; k += kOrderThreads) {
      unsigned int total = s_bin[k];
#pragma unroll
      for (int g = 0; g < GROUPS; ++g) total += s_count[g * places + k];
      s_bin[k] = total;
    }
    __syncthreads();
  }
}

// (per call: the attribute belongs to the device the call runs on)
int allow_lds(const void* kernel, size_t bytes, const char* who) {
  if (bytes <= 48 * 1024) return GS_OK;
  const hipError_t allowed = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                                 static_cast<int>(bytes));
  if (allowed == hipSuccess) return GS_OK;
  set_error_text("%s: %s", who, hipGetErrorString(allowed));
  return GS_ERR_LAUNCH;
}

template <typename IdT>
int order_columns_launch(int64_t kept, int node_bits, hipStream_t st,
                         const void* kept_key, const void* kept_pos, const int64_t* indptr,
                         const void* row, const float* data, const float* divisor, void* out_row,
                         float* out_value) {
  // one workgroup for each multiple of 257 among the kept edges
  const unsigned int long_blocks = static_cast<unsigned int>((kept - 1) / (kShortColumn + 1) + 1);
  const dim3 grid(long_blocks + static_cast<unsigned>(blocks_for(kept, kOrderThreads)));
  const size_t places = size_t(1) << node_bits;
  const int groups = order_groups(node_bits);
  size_t lds = ((places < 4 ? 4 : places) + kColumnStage) * sizeof(unsigned int) +
               places * groups * sizeof(unsigned short);
  if (lds < kShortStage * sizeof(IdT)) lds = kShortStage * sizeof(IdT);
  auto* kernel = groups == 16  ? order_columns_kernel<IdT, 16>
                 : groups == 8 ? order_columns_kernel<IdT, 8>
                               : order_columns_kernel<IdT, 4>;
  GS_RETURN_IF_ERROR(allow_lds(reinterpret_cast<const void*>(kernel), lds, "gs_coo_block_values"));
  hipLaunchKernelGGL(kernel, grid, dim3(kOrderThreads), lds, st, static_cast<const IdT*>(kept_key),
                     static_cast<const IdT*>(kept_pos), node_bits, indptr,
                     static_cast<const IdT*>(row), data, divisor, static_cast<IdT*>(out_row),
                     out_value, long_blocks, kept);
  return GS_OK;
}

inline int bits_of(int64_t n) {  // smallest b with 2^b >= n
  int b = 0;
  while ((int64_t(1) << b) < n) ++b;
  return b;
}

template <typename IdT, int PER>
int sorted_union_launch(const void* a, int64_t na, const void* b, int64_t nb, void* out,
                        int64_t* count, hipStream_t st) {
  const size_t lds = sizeof(IdT) * kUnionThreads * PER;
  GS_RETURN_IF_ERROR(allow_lds(reinterpret_cast<const void*>(sorted_union_kernel<IdT, PER>), lds,
                               "gs_sorted_union"));
  hipLaunchKernelGGL((sorted_union_kernel<IdT, PER>), dim3(1), dim3(kUnionThreads), lds, st,
                     static_cast<const IdT*>(a), na, static_cast<const IdT*>(b), nb,
                     static_cast<IdT*>(out), count);
  return check_launch("sorted_union");
}

template <typename IdT>
int sorted_union_t(const void* a, int64_t na, const void* b, int64_t nb, void* out, int64_t* count,
                   hipStream_t st) {
  const int64_t n = na + nb;
  const auto launch = n <= kUnionThreads       ? sorted_union_launch<IdT, 1>
                      : n <= 2 * kUnionThreads ? sorted_union_launch<IdT, 2>
                      : n <= 4 * kUnionThreads ? sorted_union_launch<IdT, 4>
                                               : sorted_union_launch<IdT, 8>;
  return launch(a, na, b, nb, out, count, st);
}

template <typename IdT>
int pick_rows_t(const void* row, const void* col, int64_t E, const void* nodes,
                const int64_t* num_nodes, int max_nodes, void* kept_key, void* kept_pos,
                int64_t* totals, gs_mailbox* box, int64_t ticket, void* workspace,
                size_t workspace_bytes, hipStream_t st) {
  const int64_t tiles = blocks_for(E, kPickTile);
  Carver ws(workspace, workspace_bytes);
  int64_t* counts = ws.take<int64_t>(tiles);
  int64_t* offsets = ws.take<int64_t>(tiles + 1);
  int64_t* scan_ws = ws.take<int64_t>(scan_num_tiles(tiles) + 1);
  int* packed = ws.take<int>(E);
  if (!ws.ok) {
    set_error_text("gs_coo_pick_rows: workspace needs %zu bytes, 256-byte aligned",
                   gs_coo_pick_rows_workspace_bytes(E));
    return GS_ERR_WORKSPACE;
  }
  const int node_bits = bits_of(max_nodes);
  const size_t lds = sizeof(IdT) << node_bits;
  GS_RETURN_IF_ERROR(allow_lds(reinterpret_cast<const void*>(pick_count_kernel<IdT>), lds,
                               "gs_coo_pick_rows"));
  const dim3 grid(static_cast<unsigned>(tiles));
  hipLaunchKernelGGL(pick_count_kernel<IdT>, grid, dim3(kPickThreads), lds, st,
                     static_cast<const IdT*>(row), E, static_cast<const IdT*>(nodes), num_nodes,
                     max_nodes, node_bits, packed, counts);
  // up to 4096 tiles (16 M edges) a tile adds up the counts before it by itself, at most sixteen
  // reads a thread, instead of a launch for their scan
  if (tiles <= kScanSelfPrefixTiles) {
    hipLaunchKernelGGL((pick_fill_kernel<IdT, true>), grid, dim3(kPickThreads), 0, st, packed,
                       static_cast<const IdT*>(col), node_bits, counts,
                       static_cast<const int64_t*>(nullptr), tiles, num_nodes,
                       static_cast<IdT*>(kept_key), static_cast<IdT*>(kept_pos), totals, box, ticket);
  } else {
    LoadCounts f{counts};
    GS_RETURN_IF_ERROR(exclusive_scan(f, tiles, offsets, scan_ws, st));
    hipLaunchKernelGGL((pick_fill_kernel<IdT, false>), grid, dim3(kPickThreads), 0, st, packed,
                       static_cast<const IdT*>(col), node_bits, counts, offsets, tiles, num_nodes,
                       static_cast<IdT*>(kept_key), static_cast<IdT*>(kept_pos), totals, box, ticket);
  }
  return check_launch("coo_pick_rows");
}

}  // namespace
}  // namespace gs

using namespace gs;

extern "C" {

int gs_sorted_union(const void* a, int64_t na, const void* b, int64_t nb, int id_bytes, void* out,
                    int64_t* count, void* stream) {
  GS_REQUIRE(na >= 0 && nb >= 0 && na + nb >= 1 && na + nb <= gs_sorted_union_max(id_bytes),
             "gs_sorted_union: %lld + %lld values, takes 1 to %lld",
             static_cast<long long>(na), static_cast<long long>(nb),
             static_cast<long long>(gs_sorted_union_max(id_bytes)));
  GS_REQUIRE((na == 0 || a) && (nb == 0 || b) && out && count, "gs_sorted_union: null pointer");
  GS_REQUIRE(valid_id_bytes(id_bytes), "gs_sorted_union: id_bytes must be 4 or 8, got %d", id_bytes);
  hipStream_t st = static_cast<hipStream_t>(stream);
  return id_bytes == 8 ? sorted_union_t<int64_t>(a, na, b, nb, out, count, st)
                       : sorted_union_t<int32_t>(a, na, b, nb, out, count, st);
}

int64_t gs_sorted_union_max(int) { return 8192; }

size_t gs_coo_pick_rows_workspace_bytes(int64_t E) {
  const int64_t tiles = blocks_for(E, kPickTile);
  auto pad = [](size_t b) { return (b + 255u) & ~size_t(255); };
  return pad(tiles * 8) + pad((tiles + 1) * 8) + pad((scan_num_tiles(tiles) + 1) * 8) +
         pad(static_cast<size_t>(E < 1 ? 1 : E) * sizeof(int));
}

int gs_coo_pick_rows(const void* row, const void* col, int id_bytes, int64_t E, const void* nodes,
                     const int64_t* num_nodes, int64_t max_nodes, void* kept_key, void* kept_pos,
                     int64_t* totals, gs_mailbox* mailbox, int64_t ticket, void* workspace,
                     size_t workspace_bytes, void* stream) {
  GS_REQUIRE(valid_id_bytes(id_bytes), "gs_coo_pick_rows: id_bytes must be 4 or 8, got %d", id_bytes);
  GS_REQUIRE(E >= 1 && (id_bytes == 8 || E < (int64_t(1) << 31)),
             "gs_coo_pick_rows: %lld edges (at least one; below 2^31 with 4-byte ids)",
             static_cast<long long>(E));
  GS_REQUIRE(max_nodes >= 1 && max_nodes <= gs_sorted_union_max(id_bytes),
             "gs_coo_pick_rows: room for %lld nodes, takes 1 to %lld",
             static_cast<long long>(max_nodes), static_cast<long long>(gs_sorted_union_max(id_bytes)));
  GS_REQUIRE(row && col && nodes && num_nodes && kept_key && kept_pos && totals,
             "gs_coo_pick_rows: null pointer");
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int n = static_cast<int>(max_nodes);
  return id_bytes == 8 ? pick_rows_t<int64_t>(row, col, E, nodes, num_nodes, n, kept_key, kept_pos,
                                              totals, mailbox, ticket, workspace, workspace_bytes, st)
                       : pick_rows_t<int32_t>(row, col, E, nodes, num_nodes, n, kept_key, kept_pos,
                                              totals, mailbox, ticket, workspace, workspace_bytes, st);
}

size_t gs_coo_block_values_workspace_bytes(int64_t) { return 0; }

int gs_coo_block_values(const void* kept_key, const void* kept_pos, int64_t kept, int64_t max_nodes,
                        const void* row, int id_bytes, const float* data, const float* divisor,
                        int64_t num_cols, void* out_row, float* out_value, int64_t* out_indptr,
                        void* workspace, size_t workspace_bytes, void* stream) {
  GS_REQUIRE(valid_id_bytes(id_bytes), "gs_coo_block_values: id_bytes must be 4 or 8, got %d",
             id_bytes);
  GS_REQUIRE(kept >= 0 && num_cols >= 0, "gs_coo_block_values: negative size");
  GS_REQUIRE(max_nodes >= 1 && max_nodes <= gs_sorted_union_max(id_bytes),
             "gs_coo_block_values: room for %lld nodes, takes 1 to %lld",
             static_cast<long long>(max_nodes), static_cast<long long>(gs_sorted_union_max(id_bytes)));
  GS_REQUIRE(out_indptr && (kept == 0 || (kept_key && kept_pos && row && divisor && out_row && out_value)),
             "gs_coo_block_values: null pointer");
  (void)workspace;
  (void)workspace_bytes;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int node_bits = bits_of(max_nodes);
  const dim3 by_edge(static_cast<unsigned>(blocks_for(kept, 256)));
  if (id_bytes == 8)
    hipLaunchKernelGGL(column_offsets_kernel<int64_t>, by_edge, dim3(256), 0, st,
                       static_cast<const int64_t*>(kept_key), kept, node_bits, num_cols, out_indptr);
  else
    hipLaunchKernelGGL(column_offsets_kernel<int32_t>, by_edge, dim3(256), 0, st,
                       static_cast<const int32_t*>(kept_key), kept, node_bits, num_cols, out_indptr);
  if (kept > 0 && num_cols > 0) {
    auto* order = id_bytes == 8 ? order_columns_launch<int64_t> : order_columns_launch<int32_t>;
    GS_RETURN_IF_ERROR(order(kept, node_bits, st, kept_key, kept_pos, out_indptr, row, data, divisor,
                             out_row, out_value));
  }
  return check_launch("coo_block_values");
}

}  // extern "C"
