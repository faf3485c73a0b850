// Sparse-format conversion on gfx950: CSC -> COO column expansion and
// COO -> CSC by a stable least-significant-digit radix sort.
//
// Replaces impl::CSC2COOCUDA and impl::COO2CSCCUDA (reference
// src/cuda/format_transform.cu:35,135; the reference leans on cub radix sort,
// whose stability pins the edge order, format_transform.cu:81-100).
//
//  * csc2coo: edge-balanced.  A workgroup owns 4096 consecutive edges; a first
//    launch over the columns has left the column of each tile's first edge in the
//    output, the offsets are read in order from there, the columns mark their first
//    edge in LDS and a running maximum turns the marks into column numbers (the
//    reference runs a full global binary search per edge, format_transform.cu:24-33).
//  * coo2csc: 8-bit digits, only ceil(log2(num_keys)/8) passes
//    (format_transform.cu:58-72 also sorts just the significant bits).  Each
//    pass is histogram -> scan -> stable scatter; the scatter ranks equal digits
//    inside a wave with 8 ballots (no LDS atomics, order preserved) and across
//    waves with a small LDS table.  What moves is one 64-bit word per edge, key
//    above and original position below, and the value in 32 bits, so a pass is 12
//    bytes in and 12 bytes out per edge and the permutation falls out of the last
//    pass.  indptr comes from the tiles of the last pass where the values travel in
//    the words, else from the places where the sorted keys change, or, with
//    fewer edges than columns, from one search per column confined to the keys of
//    the workgroup's 256 columns.
//  * distinct ids of an edge list: a bit per possible id in LDS, slice by slice, or, for short
//    lists and large ids, a byte per possible id marked with plain stores.
#include <algorithm>

#include "gs_common.hpp"
#include "gs_one.hpp"

namespace gs {
namespace {

constexpr int kThreads = 256;
constexpr int kItems = 8;
constexpr int kTile = kThreads * kItems;

template <typename P>
__device__ __forceinline__ int64_t upper_bound(P a, int64_t n, int64_t v) {
  int64_t lo = 0, hi = n;
  while (lo < hi) {
    int64_t mid = (lo + hi) >> 1;
    if (a[mid] <= v) lo = mid + 1; else hi = mid;
  }
  return lo;
}

constexpr int kCooItems = 16;
constexpr int kCooTile = kThreads * kCooItems;

// (A thread's sixteen marks lie side by side; one spare word after every sixteen keeps the
// threads of a wave on different LDS banks when each walks its own run.)
__device__ __forceinline__ int coo_slot(int i) { return i + (i >> 4); }

// First of two launches: every column with edges writes its number at the first position of
// each 4096-edge tile that begins inside it, so that the tile's workgroup finds the column
// of its first edge with one read instead of a search through the offsets.  The numbers go
// into the output itself (the tile overwrites its own first entry at the end).  A column
// that spans more than 64 tiles is written by its whole wave.
template <typename IdT>
__global__ void __launch_bounds__(kThreads)
coo_tile_heads_kernel(const int64_t* __restrict__ indptr, int64_t num_cols, IdT* __restrict__ col) {
  const int64_t c = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
  int64_t t0 = 0, t1 = -1;
  if (c < num_cols) {
    const int64_t s = indptr[c], e = indptr[c + 1];
    if (e > s) {
      t0 = (s + kCooTile - 1) / kCooTile;
      t1 = (e - 1) / kCooTile;
    }
  }
  const bool wide = t1 - t0 >= kWave;
  if (!wide)
    for (int64_t t = t0; t <= t1; ++t) col[t * kCooTile] = static_cast<IdT>(c);
  unsigned long long todo = __ballot(wide);
  const int lane = threadIdx.x & (kWave - 1);
  while (todo) {
    const int src = __ffsll(static_cast<long long>(todo)) - 1;
    todo &= todo - 1;
    const int64_t w0 = __shfl(t0, src, kWave), w1 = __shfl(t1, src, kWave);
    const int64_t wc = __shfl(c, src, kWave);
    for (int64_t t = w0 + lane; t <= w1; t += kWave) col[t * kCooTile] = static_cast<IdT>(wc);
  }
}

// A workgroup owns kCooTile consecutive edges.  The first entry of its output holds the last
// column that starts at or before the tile (left there by the launch above); from there the
// offsets are read in order, 256 at a time.  The columns that start inside the tile mark
// their first edge in LDS (of several empty columns at one position the highest wins, which
// is the owner), and a running maximum over the marks gives every edge its column: sixteen
// consecutive edges per thread, one maximum per thread across the workgroup.  No search.
// (DCSC: stored column c stands for node ids[c], format_transform.cu:48-60; a switch at
// compile time, because a load that may or may not happen before a store makes every store
// wait for everything in flight.)
template <typename IdT, bool DCSC>
__global__ void __launch_bounds__(kThreads)
csc2coo_kernel(const int64_t* __restrict__ indptr, int64_t num_cols, int64_t nnz,
               const IdT* __restrict__ ids, IdT* __restrict__ col) {
  __shared__ int s_mark[kCooTile + kCooTile / 16];
  __shared__ int s_wave[kThreads / kWave];
  __shared__ bool s_more;
  const int64_t p0 = static_cast<int64_t>(blockIdx.x) * kCooTile;
  const int64_t p1 = p0 + kCooTile < nnz ? p0 + kCooTile : nnz;
  const int64_t base = static_cast<int64_t>(col[p0]);  // holds edge p0
  for (int i = threadIdx.x; i < kCooTile + kCooTile / 16; i += kThreads) s_mark[i] = 0;
  const int64_t kNone = INT64_MAX;
  int64_t ahead = base + 1 + threadIdx.x <= num_cols ? indptr[base + 1 + threadIdx.x] : kNone;
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  __syncthreads();
  // columns base + 1 ... that start before p1 start inside the tile (after p0: the last one
  // that starts at p0 is the base); the offsets are in order, so the last thread tells
  // whether the next 256 have to be looked at as well
  for (int64_t r = base + 1 + threadIdx.x;; r += kThreads) {
    const bool inside = ahead < p1;
    if (inside)
      atomicMax(&s_mark[coo_slot(static_cast<int>(ahead - p0))], static_cast<int>(r - base));
    if (threadIdx.x == kThreads - 1) s_more = inside;
    __syncthreads();
    if (!s_more) break;
    ahead = r + kThreads <= num_cols ? indptr[r + kThreads] : kNone;
    __syncthreads();  // (everyone has read the flag before it is written again)
  }
  const int at0 = threadIdx.x * (kCooItems + 1);
  int m[kCooItems];
  int run = 0;
#pragma unroll
  for (int k = 0; k < kCooItems; ++k) {
    const int v = s_mark[at0 + k];
    run = v > run ? v : run;
    m[k] = run;  // relative to what holds where the thread begins
  }
  // exclusive running maximum of the threads' last values
  int incl = run;
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    const int y = __shfl_up(incl, d, kWave);
    if (lane >= d && y > incl) incl = y;
  }
  if (lane == kWave - 1) s_wave[wave] = incl;
  __syncthreads();
  int before = __shfl_up(incl, 1, kWave);
  if (lane == 0) before = 0;
  for (int w = 0; w < wave; ++w) before = s_wave[w] > before ? s_wave[w] : before;
  // column numbers (relative to base) go back into the marks' place, so that the stores
  // below are coalesced whatever the id width
#pragma unroll
  for (int k = 0; k < kCooItems; ++k) s_mark[at0 + k] = m[k] > before ? m[k] : before;
  __syncthreads();
  IdT out[kCooItems];
#pragma unroll
  for (int k = 0; k < kCooItems; ++k) {
    const int64_t c = base + s_mark[coo_slot(k * kThreads + threadIdx.x)];
    if (DCSC)
      out[k] = p0 + k * kThreads + threadIdx.x < p1 ? ids[c] : IdT(0);
    else
      out[k] = static_cast<IdT>(c);
  }
#pragma unroll
  for (int k = 0; k < kCooItems; ++k) {
    const int64_t p = p0 + k * kThreads + threadIdx.x;
    if (p < p1) col[p] = out[k];
  }
}

template <typename IdT, bool DCSC>
void launch_csc2coo(const int64_t* indptr, int64_t num_cols, int64_t nnz, const IdT* ids, IdT* col,
                    hipStream_t st) {
  hipLaunchKernelGGL((coo_tile_heads_kernel<IdT>), dim3(blocks_for(num_cols, kThreads)),
                     dim3(kThreads), 0, st, indptr, num_cols, col);
  hipLaunchKernelGGL((csc2coo_kernel<IdT, DCSC>), dim3(blocks_for(nnz, kCooTile)), dim3(kThreads),
                     0, st, indptr, num_cols, nnz, ids, col);
}

// CSC -> doubly-compressed CSC: the columns that own at least one edge, in order, and
// their offsets (what format_transform.cu:172-203 builds from the sorted COO).
struct NonEmptyColumn {
  const int64_t* indptr;
  __device__ __forceinline__ int64_t operator()(int64_t c) const {
    return indptr[c + 1] > indptr[c] ? 1 : 0;
  }
};

template <typename IdT>
__global__ void __launch_bounds__(kThreads)
compress_kernel(const int64_t* __restrict__ indptr, int64_t num_cols,
                const int64_t* __restrict__ prefix, IdT* __restrict__ val_ids,
                int64_t* __restrict__ out_indptr, int64_t* __restrict__ num_valid) {
  const int64_t c = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
  if (c > num_cols) return;
  if (c == num_cols) {
    const int64_t total = prefix[num_cols];
    out_indptr[total] = indptr[num_cols];
    *num_valid = total;
    return;
  }
  const int64_t begin = indptr[c];
  if (indptr[c + 1] > begin) {
    const int64_t w = prefix[c];
    val_ids[w] = static_cast<IdT>(c);
    out_indptr[w] = begin;
  }
}

// Sorted keys as the kernels below read them.
template <typename KeyT>
struct PlainKeys {
  const KeyT* key;
  __device__ __forceinline__ int64_t operator()(int64_t i) const {
    return static_cast<int64_t>(key[i]);
  }
};
// (keys beyond 32 bits: the sort keeps no copy of them)
template <typename KeyT>
struct PermutedKeys {
  const KeyT* key;
  const int64_t* perm;
  __device__ __forceinline__ int64_t operator()(int64_t i) const {
    return static_cast<int64_t>(key[perm[i]]);
  }
};

template <typename Keys>
__device__ __forceinline__ int64_t first_not_below(const Keys& key, int64_t lo, int64_t hi,
                                                   int64_t c) {
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if (key(mid) < c) lo = mid + 1; else hi = mid;
  }
  return lo;
}

// First position in [0, E) whose key is >= c, found by a whole wave: 64 probes split the
// range per step, so 2.7 M keys take four dependent loads instead of twenty-two.  Every
// lane of the wave calls this and gets the answer.
template <typename Keys>
__device__ __forceinline__ int64_t wave_first_not_below(const Keys& key, int64_t E, int64_t c) {
  const int lane = threadIdx.x & (kWave - 1);
  int64_t lo = 0, hi = E;
  while (lo < hi) {
    const int64_t step = (hi - lo + kWave - 1) / kWave;
    const int64_t at = lo + lane * step;
    const bool below = at < hi && key(at) < c;
    const int count = __popcll(__ballot(below));  // probes are sorted: the first `count` are below
    const int64_t new_lo = count > 0 ? lo + (count - 1) * step + 1 : lo;
    const int64_t end = lo + count * step;        // first probe that is not below, if there is one
    hi = (count < kWave && end < hi) ? end : hi;
    lo = new_lo;
  }
  return lo;
}

// indptr from sorted keys: indptr[c] = number of keys < c (format_transform.cu:123-156
// searches the whole key array once per column).  A workgroup owns 256 consecutive
// columns: two wave-wide searches bound the keys that belong to them, and the per-column
// searches run inside that range -- in LDS when it holds at most 4096 keys, which is every
// tile but those of hub columns.
constexpr int kPtrCols = kThreads;
constexpr int kPtrStage = 4096;

template <typename Keys>
__global__ void __launch_bounds__(kThreads)
indptr_from_sorted_kernel(Keys key, int64_t E, int64_t num_keys, int64_t* __restrict__ indptr) {
  __shared__ int64_t s_range[2];
  __shared__ int s_key[kPtrStage];
  const int64_t c0 = static_cast<int64_t>(blockIdx.x) * kPtrCols;
  const int64_t c1 = c0 + kPtrCols < num_keys + 1 ? c0 + kPtrCols : num_keys + 1;
  const int wave = threadIdx.x / kWave;
  if (wave < 2) {
    const int64_t at = wave_first_not_below(key, E, wave == 0 ? c0 : c1);
    if ((threadIdx.x & (kWave - 1)) == 0) s_range[wave] = at;
  }
  __syncthreads();
  const int64_t lo = s_range[0], hi = s_range[1];
  const int n = static_cast<int>(hi - lo <= kPtrStage ? hi - lo : -1);
  if (n >= 0) {
    for (int i = threadIdx.x; i < n; i += kThreads) s_key[i] = static_cast<int>(key(lo + i) - c0);
    __syncthreads();
  }
  const int64_t c = c0 + threadIdx.x;
  if (c >= c1) return;
  if (n >= 0) {
    const int want = static_cast<int>(c - c0);
    int a = 0, b = n;
    while (a < b) {
      const int mid = (a + b) >> 1;
      if (s_key[mid] < want) a = mid + 1; else b = mid;
    }
    indptr[c] = lo + a;
  } else {
    indptr[c] = first_not_below(key, lo, hi, c);
  }
}

// The same offsets from the places where the keys change: item i of [0, E] (key E is the number of
// columns) writes offset i for the columns after key i - 1 up to key i.  Every key is read once,
// coalesced, where the searches above cost a workgroup five dependent trips before it starts.
// Gaps longer than kGapAlone columns are set aside and filled by whole waves, so that a run of
// absent ids does not become one lane's loop; with fewer edges than columns (a slice's rows among
// all rows) nearly every item would be such a gap and the searches are the better split.  With many
// edges per column they are too, since the fill reads all keys and they read a few per column.
// Fill against searches, us, 4-byte keys / 8-byte keys, by edges per column:
//                  1          5.7         16          50         160         500
//    1 M keys               5/6 5/6     5/6 5/6     5/6 5/5     5/6 5/5    4/6 5/5
//   14 M keys  27/37 100/104  19/27 36/39  18/26 26/30  17/26 26/30  16/23 12/14  15/22 7/8
//  114 M keys 262/343 1000/1029 136/212 289/322 124/206 189/229 123/207 174/207 109/187 101/108 102/188 34/36
// (even columns; with hubs the searches gain at 50, 17/24 against 15/20 for 14 M): the line lies at
// 64 edges per column for 4-byte keys, 32 for 8-byte ones.
constexpr int kFillItems = 16;
constexpr int kFillTile = kThreads * kFillItems;
constexpr int kGapAlone = 16;
constexpr int kGapWide = 2048;  // columns from which a gap is filled by the whole workgroup

template <typename KeyT>
__global__ void __launch_bounds__(kThreads)
indptr_fill_kernel(const KeyT* __restrict__ key, int64_t E, int64_t num_keys,
                   int64_t* __restrict__ indptr) {
  __shared__ unsigned short s_gap[kFillTile];
  __shared__ int s_gaps;
  if (threadIdx.x == 0) s_gaps = 0;
  __syncthreads();
  const int64_t base = static_cast<int64_t>(blockIdx.x) * kFillTile;
  // (keys outside [0, num_keys) count as the nearest end: every store stays inside indptr)
  auto bounded = [&](KeyT k) {
    const int64_t v = static_cast<int64_t>(k);
    return v < 0 ? int64_t(-1) : (v > num_keys ? num_keys : v);
  };
  KeyT hi[kFillItems], lo[kFillItems];
#pragma unroll
  for (int k = 0; k < kFillItems; ++k) {
    const int64_t i = base + k * kThreads + threadIdx.x;
    hi[k] = key[i < E ? i : E - 1];
  }
#pragma unroll
  for (int k = 0; k < kFillItems; ++k) {
    const int64_t i = base + k * kThreads + threadIdx.x;
    lo[k] = key[i < 1 ? 0 : (i <= E ? i - 1 : E - 1)];
  }
#pragma unroll
  for (int k = 0; k < kFillItems; ++k) {
    const int at = k * kThreads + threadIdx.x;
    const int64_t i = base + at;
    if (i > E) continue;
    const int64_t first = i == 0 ? 0 : bounded(lo[k]) + 1;
    const int64_t last = i == E ? num_keys : bounded(hi[k]);
    if (last - first < kGapAlone) {
      for (int64_t c = first; c <= last; ++c) indptr[c] = i;
    } else {
      s_gap[atomicAdd(&s_gaps, 1)] = static_cast<unsigned short>(at);
    }
  }
  __syncthreads();
  const int n = s_gaps;
  const int wave = threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
  for (int g = 0; g < n; ++g) {
    const int64_t i = base + s_gap[g];
    const int64_t first = i == 0 ? 0 : bounded(key[i - 1]) + 1;
    const int64_t last = i == E ? num_keys : bounded(key[i]);
    if (last - first >= kGapWide) {
      for (int64_t c = first + threadIdx.x; c <= last; c += kThreads) indptr[c] = i;
    } else if ((g & (kThreads / kWave - 1)) == wave) {
      for (int64_t c = first + lane; c <= last; c += kWave) indptr[c] = i;
    }
  }
}

template <typename KeyT>
void launch_indptr(const KeyT* key, int64_t E, int64_t num_keys, int64_t* indptr, hipStream_t st) {
  if (E > 0 && num_keys <= E && E * static_cast<int64_t>(sizeof(KeyT)) <= 256 * num_keys) {
    hipLaunchKernelGGL((indptr_fill_kernel<KeyT>), dim3(blocks_for(E + 1, kFillTile)),
                       dim3(kThreads), 0, st, key, E, num_keys, indptr);
    return;
  }
  PlainKeys<KeyT> keys{key};
  hipLaunchKernelGGL((indptr_from_sorted_kernel<PlainKeys<KeyT>>),
                     dim3(blocks_for(num_keys + 1, kPtrCols)), dim3(kThreads), 0, st, keys, E,
                     num_keys, indptr);
}

// ------------------------------------------------------------ radix sort ----
// The sort moves ONE 64-bit word per edge: key above, position of the edge below
// (idx_bits = bits of the edge count).  Sorting the words is the stable sort of the keys,
// the low bits of the result are the permutation, and a pass reads and writes 8 bytes per
// edge instead of a widened key and a permutation entry each way.
constexpr int kRadixBits = 8;
constexpr int kRadix = 1 << kRadixBits;

__device__ __forceinline__ int digit_of(unsigned long long word, int shift) {
  return static_cast<int>((word >> shift) & (kRadix - 1));
}

// words of the first pass, made from the caller's keys on the fly (STREAM: read past the caches)
template <typename IdT, bool STREAM = false>
struct FreshWords {
  const IdT* key;
  int idx_bits;
  // word j of the tile that begins at `base`
  __device__ __forceinline__ unsigned long long operator()(int64_t base, uint32_t j) const {
    const IdT* p = key + base + j;
    const IdT k = STREAM ? __builtin_nontemporal_load(p) : *p;
    return (static_cast<unsigned long long>(k) << idx_bits) |
           static_cast<unsigned long long>(base + j);
  }
};
struct StoredWords {
  const unsigned long long* word;
  __device__ __forceinline__ unsigned long long operator()(int64_t base, uint32_t j) const {
    return (word + base)[j];
  }
};

// A tile of the sort.  Its items leave digit by digit, so a run is a 256th of the tile on
// average: the larger tile writes runs of 256 bytes where the smaller one writes 128, which
// is what the scatter waits for once there are enough tiles to fill the chip; with few
// tiles the smaller one spreads them over more compute units.
template <int THREADS, int PER_THREAD>
struct SortTile {
  static constexpr int kThreadsPerTile = THREADS;
  static constexpr int kPerThread = PER_THREAD;
  static constexpr int kSize = THREADS * PER_THREAD;
  static constexpr int kWaves = THREADS / kWave;
  static constexpr bool kStreams = THREADS > 256;  // reads past the caches (packed_pass_kernel)
};
using SmallTile = SortTile<256, 16>;
using LargeTile = SortTile<1024, 8>;
constexpr int64_t kLargeTileItems = int64_t(1) << 22;  // 512 large tiles: two for every compute unit

// counts[b * 256 + d] = items of tile b with digit d (a tile's side by side: digit by digit they were
// 437 k stores to as many lines for 14 M edges, 24 -> 19 us).  Four copies of the histogram, lane
// by lane in turn: on a skewed graph half a wave holds one digit, and additions to one LDS word
// queue up.
// What bounds it is the list's bytes.  Large tiles read it past the caches: a plain read of a list that the
// memory-side cache does not hold takes the place of lines there that were written last (the sort's own words) and
// waits for them to be written back: 112 MB 42 us plain, 20 so.  The first pass, which then found the list there, takes
// 81 for 62; the list loaded and sorted 379 -> 372.
constexpr int kHistCopies = 4;

template <typename T, typename Src, typename Count>
__global__ void __launch_bounds__(T::kThreadsPerTile)
radix_hist_kernel(Src src, int64_t E, int shift, Count* __restrict__ counts,
                  int* __restrict__ clear) {
  __shared__ int s_hist[kHistCopies][kRadix + 1];
  const int64_t base = static_cast<int64_t>(blockIdx.x) * T::kSize;
  const uint32_t n = E - base < T::kSize ? static_cast<uint32_t>(E - base) : T::kSize;
  unsigned long long word[T::kPerThread];
#pragma unroll
  for (int k = 0; k < T::kPerThread; ++k) {
    const uint32_t j = k * T::kThreadsPerTile + threadIdx.x;
    word[k] = src(base, j < n ? j : n - 1);
  }
  for (int j = threadIdx.x; j < kHistCopies * (kRadix + 1); j += T::kThreadsPerTile)
    (&s_hist[0][0])[j] = 0;
  if (clear && blockIdx.x == 0 && threadIdx.x < 2) clear[threadIdx.x] = 0;
  lds_barrier();  // (the words stay on their way)
#pragma unroll
  for (int k = 0; k < T::kPerThread; ++k) {
    const int d = k * T::kThreadsPerTile + threadIdx.x < n ? digit_of(word[k], shift) : kRadix;
    atomicAdd(&s_hist[threadIdx.x & (kHistCopies - 1)][d], 1);
  }
  __syncthreads();
  if (threadIdx.x < kRadix) {
    int n = 0;
#pragma unroll
    for (int c = 0; c < kHistCopies; ++c) n += s_hist[c][threadIdx.x];
    counts[static_cast<int64_t>(blockIdx.x) * kRadix + threadIdx.x] = n;
  }
}

// The same from the digits alone, a byte each (a multiple of eight can be read): eight a read.  14 M
// edges: 24 us from the words, 14 byte by byte, 13 so (8 with the counts of a tile side by side).
template <typename T>
__global__ void __launch_bounds__(T::kThreadsPerTile)
digit_hist_kernel(const unsigned char* __restrict__ digit, int64_t E, uint32_t* __restrict__ counts) {
  constexpr int kReads = T::kPerThread / 8;
  __shared__ int s_hist[kHistCopies][kRadix + 1];
  const int64_t base = static_cast<int64_t>(blockIdx.x) * T::kSize;
  const uint32_t n = E - base < T::kSize ? static_cast<uint32_t>(E - base) : T::kSize;
  unsigned long long eight[kReads];
#pragma unroll
  for (int k = 0; k < kReads; ++k) {
    const uint32_t j = (k * T::kThreadsPerTile + threadIdx.x) * 8;
    eight[k] = *reinterpret_cast<const unsigned long long*>(digit + base + (j < n ? j : 0u));
  }
  for (int j = threadIdx.x; j < kHistCopies * (kRadix + 1); j += T::kThreadsPerTile)
    (&s_hist[0][0])[j] = 0;
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kReads; ++k) {
    const uint32_t j = (k * T::kThreadsPerTile + threadIdx.x) * 8;
#pragma unroll
    for (int b = 0; b < 8; ++b)
      if (j + b < n)
        atomicAdd(&s_hist[threadIdx.x & (kHistCopies - 1)][static_cast<int>(eight[k] >> (8 * b)) & (kRadix - 1)], 1);
  }
  __syncthreads();
  if (threadIdx.x < kRadix) {
    int all = 0;
#pragma unroll
    for (int c = 0; c < kHistCopies; ++c) all += s_hist[c][threadIdx.x];
    counts[static_cast<int64_t>(blockIdx.x) * kRadix + threadIdx.x] = all;
  }
}

// Where a digit's items of a tile start among that digit's items (offsets[d * num_blocks + b]),
// and how many the digit has (totals): a workgroup a digit, 2048 tiles at a time.  What the digits
// below it hold, every workgroup of the pass adds up from the 256 totals by itself.  (One scan over
// the whole table, which that leaves out, is two launches: 1709 tiles 11 -> 5 us a pass.)  The digits
// whose counts share lines are one die's.
constexpr int kDigitThreads = 1024;
constexpr int kDigitItems = 2;

template <typename Count>
__global__ void __launch_bounds__(kDigitThreads)
digit_offsets_kernel(const Count* __restrict__ counts, int64_t num_blocks,
                     Count* __restrict__ offsets, int64_t* __restrict__ totals) {
  __shared__ int64_t s_scan[kDigitThreads / kWave + 1];
  const int digit = blockIdx.x % kXcds * (kRadix / kXcds) + blockIdx.x / kXcds;
  const int64_t row = static_cast<int64_t>(digit) * num_blocks;
  int64_t run = 0;
  for (int64_t t0 = 0; t0 < num_blocks; t0 += kDigitThreads * kDigitItems) {
    const int64_t t = t0 + threadIdx.x * kDigitItems;
    int64_t n[kDigitItems], mine = 0;
#pragma unroll
    for (int k = 0; k < kDigitItems; ++k)
      n[k] = static_cast<int64_t>(counts[(t + k < num_blocks ? t + k : 0) * kRadix + digit]);
#pragma unroll
    for (int k = 0; k < kDigitItems; ++k) {
      if (t + k >= num_blocks) n[k] = 0;
      mine += n[k];
    }
    int64_t all;
    int64_t at = run + block_exclusive_scan<kDigitThreads>(mine, &all, s_scan);
#pragma unroll
    for (int k = 0; k < kDigitItems; ++k) {
      if (t + k < num_blocks) offsets[row + t + k] = static_cast<Count>(at);
      at += n[k];
    }
    run += all;
  }
  if (threadIdx.x == 0) totals[digit] = run;
}

// where the last pass of the sort writes: the values in key order, the permutation, and
// the sorted keys themselves (for the offsets; null when nobody builds any)
template <typename IdT>
struct SortOutputs {
  IdT* value;
  int64_t* perm;
  uint32_t* key;
  int idx_bits;
  int* wide;  // [0]: raised when a 64-bit value does not fit 32 bits, [1]: gaps left (null: 32-bit values)
  bool stream;  // packed_pass_kernel: results as streams (kStreamResults)
  int64_t* indptr;  // packed_pass_kernel: the columns' offsets, from the tiles themselves (null: not here)
  int64_t num_keys;
  uint4* gaps;  // runs of columns of one offset that the last pass leaves to gap_fill_kernel: first, how many, offset
};

// One pass of the sort over one tile, stable.  A wave owns its share of the tile, in index
// order, and visits it 64 consecutive items at a time: the rank of an item among the equal
// digits of its round comes from 8 ballots, the count of the wave's earlier rounds from a
// small LDS table only that wave touches (no workgroup barrier per round).  One barrier
// later the digits' totals are scanned, every item knows its place in the tile's sorted
// order and goes there in LDS together with its value; the tile then leaves in that
// order, so that the items of a digit are written as one run -- coalesced stores, where a
// scatter straight from registers wrote 8 bytes here and 8 bytes there.
// The value rides along with its word from the first pass on (read in input order then), so
// no pass gathers it by position; the LAST pass writes values, permutation and keys instead
// of words.  64-bit values travel in their low 32 bits: ids of any graph that fits the card do,
// and a value that does not raises `wide`, on which widen_values_kernel fetches all of them
// again through the permutation.  14 M edges with 64-bit ids and 22-bit keys: 78 us the first pass
// (it reads the ids as they come), 67 and 82 the others; with the values inside the words
// (packed_pass_kernel) 67, 59 and 82.
// SELF: `offsets` holds the tiles' raw counts and every workgroup adds up for itself where its
// runs start (a sort of few tiles: a launch less per pass than scanning the counts first).
constexpr int64_t kSelfScanTiles = 64;
static_assert(kLargeTileItems / LargeTile::kSize > kSelfScanTiles, "large tiles never scan themselves");

template <typename T, typename IdT, typename ValT, typename Src, bool LAST, bool SELF>
__global__ void __launch_bounds__(T::kThreadsPerTile, T::kWaves == 16 ? 8 : 4)  // (what LDS allows)
radix_pass_kernel(Src src, const ValT* __restrict__ val_in, int64_t E, int shift,
                  int64_t num_blocks, const int64_t* __restrict__ offsets,
                  const int64_t* __restrict__ totals, unsigned long long* __restrict__ out,
                  uint32_t* __restrict__ val_out, SortOutputs<IdT> last) {
  constexpr int kThreadsHere = T::kThreadsPerTile, kItemsHere = T::kPerThread;
  __shared__ unsigned long long s_word[T::kSize];
  __shared__ int64_t s_base[kRadix];        // memory position of a digit's run minus its place in the tile
  __shared__ unsigned short s_cnt[T::kWaves][kRadix];  // per wave: count, then count of the earlier waves
  __shared__ int s_start[kRadix];           // where the run of a digit starts in the tile
  __shared__ int s_scan[kRadix / kWave];
  __shared__ int64_t s_digits[kRadix / kWave];
  __shared__ int64_t s_all[kRadix];         // a digit's items in all tiles, and in the tiles before this one
  // Consecutive tiles on one XCD (workgroup w runs on XCD w % 8): the runs of a digit that they
  // write lie side by side, and the line that two of them share is filled in one L2.  Load +
  // CSC of 14 M edges: 645 -> 623 us.
  const int64_t share = num_blocks / kXcds, more = num_blocks % kXcds, xcd = blockIdx.x % kXcds;
  const int64_t tile = xcd * share + (xcd < more ? xcd : more) + blockIdx.x / kXcds;
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x / kWave;
  const int digit = threadIdx.x;  // of the first 256 threads
  int64_t all = 0, before_tile = 0;
  if (digit < kRadix) {
    if (SELF) {
      for (int64_t b = 0; b < num_blocks; ++b) {
        const int64_t c = offsets[b * kRadix + digit];
        all += c;
        before_tile += b < tile ? c : 0;
      }
    } else {
      all = totals[digit];
      before_tile = offsets[static_cast<int64_t>(digit) * num_blocks + tile];
    }
  }
  for (int j = threadIdx.x; j < T::kWaves * kRadix / 2; j += kThreadsHere)
    reinterpret_cast<uint32_t*>(&s_cnt[0][0])[j] = 0u;
  const int64_t base = tile * T::kSize;
  // (indices clamped instead of reads left out: all of a thread's reads go out together; counted
  // from the tile's start, in 32 bits, so that they take one register each)
  const uint32_t n = E - base < T::kSize ? static_cast<uint32_t>(E - base) : T::kSize;
  const uint32_t mine0 = wave * (T::kSize / T::kWaves) + lane;
  unsigned long long word[kItemsHere];
#pragma unroll
  for (int r = 0; r < kItemsHere; ++r) {
    const uint32_t j = mine0 + r * kWave;
    word[r] = src(base, j < n ? j : n - 1);
  }
  // (what lies behind the last edge takes the last digit; it comes last in index order, so its
  // places are those behind the tile's live items and none of them is written out)
#pragma unroll
  for (int r = 0; r < kItemsHere; ++r)
    if (mine0 + r * kWave >= n) word[r] = ~0ull;
  if (digit < kRadix) {  // (out of the registers until the items are counted)
    s_all[digit] = all;
    s_base[digit] = before_tile;
  }
  __syncthreads();  // the tables are zero
  int place[kItemsHere];
#pragma unroll
  for (int r = 0; r < kItemsHere; ++r) {
    const int d = digit_of(word[r], shift);
    // lanes with this digit: per bit, the lanes whose bit equals this lane's (two instructions a
    // half-word, and-not-xor in one; sixty-four selects and masks a round bounded the pass before)
    uint32_t lo = ~0u, hi = ~0u;
#pragma unroll
    for (int b = 0; b < kRadixBits; ++b) {
      const int mine = static_cast<int>(static_cast<uint32_t>(d) << (31 - b)) >> 31;
      const unsigned long long bal = __ballot(mine);
      lo = __builtin_amdgcn_bitop3_b32(lo, static_cast<uint32_t>(bal), mine, 0x90);
      hi = __builtin_amdgcn_bitop3_b32(hi, static_cast<uint32_t>(bal >> 32), mine, 0x90);
    }
    const int rank = __builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, 0));
    const int before = s_cnt[wave][d];  // the wave's earlier rounds (LDS operations of a wave keep their order)
    place[r] = before + rank;
    if (rank == 0) s_cnt[wave][d] = static_cast<unsigned short>(before + __popc(lo) + __popc(hi));
  }
  // The values are asked for only now and needed behind the words' way out: on their way from the
  // start, they did not fit the registers beside the words, and every one was waited for and
  // set aside in memory before the next (14 M edges, 64-bit ids, with tiles of 1024 threads instead
  // of 512: first pass 102 -> 78 us, the others 72 -> 67 and 84 -> 82).
  ValT raw[kItemsHere];
  const ValT* __restrict__ tile_val = val_in + base;
  uint32_t again0 = mine0;  // (indices and digits made a second time rather than kept)
  asm volatile("" : "+v"(again0), "+s"(shift));
#pragma unroll
  for (int r = 0; r < kItemsHere; ++r) {
    const uint32_t j = again0 + r * kWave;
    raw[r] = tile_val[j < n ? j : n - 1];
  }
  __syncthreads();
  // digit by digit: counts of the waves -> counts of the earlier waves, total -> start; and where
  // the digit's items of this tile go, behind the smaller digits' of all tiles
  int total = 0, incl = 0;
  int64_t run_at = 0;
  if (digit < kRadix) {
    run_at = s_all[digit];
#pragma unroll
    for (int w = 0; w < T::kWaves; ++w) {
      const int c = s_cnt[w][digit];
      s_cnt[w][digit] = static_cast<unsigned short>(total);
      total += c;
    }
    incl = total;
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
      const int y = __shfl_up(incl, d, kWave);
      const int64_t z = __shfl_up(run_at, d, kWave);
      if (lane >= d) {
        incl += y;
        run_at += z;
      }
    }
    if (lane == kWave - 1) {
      s_scan[wave] = incl;
      s_digits[wave] = run_at;
    }
  }
  __syncthreads();
  if (digit < kRadix) {
    int start = incl - total;
    run_at += s_base[digit] - s_all[digit];
    for (int w = 0; w < wave; ++w) {
      start += s_scan[w];
      run_at += s_digits[w];
    }
    s_start[digit] = start;
    s_base[digit] = run_at - start;
  }
  __syncthreads();
  // (words first, then the values through the same LDS: half the footprint of staging both
  // at once, and twice the workgroups per compute unit)
#pragma unroll
  for (int r = 0; r < kItemsHere; ++r) {
    const int d = digit_of(word[r], shift);
    place[r] += s_start[d] + s_cnt[wave][d];
    s_word[place[r]] = word[r];
  }
  __syncthreads();
  int out_digit[kItemsHere];
#pragma unroll
  for (int k = 0; k < kItemsHere; ++k) {
    const uint32_t j = k * kThreadsHere + threadIdx.x;
    out_digit[k] = 0;
    if (j < n) {
      const unsigned long long w = s_word[j];
      out_digit[k] = digit_of(w, shift);
      const int64_t dst = s_base[out_digit[k]] + j;
      if (LAST) {
        last.perm[dst] = static_cast<int64_t>(w & ((1ull << last.idx_bits) - 1ull));
        if (last.key) last.key[dst] = static_cast<uint32_t>(w >> last.idx_bits);
      } else {
        out[dst] = w;
      }
    }
  }
  bool wide = false;
#pragma unroll
  for (int r = 0; r < kItemsHere; ++r)
    if (sizeof(ValT) == 8) wide |= static_cast<uint64_t>(raw[r]) != static_cast<uint32_t>(raw[r]);
  if (sizeof(ValT) == 8 && wide) *last.wide = 1;
  __syncthreads();
  uint32_t* s_val = reinterpret_cast<uint32_t*>(s_word);
#pragma unroll
  for (int r = 0; r < kItemsHere; ++r) s_val[place[r]] = static_cast<uint32_t>(raw[r]);
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kItemsHere; ++k) {
    const uint32_t j = k * kThreadsHere + threadIdx.x;
    if (j < n) {
      const int64_t dst = s_base[out_digit[k]] + j;
      if (LAST)
        last.value[dst] = static_cast<IdT>(s_val[j]);
      else
        val_out[dst] = s_val[j];
    }
  }
}

// The same with the value INSIDE the word, which then is all that a pass moves: what is left of the
// key, then the value, then the position of the edge.  The word of a pass does not
// hold the digit that the pass sorted by: the next pass knows it from where it finds the word
// (the digits' totals) and puts it in the place of its own, so that a key of three digits
// needs room for two, and one of two for one.  A value that does not fit the bits that are left raises
// `wide`.  The next pass's digits are written beside the words, for its histogram to read a byte an edge.
// 14 M edges, 22-bit keys (24 bits each for value and position): the passes 72 + 65 + 82 us with the
// values beside the words, 67 + 59 + 81 so; the last two histograms 24 -> 8 each.
// What a pass of large tiles reads, nothing reads again before it has left the caches, so it reads past them (14 M
// edges with 64-bit ids, loaded and sorted: 420 -> 415 us; 11 M / 8 M with 32-bit ids 322 -> 301, 290 -> 277).  Up to
// 4 M edges (small tiles) the lists and the words stay in the L2s, plain / past the caches, lists loaded and sorted again
// and again: 2.3 M edges, 64-bit ids 136/140 us, 4.0 M 183/189, 32-bit ids 174/178; 6.1 M 223/208, 193/191.
// The words it writes are the next
// pass's: written past the caches they cost 456.  The last pass's results go past them where they
// fill more than half of the memory-side cache (14 M: 415 -> 404, 11 M: 301 -> 290; 8 M, 128 MB: 277, 278).
// The last pass leaves the columns' offsets too where edges are many for the columns (coo2csc_impl): it holds a tile in key order, and
// the keys that it wrote for a launch behind the sort to read back were 112 of the 1500 MB that a list of 14 M edges
// moves: that pass 84 -> 85 us, the launch behind it, 19, gone; the list loaded and sorted 392 -> 379.
constexpr int kPackedPasses = 3;
constexpr uint32_t kWideTile = 16;  // offsets a thread beyond which a tile has long gaps
// There a tile goes by its items: one item's columns, those from the item before on, have one offset.  Up to kGapLane of
// them its lane stores, up to kGapHere its wave together, and more are left to a launch behind the sort in pieces of
// kGapPiece: the columns above the last lower digit in use are all one tile's, 2.4 M of them where the lower 16 bits of
// 2.45 M ids stay below 100.  Sorts of such lists and of ids whose lower bits are 30000 to 30004, us, by written keys / by
// one workgroup with a search a column / so: 14 M edges 340/534/293 and 328/1080/288, 5 M 183/673/162 and 170/1440/155.
// With two digits no item has more than 256 columns, and a launch that finds nothing would be 2 us of 25 to 40.
constexpr int64_t kThreeDigitItems = 1'300'000;  // edges from which small tiles' last pass of three leaves the offsets
constexpr int kGapBlocks = 512;
constexpr uint32_t kGapLane = 4, kGapHere = 128, kGapPiece = 2048;
constexpr int64_t kStreamResults = int64_t(1) << 27;  // bytes
constexpr int rest_at(int passes) { return 64 - kRadixBits * (passes - 1); }  // of the key's digits in a word

template <typename T, typename IdT, int PASSES, int PASS>
__global__ void __launch_bounds__(T::kThreadsPerTile, T::kWaves == 16 ? 8 : 4)  // (what LDS allows)
packed_pass_kernel(const IdT* __restrict__ key, const IdT* __restrict__ value,
                   const unsigned long long* __restrict__ in, int64_t E, int value_bits,
                   int64_t num_blocks, const uint32_t* __restrict__ offsets,
                   const int64_t* __restrict__ totals, const int64_t* __restrict__ totals_before,
                   unsigned long long* __restrict__ out, unsigned char* __restrict__ next_digit,
                   SortOutputs<IdT> last) {
  constexpr int kThreadsHere = T::kThreadsPerTile, kItemsHere = T::kPerThread;
  constexpr bool FIRST = PASS == 0, LAST = PASS == PASSES - 1;
  constexpr int kRestAt = rest_at(PASSES);
  constexpr int kCountBytes = T::kWaves * kRadix * 2;
  __shared__ unsigned long long s_word[T::kSize];
  __shared__ int64_t s_base[kRadix];  // memory position of a digit's run minus its place in the tile
  __shared__ int64_t s_all[kRadix];
  // per wave: count, then count of the earlier waves; and when every item has its place, the
  // digits in the tile's sorted order
  __shared__ __attribute__((aligned(16))) unsigned char
      s_shared[kCountBytes > T::kSize ? kCountBytes : T::kSize];
  __shared__ int s_start[kRadix];     // where the run of a digit starts in the tile
  __shared__ uint32_t s_bound[kRadix];  // where the items of a digit of the pass before end
  __shared__ int s_scan[kRadix / kWave];
  __shared__ uint32_t s_ends[kRadix / kWave];
  __shared__ int64_t s_digits[kRadix / kWave];
  __shared__ uint32_t s_lows[2];  // LAST: the tile's lower digits, from and to (offsets below)
  unsigned short (*s_cnt)[kRadix] = reinterpret_cast<unsigned short (*)[kRadix]>(s_shared);
  unsigned char* s_dig = s_shared;
  // consecutive tiles on one XCD, as above
  const int64_t share = num_blocks / kXcds, more = num_blocks % kXcds, xcd = blockIdx.x % kXcds;
  const int64_t tile = xcd * share + (xcd < more ? xcd : more) + blockIdx.x / kXcds;
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x / kWave;
  const int digit = threadIdx.x;  // of the first 256 threads
  // (a value that did not fit its bits, met by the first pass: they are all fetched again)
  const bool refetch = LAST && *last.wide != 0;
  auto once = [](const auto* p) { return T::kStreams ? __builtin_nontemporal_load(p) : *p; };
  int64_t all = 0, before_tile = 0;
  uint32_t ends = 0;
  if (digit < kRadix) {
    all = totals[digit];
    before_tile = offsets[static_cast<int64_t>(digit) * num_blocks + tile];
    if (!FIRST) ends = static_cast<uint32_t>(totals_before[digit]);
  }
  for (int j = threadIdx.x; j < kCountBytes / 4; j += kThreadsHere)
    reinterpret_cast<uint32_t*>(s_shared)[j] = 0u;
  const int64_t base = tile * T::kSize;
  const uint32_t n = E - base < T::kSize ? static_cast<uint32_t>(E - base) : T::kSize;
  const uint32_t mine0 = wave * (T::kSize / T::kWaves) + lane;
  uint32_t fresh[FIRST ? kItemsHere : 1];
  unsigned long long word[FIRST ? 1 : kItemsHere];
#pragma unroll
  for (int r = 0; r < kItemsHere; ++r) {
    const uint32_t j = mine0 + r * kWave;
    if constexpr (FIRST)
      fresh[r] = static_cast<uint32_t>(once(key + base + (j < n ? j : n - 1)));
    else
      word[r] = once(in + base + (j < n ? j : n - 1));
  }
  unsigned long long ahead = 0;  // the word in front of the tile
  if constexpr (LAST) ahead = in[tile > 0 ? base - 1 : 0];
  // (what lies behind the last edge takes the last digit, as above)
#pragma unroll
  for (int r = 0; r < kItemsHere; ++r) {
    if (mine0 + r * kWave >= n) {
      if constexpr (FIRST) fresh[r] = ~0u; else word[r] = ~0ull;
    }
  }
  if (digit < kRadix) {
    s_all[digit] = all;
    s_base[digit] = before_tile;
    if (!FIRST) {
#pragma unroll
      for (int d = 1; d < kWave; d <<= 1) {
        const uint32_t y = __shfl_up(ends, d, kWave);
        if (lane >= d) ends += y;
      }
      s_bound[digit] = ends;
      if (lane == kWave - 1) s_ends[wave] = ends;
    }
  }
  lds_barrier();  // the tables are zero
  auto digit_here = [&](int r) {
    if constexpr (FIRST)
      return static_cast<int>(fresh[r] & (kRadix - 1));
    else
      return static_cast<int>(word[r] >> (kRestAt + kRadixBits * (PASS - 1))) & (kRadix - 1);
  };
  int place[kItemsHere];
#pragma unroll
  for (int r = 0; r < kItemsHere; ++r) {
    const int d = digit_here(r);
    uint32_t lo = ~0u, hi = ~0u;  // lanes with this digit, as above
#pragma unroll
    for (int b = 0; b < kRadixBits; ++b) {
      const int mine = static_cast<int>(static_cast<uint32_t>(d) << (31 - b)) >> 31;
      const unsigned long long bal = __ballot(mine);
      lo = __builtin_amdgcn_bitop3_b32(lo, static_cast<uint32_t>(bal), mine, 0x90);
      hi = __builtin_amdgcn_bitop3_b32(hi, static_cast<uint32_t>(bal >> 32), mine, 0x90);
    }
    const int rank = __builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, 0));
    const int before = s_cnt[wave][d];  // the wave's earlier rounds (LDS operations of a wave keep their order)
    place[r] = before + rank;
    if (rank == 0) s_cnt[wave][d] = static_cast<unsigned short>(before + __popc(lo) + __popc(hi));
  }
  IdT raw[FIRST ? kItemsHere : 1];
  if constexpr (FIRST) {  // the values, asked for behind the ranking: see above
    const IdT* __restrict__ tile_val = value + base;
    uint32_t again0 = mine0;
    asm volatile("" : "+v"(again0));
#pragma unroll
    for (int r = 0; r < kItemsHere; ++r) {
      const uint32_t j = again0 + r * kWave;
      raw[r] = once(tile_val + (j < n ? j : n - 1));
    }
  }
  lds_barrier();
  int total = 0, incl = 0;
  int64_t run_at = 0;
  if (digit < kRadix) {
    run_at = s_all[digit];
    if (!FIRST)
      for (int w = 0; w < wave; ++w) ends += s_ends[w];
#pragma unroll
    for (int w = 0; w < T::kWaves; ++w) {
      const int c = s_cnt[w][digit];
      s_cnt[w][digit] = static_cast<unsigned short>(total);
      total += c;
    }
    incl = total;
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
      const int y = __shfl_up(incl, d, kWave);
      const int64_t z = __shfl_up(run_at, d, kWave);
      if (lane >= d) {
        incl += y;
        run_at += z;
      }
    }
    if (lane == kWave - 1) {
      s_scan[wave] = incl;
      s_digits[wave] = run_at;
    }
  }
  lds_barrier();
  if (digit < kRadix) {
    int start = incl - total;
    run_at += s_base[digit] - s_all[digit];
    for (int w = 0; w < wave; ++w) {
      start += s_scan[w];
      run_at += s_digits[w];
    }
    s_start[digit] = start;
    s_base[digit] = run_at - start;
    if (!FIRST) s_bound[digit] = ends;
  }
  lds_barrier();
#pragma unroll
  for (int r = 0; r < kItemsHere; ++r) {
    const int d = digit_here(r);
    place[r] += s_start[d] + s_cnt[wave][d];
  }
  // the digit of the pass before at the thread's first item; its later ones lie behind
  int was = 0;
  auto digit_before = [&](uint32_t at) {
    int d = 0;
#pragma unroll
    for (int step = kRadix / 2; step > 0; step >>= 1)
      if (s_bound[d + step - 1] <= at) d += step;
    return d;
  };
  constexpr int kAt = kRestAt + kRadixBits * (PASS - 1);  // this pass's digit (not of the first)
  auto with_digit_before = [](unsigned long long w, int d) {
    return (w & ~(static_cast<unsigned long long>(kRadix - 1) << kAt)) |
           static_cast<unsigned long long>(d) << kAt;
  };
  if constexpr (!FIRST) was = digit_before(static_cast<uint32_t>(base) + mine0);
  if constexpr (LAST) {
    if (last.indptr && threadIdx.x == 0) {
      uint32_t from = 0;
      if (tile > 0)
        from = static_cast<uint32_t>(with_digit_before(ahead, digit_before(static_cast<uint32_t>(base) - 1)) >>
                                     kRestAt) + 1;
      s_lows[0] = from;
    }
  }
  lds_barrier();  // (the counts make room for the digits)
  bool wide = false;
  uint32_t third0 = mine0;  // (indices made once more rather than kept)
  asm volatile("" : "+v"(third0));
#pragma unroll
  for (int r = 0; r < kItemsHere; ++r) {
    const uint32_t j = third0 + r * kWave;
    const int d = digit_here(r);
    unsigned long long w;
    if constexpr (FIRST) {
      const unsigned long long v = static_cast<unsigned long long>(raw[r]);
      wide |= (v >> value_bits) != 0ull;
      w = static_cast<unsigned long long>(fresh[r] >> kRadixBits) << kRestAt |
          (v & ((1ull << value_bits) - 1ull)) << (kRestAt - value_bits) | static_cast<uint32_t>(base + j);
    } else {
      const uint32_t at = static_cast<uint32_t>(base) + j;
      while (was < kRadix - 1 && s_bound[was] <= at) ++was;
      w = with_digit_before(word[r], was);
      if (LAST && j == n - 1)
        s_lows[1] = base + n == E ? 1u << (kRadixBits * PASS) : static_cast<uint32_t>(w >> kRestAt) + 1;
    }
    s_word[place[r]] = w;
    s_dig[place[r]] = static_cast<unsigned char>(d);
  }
  if (FIRST && wide) *last.wide = 1;  // (the last edge's value again past the end)
  lds_barrier();
#pragma unroll
  for (int k = 0; k < kItemsHere; ++k) {
    const uint32_t j = k * kThreadsHere + threadIdx.x;
    if (j < n) {
      const unsigned long long w = s_word[j];
      const uint32_t d = s_dig[j];
      const int64_t dst = s_base[d] + j;
      if (LAST) {
        const int64_t from = static_cast<int64_t>(w & ((1ull << (kRestAt - value_bits)) - 1ull));
        IdT v = static_cast<IdT>((w & ((1ull << kRestAt) - 1ull)) >> (kRestAt - value_bits));
        if (refetch) v = value[from];
        if (last.stream) {
          __builtin_nontemporal_store(from, last.perm + dst);
          __builtin_nontemporal_store(v, last.value + dst);
        } else {
          last.perm[dst] = from;
          last.value[dst] = v;
        }
        if (last.key)
          last.key[dst] = d << (kRadixBits * PASS) | static_cast<uint32_t>(w >> kRestAt);
      } else {
        out[dst] = w;
        next_digit[dst] = static_cast<unsigned char>(w >> (kRestAt + kRadixBits * PASS));
      }
    }
  }
  // The offsets of the columns whose lower digits begin in this tile, whatever their last digit: all
  // edges with lower digits below come before the tile's or lie in it, so the offset is the place of the
  // digit's first edge that is not below.  Every column is one tile's, with or without edges.
  if constexpr (LAST) {
    if (!last.indptr) return;
    constexpr int kLowBits = kRadixBits * PASS;
    const uint32_t from = s_lows[0], lows = s_lows[1] - from;
    const int64_t most = (last.num_keys >> kLowBits) + 1;  // (offset num_keys among them)
    const uint32_t digits = most < kRadix ? static_cast<uint32_t>(most) : kRadix;
    auto leave = [&](uint32_t d, uint32_t low, uint32_t lo, uint32_t hi) {
      const int64_t c = static_cast<int64_t>(d) << kLowBits | low;
      if (c > last.num_keys) return;
      while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        if (static_cast<uint32_t>(s_word[mid] >> kRestAt) < low) lo = mid + 1; else hi = mid;
      }
      last.indptr[c] = s_base[d] + lo;
    };
    auto run_end = [&](uint32_t d) -> uint32_t { return d == kRadix - 1 ? n : s_start[d + 1]; };
    if (lows * digits <= kWideTile * kThreadsHere) {
      for (uint32_t i = threadIdx.x; i < lows * digits; i += kThreadsHere) {
        const uint32_t d = i / lows;
        leave(d, from + i % lows, s_start[d], run_end(d));
      }
    } else {  // long gaps: by items, and what lies behind a digit's last one
      constexpr uint32_t kHere = kLowBits == kRadixBits ? uint32_t(kRadix) : kGapHere;  // (with two digits none is longer)
      for (uint32_t u0 = wave * kWave; u0 < n + digits; u0 += kThreadsHere) {
        const uint32_t u = u0 + lane;
        uint32_t first = 0, count = 0, offset = 0;
        if (u < n + digits) {
          const uint32_t d = u < n ? s_dig[u] : u - n;
          const uint32_t j = u < n ? u : run_end(d);
          const uint32_t begin = j > static_cast<uint32_t>(s_start[d]) ? static_cast<uint32_t>(s_word[j - 1] >> kRestAt) + 1 : from;
          const uint32_t end = u < n ? static_cast<uint32_t>(s_word[u] >> kRestAt) + 1 : from + lows;
          first = (d << kLowBits) + begin;
          const uint32_t most_here = static_cast<uint32_t>(last.num_keys) + 1;
          if (first < most_here) count = (end < most_here - first + begin ? end : most_here - first + begin) - begin;
          offset = static_cast<uint32_t>(s_base[d] + j);
        }
        if (count <= kGapLane) {
          for (uint32_t k = 0; k < count; ++k) last.indptr[first + k] = offset;
        } else if (count > kHere) {
          uint32_t at = atomicAdd(last.wide + 1, (count + kGapPiece - 1) / kGapPiece);
          for (uint32_t k = 0; k < count; k += kGapPiece, ++at)
            last.gaps[at] = make_uint4(first + k, count - k < kGapPiece ? count - k : kGapPiece, offset, 0u);
        }
        for (unsigned long long some = __ballot(count > kGapLane && count <= kHere); some; some &= some - 1) {
          const int from_lane = __builtin_ctzll(some);
          const uint32_t f = __builtin_amdgcn_readlane(first, from_lane), c = __builtin_amdgcn_readlane(count, from_lane);
          const uint32_t o = __builtin_amdgcn_readlane(offset, from_lane);
          for (uint32_t k = lane; k < c; k += kWave) last.indptr[f + k] = o;
        }
      }
    }
    if (threadIdx.x == 0 && base + n == E && last.num_keys >> kLowBits == kRadix) last.indptr[last.num_keys] = E;
  }
}

// The long gaps of the columns' offsets, a wave a piece.
__global__ void __launch_bounds__(kThreads)
gap_fill_kernel(const uint4* __restrict__ gaps, const int* __restrict__ num_gaps, int64_t* __restrict__ indptr) {
  const int n = *num_gaps, lane = threadIdx.x & (kWave - 1);
  for (int g = blockIdx.x * (kThreads / kWave) + threadIdx.x / kWave; g < n; g += gridDim.x * (kThreads / kWave)) {
    const uint4 gap = gaps[g];
    for (uint32_t k = lane; k < gap.y; k += kWave) indptr[gap.x + k] = gap.z;
  }
}

// Behind a sort with the values beside the words: fetches them all again when one did not fit 32 bits.
template <typename IdT>
__global__ void __launch_bounds__(kThreads)
widen_values_kernel(const IdT* __restrict__ value, const int64_t* __restrict__ perm, int64_t E,
                    const int* __restrict__ wide, IdT* __restrict__ out) {
  if (*wide == 0) return;
  const int64_t stride = static_cast<int64_t>(gridDim.x) * kThreads;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x; i < E; i += stride)
    out[i] = value[perm[i]];
}

int bits_for(int64_t n) {  // smallest b with 2^b >= n
  int bits = 0;
  while ((int64_t(1) << bits) < n) ++bits;
  return bits;
}

int num_passes(int64_t num_keys) {
  return (bits_for(num_keys) + kRadixBits - 1) / kRadixBits;  // format_transform.cu:58-72
}

// Offsets of B consecutive column ranges, each re-based to start at 0 and laid
// out one after the other (batch b: offsets[b+1]-offsets[b]+1 entries starting
// at offsets[b] + b).  One output entry per lane, batch by binary search -- over a
// copy of the batch offsets in LDS when there are at most 1023 batches, so that only
// the two reads of indptr go to memory.
constexpr int kSplitStage = 1024;

__global__ void __launch_bounds__(kThreads)
indptr_split_kernel(const int64_t* __restrict__ indptr, const int64_t* __restrict__ offsets,
                    int64_t B, int64_t total, int64_t* __restrict__ out,
                    int64_t* __restrict__ cuts) {
  __shared__ int64_t s_off[kSplitStage];
  const bool staged = B <= kSplitStage;
  if (staged) {
    for (int64_t b = threadIdx.x; b < B; b += kThreads) s_off[b] = offsets[b];
    __syncthreads();
  }
  const int64_t* off = staged ? s_off : offsets;
  const int64_t q = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
  // where every batch's entries start (and the last one's end), for the caller's next cut
  if (cuts && q <= B) cuts[q] = indptr[offsets[q]];
  if (q >= total) return;
  int64_t lo = 0, hi = B - 1;  // last b with offsets[b] + b <= q
  while (lo < hi) {
    const int64_t mid = (lo + hi + 1) >> 1;
    if (off[mid] + mid <= q) lo = mid; else hi = mid - 1;
  }
  const int64_t begin = off[lo];
  out[q] = indptr[begin + (q - begin - lo)] - indptr[begin];
}

template <typename T, typename IdT, typename ValT, typename Src>
void launch_pass(Src src, bool last, bool self, hipStream_t st, const ValT* vin, int64_t E, int shift,
                 int64_t blocks, const int64_t* where, const int64_t* totals,
                 unsigned long long* wout, uint32_t* vout, const SortOutputs<IdT>& outs) {
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(blocks)), dim3(T::kThreadsPerTile), 0, st,
                       src, vin, E, shift, blocks, where, totals, wout, vout, outs);
  };
  if constexpr (std::is_same<T, SmallTile>::value) {  // (a sort by large tiles has 512 at least)
    if (self) {
      if (last) go(radix_pass_kernel<T, IdT, ValT, Src, true, true>);
      else go(radix_pass_kernel<T, IdT, ValT, Src, false, true>);
      return;
    }
  }
  if (last) go(radix_pass_kernel<T, IdT, ValT, Src, true, false>);
  else go(radix_pass_kernel<T, IdT, ValT, Src, false, false>);
}

// the sort's scratch memory
struct SortSpace {
  unsigned long long* word[2];
  uint32_t* value[2];
  int64_t *counts, *offsets, *totals, *totals_before;
  uint32_t* keys;
  int* wide;  // [2]
};
// (tables sized for the smaller tile, which has the larger ones)
inline size_t sort_space_bytes(int64_t E) {
  const int64_t table = kRadix * static_cast<int64_t>(blocks_for(E, SmallTile::kSize));
  const size_t n = static_cast<size_t>(E > 0 ? E : 1);
  return 2 * padded(n * 8) + 3 * padded(n * 4) + 2 * padded(static_cast<size_t>(table) * 8) +
         2 * padded(kRadix * 8) + 256;
}
inline bool carve_sort(Carver& ws, int64_t E, SortSpace* s) {
  const int64_t table = kRadix * static_cast<int64_t>(blocks_for(E, SmallTile::kSize));
  const size_t n = static_cast<size_t>(E > 0 ? E : 1);
  for (auto& w : s->word) w = ws.take<unsigned long long>(n);
  for (auto& v : s->value) v = ws.take<uint32_t>(n);
  s->keys = ws.take<uint32_t>(n);
  s->counts = ws.take<int64_t>(static_cast<size_t>(table));
  s->offsets = ws.take<int64_t>(static_cast<size_t>(table));
  s->totals = ws.take<int64_t>(kRadix);
  s->totals_before = ws.take<int64_t>(kRadix);
  s->wide = ws.take<int>(2);
  return ws.ok;
}

template <typename T, typename IdT>
int sort_passes(const IdT* key, const IdT* value, int64_t E, int passes, int idx_bits,
                const SortSpace& s, const SortOutputs<IdT>& outs, hipStream_t st) {
  const int64_t blocks = blocks_for(E, T::kSize);
  const dim3 grid(static_cast<unsigned>(blocks));
  const bool self = blocks <= kSelfScanTiles;
  const int64_t* where = self ? s.counts : s.offsets;
  for (int p = 0; p < passes; ++p) {
    const int shift = idx_bits + p * kRadixBits;
    const bool last = p == passes - 1;
    const FreshWords<IdT> fresh{key, idx_bits};
    const StoredWords stored{s.word[(p + 1) & 1]};
    if (p == 0)
      hipLaunchKernelGGL((radix_hist_kernel<T, FreshWords<IdT>, int64_t>), grid, dim3(T::kThreadsPerTile), 0,
                         st, fresh, E, shift, s.counts, outs.wide);
    else
      hipLaunchKernelGGL((radix_hist_kernel<T, StoredWords, int64_t>), grid, dim3(T::kThreadsPerTile), 0, st,
                         stored, E, shift, s.counts, static_cast<int*>(nullptr));
    if (!self)
      hipLaunchKernelGGL(digit_offsets_kernel<int64_t>, dim3(kRadix), dim3(kDigitThreads), 0, st, s.counts,
                         blocks, s.offsets, s.totals);
    if (p == 0)
      launch_pass<T>(fresh, last, self, st, value, E, shift, blocks, where, s.totals, s.word[0],
                     s.value[0], outs);
    else
      launch_pass<T>(stored, last, self, st, static_cast<const uint32_t*>(s.value[(p + 1) & 1]), E,
                     shift, blocks, where, s.totals, s.word[p & 1], s.value[p & 1], outs);
  }
  return check_launch("coo2csc");
}

// Bits of a value in the words of a sort; 0: not packed (few tiles, one pass or more than three, or too
// few bits for the values, which are expected below num_values).  A value that does not fit after all costs the
// last pass a gather of all of them by their positions: 14 M edges, 2.45 M keys, 64-bit ids up to 100 M 552 us
// where ids that fit take 312 (32-bit ids 512, 262; gathered by a launch behind the sort 587, 532).
inline int packed_value_bits(int64_t E, int64_t num_values, int passes, int64_t tiles) {
  if (passes < 2 || passes > kPackedPasses || E >= (int64_t(1) << 32) || tiles <= kSelfScanTiles) return 0;
  const int left = rest_at(passes) - bits_for(E), bits = left < 32 ? left : 32;
  return bits >= bits_for(num_values) ? bits : 0;
}

template <typename T, typename IdT>
int packed_passes(const IdT* key, const IdT* value, int64_t E, int passes, int value_bits,
                  const SortSpace& s, const SortOutputs<IdT>& outs, hipStream_t st) {
  const int64_t blocks = blocks_for(E, T::kSize);
  const dim3 grid(static_cast<unsigned>(blocks)), threads(T::kThreadsPerTile);
  const int idx_bits = bits_for(E);
  unsigned char* digits = reinterpret_cast<unsigned char*>(s.value[0]);  // (the values have no place of their own)
  uint32_t* counts = reinterpret_cast<uint32_t*>(s.counts);    // (fewer than 2^32 edges: half the tables' size)
  uint32_t* offsets = reinterpret_cast<uint32_t*>(s.offsets);
  for (int p = 0; p < passes; ++p) {
    const bool last = p == passes - 1;
    const unsigned long long* in = s.word[(p + 1) & 1];
    if (p == 0)
      hipLaunchKernelGGL((radix_hist_kernel<T, FreshWords<IdT, T::kStreams>, uint32_t>), grid, threads, 0, st,
                         FreshWords<IdT, T::kStreams>{key, idx_bits}, E, idx_bits, counts, outs.wide);
    else
      hipLaunchKernelGGL(digit_hist_kernel<T>, grid, threads, 0, st, digits, E, counts);
    int64_t* totals = p & 1 ? s.totals_before : s.totals;
    const int64_t* totals_before = p & 1 ? s.totals : s.totals_before;
    hipLaunchKernelGGL(digit_offsets_kernel<uint32_t>, dim3(kRadix), dim3(kDigitThreads), 0, st, counts, blocks,
                       offsets, totals);
    const auto kernel = passes == 2 ? (last ? packed_pass_kernel<T, IdT, 2, 1> : packed_pass_kernel<T, IdT, 2, 0>)
                        : p == 0 ? packed_pass_kernel<T, IdT, 3, 0>
                        : last ? packed_pass_kernel<T, IdT, 3, 2>
                               : packed_pass_kernel<T, IdT, 3, 1>;
    hipLaunchKernelGGL(kernel, grid, threads, 0, st, key, value, in, E, value_bits, blocks, offsets,
                       totals, totals_before, s.word[p & 1], digits, outs);
  }
  return check_launch("coo2csc");
}

template <typename IdT>
int coo2csc_impl(const IdT* key, const IdT* value, int64_t E, int64_t num_keys, int64_t num_values, int sorted,
                 int64_t* indptr, IdT* out_value, int64_t* perm, void* workspace,
                 size_t workspace_bytes, hipStream_t st) {
  if (E == 0 && !indptr) return GS_OK;
  if (sorted || E == 0) {
    launch_indptr(key, E, num_keys, indptr, st);
    return check_launch("coo2csc");
  }
  const int idx_bits = bits_for(E);
  int passes = num_passes(num_keys);
  if (passes == 0) passes = 1;  // one key: still produces perm = identity
  if (idx_bits + passes * kRadixBits > 64) {
    set_error_text("gs_coo2csc: %lld edges with keys below %lld do not fit the sort's 64-bit words",
                   static_cast<long long>(E), static_cast<long long>(num_keys));
    return GS_ERR_UNSUPPORTED;
  }
  Carver ws(workspace, workspace_bytes);
  SortSpace s;
  if (!carve_sort(ws, E, &s)) {
    set_error_text("gs_coo2csc: workspace needs %zu bytes, 256-byte aligned",
                   gs_coo2csc_workspace_bytes(E, num_keys));
    return GS_ERR_WORKSPACE;
  }
  const bool large = E >= kLargeTileItems;
  const int value_bits =
      packed_value_bits(E, num_values, passes, blocks_for(E, large ? LargeTile::kSize : SmallTile::kSize));
  const bool may_be_wide = sizeof(IdT) == 8 || value_bits > 0;
  const bool short_keys = passes * kRadixBits <= 32;
  // (offsets by the last pass's tiles; written keys and a launch of their own / so, us: 14 M edges, 2.45 M columns 301/270,
  // 20 k 178/157, the first of 2.45 M has all 626/302; 5 M, 5 M 150/139; small tiles: 300 k edges, 60 k columns 39/37, 1 M,
  // 20 k 45/41, 1.5 M, 375 k 74/71, 3 M, 750 k 91/84, but 1 M, 1 M 66/73 and 300 k, 300 k 58/67, a few tiles' searches, and
  // with three digits 300 k, 75 k 56/57, 1 M, 250 k 64/66, 32-bit ids, 1.25 M, 312 k 72/70 and 73/73, too few tiles)
  const bool by_tiles = indptr && value_bits > 0 &&
                        (large ? num_keys <= E : 4 * num_keys <= E && (passes == 2 || E >= kThreeDigitItems));
  const bool by_keys = indptr && short_keys && !by_tiles;
  const SortOutputs<IdT> outs{out_value, perm, by_keys ? s.keys : nullptr, idx_bits,
                              may_be_wide ? s.wide : nullptr,
                              E * static_cast<int64_t>(sizeof(int64_t) + sizeof(IdT) + sizeof(uint32_t)) >= kStreamResults,
                              by_tiles ? indptr : nullptr, num_keys, reinterpret_cast<uint4*>(s.keys)};
  // (a gap is of more than kGapHere columns, of which there are no more than edges)
  static_assert(kGapPiece >= kGapHere && 2 * sizeof(uint4) <= kGapHere * sizeof(uint32_t), "gaps fit in place of the keys");
  if (value_bits > 0) {
    const auto sort = large ? packed_passes<LargeTile, IdT> : packed_passes<SmallTile, IdT>;
    GS_RETURN_IF_ERROR(sort(key, value, E, passes, value_bits, s, outs, st));
  } else {
    const auto sort = large ? sort_passes<LargeTile, IdT> : sort_passes<SmallTile, IdT>;
    GS_RETURN_IF_ERROR(sort(key, value, E, passes, idx_bits, s, outs, st));
  }
  if (may_be_wide && value_bits == 0)  // (words with the value inside: the last pass does it)
    hipLaunchKernelGGL(widen_values_kernel<IdT>, dim3(E < (int64_t(1) << 20) ? 64 : 1024),
                       dim3(kThreads), 0, st, value, perm, E, s.wide, out_value);
  if (by_keys)  // (null: the caller wants the sorted order only)
    launch_indptr(static_cast<const uint32_t*>(s.keys), E, num_keys, indptr, st);
  else if (by_tiles && passes > 2)
    hipLaunchKernelGGL(gap_fill_kernel, dim3(kGapBlocks), dim3(kThreads), 0, st, outs.gaps, s.wide + 1, indptr);
  else if (indptr && !by_tiles)
    hipLaunchKernelGGL((indptr_from_sorted_kernel<PermutedKeys<IdT>>),
                       dim3(blocks_for(num_keys + 1, kPtrCols)), dim3(kThreads), 0, st,
                       PermutedKeys<IdT>{key, perm}, E, num_keys, indptr);
  return check_launch("coo2csc");
}

// -------------------------------------------------- distinct ids of an edge list ----
// The larger number of different ids that the two ends of an edge list hold (the node count of
// Graph::LoadCOO, reference src/graph.cc:25-35, which sorts both ends for it): a byte per
// possible id, set by a plain store of every edge that finds it clear, then the bytes are
// counted.  Ids run from zero in practice, so `range` bytes -- about one per edge -- hold
// them; an id outside is reported and the caller counts another way.  The first end is
// counted while the second is only looked through for its largest id: when the first holds
// every id up to the largest of both, the second cannot hold more and its own count is left
// out (any list with self loops).  What bounds the marking is one request to the L2 per edge
// and the lines that every die fetches again after another's stores: 180 us of 220 for 14 M
// edges with 64-bit ids, so lists from 4 M edges on go by bits in LDS (below).
constexpr int kMarkItems = 16;
constexpr int kMarkTile = kThreads * kMarkItems;
constexpr int kCountBlocks = 128;

struct DistinctSpace {
  unsigned char* map;  // range bytes for the first end, then for the second
  int64_t* largest;    // per workgroup of the first marking launch; -1: an id outside the range
  int64_t* partial;    // per workgroup of the counting launches
  int64_t num_partial;
  int64_t* first;      // {distinct ids of the first end, 1 when the second has to be counted}
  int64_t* slices;     // by bits: slices that the first marking launch takes
  bool bits;
};

__global__ void __launch_bounds__(kThreads) clear_marks_kernel(uint4* map, int64_t n) {
  const int64_t i0 = static_cast<int64_t>(blockIdx.x) * (kThreads * 4) + threadIdx.x;
#pragma unroll
  for (int k = 0; k < 4; ++k)
    if (i0 + k * kThreads < n) map[i0 + k * kThreads] = make_uint4(0, 0, 0, 0);
}

// FIRST: workgroups with blockIdx.y 0 mark the ids of `a`, those with 1 look through `b`, all
// leave their largest id.  Otherwise: the ids of `b`, when they have to be counted.
template <typename IdT, bool FIRST>
__global__ void __launch_bounds__(kThreads)
mark_ids_kernel(const IdT* __restrict__ a, const IdT* __restrict__ b, int64_t E, int64_t range,
                DistinctSpace s) {
  __shared__ int64_t s_largest[kThreads / kWave];
  if (!FIRST && !s.first[1]) return;
  const bool marks = !FIRST || blockIdx.y == 0;
  const IdT* __restrict__ ids = FIRST && marks ? a : b;
  unsigned char* map = s.map + (FIRST ? 0 : range);
  const int64_t base = static_cast<int64_t>(blockIdx.x) * kMarkTile + threadIdx.x;
  IdT id[kMarkItems];
#pragma unroll
  for (int k = 0; k < kMarkItems; ++k) {
    const int64_t i = base + k * kThreads;
    id[k] = ids[i < E ? i : E - 1];
  }
  // (an id below zero is a huge one here, and both are outside)
  uint64_t largest = 0;
#pragma unroll
  for (int k = 0; k < kMarkItems; ++k) {
    const uint64_t v = static_cast<uint64_t>(static_cast<int64_t>(id[k]));
    largest = v > largest ? v : largest;
  }
  const uint64_t bound = static_cast<uint64_t>(range);
  if (marks) {
    uint32_t at[kMarkItems];
    unsigned char seen[kMarkItems];
#pragma unroll
    for (int k = 0; k < kMarkItems; ++k) {
      const uint64_t v = static_cast<uint64_t>(static_cast<int64_t>(id[k]));
      at[k] = v < bound ? static_cast<uint32_t>(v) : ~0u;
      seen[k] = map[v < bound ? v : 0];
    }
#pragma unroll
    for (int k = 0; k < kMarkItems; ++k)
      if (at[k] != ~0u && !seen[k]) map[at[k]] = 1;
  }
  if (!FIRST) return;
  int64_t top = largest < bound ? static_cast<int64_t>(largest) : INT64_MAX;
#pragma unroll
  for (int d = kWave / 2; d > 0; d >>= 1) {
    const int64_t o = __shfl_xor(top, d, kWave);
    top = o > top ? o : top;
  }
  if ((threadIdx.x & (kWave - 1)) == 0) s_largest[threadIdx.x / kWave] = top;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kThreads / kWave; ++w) top = s_largest[w] > top ? s_largest[w] : top;
    s.largest[static_cast<int64_t>(blockIdx.y) * gridDim.x + blockIdx.x] = top;
  }
}

// marked bytes of one end (every byte is 0 or 1)
template <bool FIRST>
__global__ void __launch_bounds__(kThreads) count_marks_kernel(DistinctSpace s, int64_t range) {
  __shared__ int64_t lds[kThreads / kWave + 1];
  if (!FIRST && !s.first[1]) return;
  const uint4* map = reinterpret_cast<const uint4*>(s.map + (FIRST ? 0 : range));
  int64_t n = 0;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x; i < range / 16;
       i += static_cast<int64_t>(kCountBlocks) * kThreads) {
    const uint4 v = map[i];
    n += __popc(v.x) + __popc(v.y) + __popc(v.z) + __popc(v.w);
  }
  int64_t total;
  block_exclusive_scan<kThreads>(n, &total, lds);
  if (threadIdx.x == 0) s.partial[blockIdx.x] = total;
}

// this thread's share of the counting launch's sums
__device__ __forceinline__ int64_t sum_partial(const DistinctSpace& s, int threads) {
  int64_t n = 0;
  for (int64_t i = threadIdx.x; i < s.num_partial; i += threads) n += s.partial[i];
  return n;
}

// after the first end: is the second to be counted?  (one workgroup)
constexpr int kDecideThreads = 1024;
__global__ void __launch_bounds__(kDecideThreads)
decide_second_kernel(DistinctSpace s, int64_t num_largest) {
  __shared__ int64_t lds[kDecideThreads / kWave + 1];
  __shared__ int64_t s_top[kDecideThreads / kWave];
  int64_t top = 0;
  for (int64_t i = threadIdx.x; i < num_largest; i += kDecideThreads)
    top = s.largest[i] > top ? s.largest[i] : top;
#pragma unroll
  for (int d = kWave / 2; d > 0; d >>= 1) {
    const int64_t o = __shfl_xor(top, d, kWave);
    top = o > top ? o : top;
  }
  if ((threadIdx.x & (kWave - 1)) == 0) s_top[threadIdx.x / kWave] = top;
  int64_t total;
  block_exclusive_scan<kDecideThreads>(sum_partial(s, kDecideThreads), &total, lds);
  if (threadIdx.x == 0) {
    for (int w = 1; w < kDecideThreads / kWave; ++w) top = s_top[w] > top ? s_top[w] : top;
    const bool outside = top == INT64_MAX;
    s.first[0] = outside ? -1 : total;
    s.first[1] = !outside && total <= top;  // (total = top + 1: every id up to the largest is there)
  }
}

__global__ void __launch_bounds__(kDecideThreads)
post_distinct_kernel(DistinctSpace s, gs_mailbox* box, int64_t ticket) {
  __shared__ int64_t lds[kDecideThreads / kWave + 1];
  int64_t second = 0;
  const bool counted = s.first[1] != 0;
  block_exclusive_scan<kDecideThreads>(counted ? sum_partial(s, kDecideThreads) : 0, &second, lds);
  // (-1 and -2, an id outside the range, leave the second end uncounted; by bits, the launch that found
  // so has posted)
  if (threadIdx.x == 0 && (counted || !s.bits)) post_mailbox(box, counted && second > s.first[0] ? second : s.first[0], ticket);
}

// The same for long lists, by bits in LDS: every compute unit keeps a bitmap of 1.28 M ids and
// marks its share of the edges there, the bitmaps go to memory and are or-ed and counted.
// How many such slices the ids take is guessed from 1024 of them (guess_slices_kernel): the first
// launch deals its workgroups out to that many, so that it reads the end once for each -- the
// workgroups of a share sit on one die, whose L2 has it for the second -- and finds the largest id
// of both ends; a second takes the slices behind those, if there are any.  Ids beyond eight
// slices are reported and the caller asks for the bytes.  14 M edges over 2.45 M nodes, 64-bit
// ids: 220 us by bytes, 145 with one slice in the first launch and a second launch for the
// rest, 113 so (the list loaded and sorted: 494 -> 462).  The bitmaps are 80 MB whatever the list, so lists below 4 M edges stay
// with the bytes.
constexpr int kBitWords = 39936;  // 156 KB of a compute unit's 160
constexpr int64_t kSliceIds = int64_t(kBitWords) * 32;
constexpr int kMaxSlices = 8;
constexpr int kBitBlocks = 256;   // one for every compute unit
constexpr int kBitThreads = 1024;
constexpr int kBitTrip = 8;
constexpr int64_t kBitMarkEdges = int64_t(1) << 22;
constexpr int kOrRows = 16, kOrVecs = kThreads / kOrRows;  // of the counting launch
constexpr int kOrBlocks = kBitWords / 4 / kOrVecs;
static_assert(kBitWords % (4 * kOrVecs) == 0, "whole workgroups per slice");

// largest id of both ends; every thread gets it
template <int THREADS>
__device__ __forceinline__ int64_t largest_of_list(const DistinctSpace& s) {
  __shared__ int64_t s_top[THREADS / kWave];
  int64_t top = 0;
  for (int i = threadIdx.x; i < kBitBlocks; i += THREADS) top = s.largest[i] > top ? s.largest[i] : top;
#pragma unroll
  for (int d = kWave / 2; d > 0; d >>= 1) {
    const int64_t o = __shfl_xor(top, d, kWave);
    top = o > top ? o : top;
  }
  if ((threadIdx.x & (kWave - 1)) == 0) s_top[threadIdx.x / kWave] = top;
  __syncthreads();
  for (int w = 0; w < THREADS / kWave; ++w) top = s_top[w] > top ? s_top[w] : top;
  return top;
}

// Slices of the second end, or none if it is not to be counted: the first end has every id up to
// the largest, or an id is beyond the slices.  Every workgroup of the second end's marking adds the
// first end's sums up for itself, and takes all slices, as the largest id is known by then: a launch
// that decides and one for the slices behind, without work, took 4.5 us each (14 M edges, list loaded
// and sorted: 422 -> 419 us).
__device__ __forceinline__ int64_t second_slices(const DistinctSpace& s) {
  __shared__ int64_t lds[kBitThreads / kWave + 1];
  int64_t n = 0;
#pragma unroll
  for (int i = threadIdx.x; i < kOrBlocks * kMaxSlices; i += kBitThreads) n += s.partial[i];
  int64_t total;
  block_exclusive_scan<kBitThreads>(n, &total, lds);
  const int64_t top = largest_of_list<kBitThreads>(s);
  const int64_t all = top / kSliceIds + 1;
  const bool outside = all > kMaxSlices;
  const bool counted = !outside && total <= top;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    s.first[0] = outside ? -2 : total;
    s.first[1] = counted;
  }
  return counted ? all : 0;
}

// Slices that the largest of a sample of both ends asks for: one id a thread of either (a compute
// unit alone fetches a line every 2.5 ns: eight a thread took 40 us).
constexpr int kGuessThreads = 512;
template <typename IdT>
__global__ void __launch_bounds__(kGuessThreads)
guess_slices_kernel(const IdT* __restrict__ a, const IdT* __restrict__ b, int64_t E, DistinctSpace s) {
  __shared__ uint64_t s_top[kGuessThreads / kWave];
  const int64_t step = E / kGuessThreads;  // (lists that are counted by bits are longer)
  const IdT x = a[threadIdx.x * step], y = b[threadIdx.x * step];
  const uint64_t u = static_cast<uint64_t>(static_cast<int64_t>(x));
  const uint64_t v = static_cast<uint64_t>(static_cast<int64_t>(y));
  uint64_t top = u > v ? u : v;
#pragma unroll
  for (int d = kWave / 2; d > 0; d >>= 1) {
    const uint64_t o = __shfl_xor(top, d, kWave);
    top = o > top ? o : top;
  }
  if ((threadIdx.x & (kWave - 1)) == 0) s_top[threadIdx.x / kWave] = top;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kGuessThreads / kWave; ++w) top = s_top[w] > top ? s_top[w] : top;
    const uint64_t n = top / static_cast<uint64_t>(kSliceIds) + 1;
    *s.slices = n <= static_cast<uint64_t>(kMaxSlices) ? static_cast<int64_t>(n) : 1;  // (beyond: reported)
  }
}

// Of the first launch, which takes `slices` slices: workgroup w works on die w % 8, takes slice
// (w / 8) % slices and one of the die's 32 / slices shares of the end.
struct FirstSlices {
  int64_t per_die;
  __device__ __forceinline__ explicit FirstSlices(int64_t slices) : per_die(kBitBlocks / kXcds / slices) {}
  __device__ __forceinline__ int64_t parts() const { return per_die * kXcds; }
  __device__ __forceinline__ int64_t workgroup(int64_t slices, int64_t slice, int64_t part) const {
    return ((part / kXcds) * slices + slice) * kXcds + part % kXcds;
  }
};

// A thread's ids of [lo, hi) to `use`, the next trip's on their way meanwhile; `before` runs behind
// the first trip's loads.  (Ids behind hi are the last one again; 419 -> 417 us, 6 M over 1 M nodes 254 -> 252.
// As streams: the list loaded and sorted 415 -> 406, 11 M edges, 32-bit ids 301 -> 295.)
template <typename IdT, typename Before, typename Use>
__device__ __forceinline__ void each_id(const IdT* __restrict__ ids, int64_t lo, int64_t hi, Before before,
                                        Use use) {
  IdT id[kBitTrip], next[kBitTrip];
  int64_t i = lo + threadIdx.x;
  auto load = [&](IdT* to) {
#pragma unroll
    for (int u = 0; u < kBitTrip; ++u) {
      const int64_t at = i + u * kBitThreads;
      to[u] = __builtin_nontemporal_load(ids + (at < hi ? at : hi - 1));
    }
  };
  if (i < hi) load(id);
  before();
  while (i < hi) {
    i += kBitTrip * kBitThreads;
    if (i < hi) load(next);
#pragma unroll
    for (int u = 0; u < kBitTrip; ++u) use(id[u]);
#pragma unroll
    for (int u = 0; u < kBitTrip; ++u) id[u] = next[u];
  }
}

// REST: the slices behind the first launch's.  look: the other end, looked through for its largest id
// (null when the largest is known).
template <typename IdT, bool REST, bool SECOND>
__global__ void __launch_bounds__(kBitThreads)
mark_bits_kernel(const IdT* __restrict__ ids, const IdT* __restrict__ look, int64_t E, DistinctSpace s,
                 gs_mailbox* box, int64_t ticket) {
  static_assert(!(REST && SECOND), "nothing is left behind the second end's launch");
  __shared__ __attribute__((aligned(16))) uint32_t s_bits[kBitWords];
  __shared__ int64_t s_wave[kBitThreads / kWave];
  int64_t slices;
  if constexpr (SECOND) {
    slices = second_slices(s);
    if (!slices) {  // the count is known: the host has it two launches earlier
      if (blockIdx.x == 0 && threadIdx.x == 0) post_mailbox(box, s.first[0], ticket);
      return;
    }
  } else {
    slices = *s.slices;
  }
  int64_t slice, part, parts;
  if (REST) {
    const int64_t all = largest_of_list<kBitThreads>(s) / kSliceIds + 1;
    if (all <= slices || all > kMaxSlices) return;
    const int64_t rest = all - slices;
    parts = kBitBlocks / rest;
    slice = slices + blockIdx.x % rest;
    part = blockIdx.x / rest;
    if (part >= parts) return;
  } else {
    const FirstSlices f(slices);
    parts = f.parts();
    slice = blockIdx.x / kXcds % slices;
    part = blockIdx.x / kXcds / slices * kXcds + blockIdx.x % kXcds;
  }
  // (a workgroup that finds no share of its own marks nothing, but looks through the other end)
  const int64_t lo = part < parts ? E * part / parts : 0;
  const int64_t hi = part < parts ? E * (part + 1) / parts : 0;
  const uint64_t first_id = static_cast<uint64_t>(slice * kSliceIds);
  uint64_t largest = 0;  // (an id below zero is a huge one here)
  each_id(ids, lo, hi,
          [&] {
            for (int j = threadIdx.x; j < kBitWords / 4; j += kBitThreads)
              reinterpret_cast<uint4*>(s_bits)[j] = make_uint4(0, 0, 0, 0);
            __syncthreads();
          },
          [&](IdT id) {
            const uint64_t v = static_cast<uint64_t>(static_cast<int64_t>(id));
            largest = v > largest ? v : largest;
            const uint64_t in = v - first_id;
            if (in < static_cast<uint64_t>(kSliceIds)) {
              const uint32_t at = static_cast<uint32_t>(in);
              atomicOr(&s_bits[at >> 5], 1u << (at & 31u));
            }
          });
  if (!REST && look) {
    const int64_t from = E * blockIdx.x / kBitBlocks, to = E * (blockIdx.x + 1) / kBitBlocks;
    each_id(look, from, to, [] {},
            [&](IdT id) {
              const uint64_t v = static_cast<uint64_t>(static_cast<int64_t>(id));
              largest = v > largest ? v : largest;
            });
    int64_t top = largest >> 62 ? INT64_MAX : static_cast<int64_t>(largest);
#pragma unroll
    for (int d = kWave / 2; d > 0; d >>= 1) {
      const int64_t o = __shfl_xor(top, d, kWave);
      top = o > top ? o : top;
    }
    if ((threadIdx.x & (kWave - 1)) == 0) s_wave[threadIdx.x / kWave] = top;
  }
  __syncthreads();
  if (!REST && look && threadIdx.x == 0) {
    int64_t top = 0;
    for (int w = 0; w < kBitThreads / kWave; ++w) top = s_wave[w] > top ? s_wave[w] : top;
    s.largest[blockIdx.x] = top;
  }
  uint4* out = reinterpret_cast<uint4*>(s.map) +
               static_cast<int64_t>((REST ? kBitBlocks : 0) + blockIdx.x) * (kBitWords / 4);
  for (int j = threadIdx.x; j < kBitWords / 4; j += kBitThreads)
    out[j] = reinterpret_cast<const uint4*>(s_bits)[j];
}

// Ids in any bitmap of slice blockIdx.y: sixteen threads share the bitmaps of a word.
template <bool SECOND>
__global__ void __launch_bounds__(kThreads) count_bits_kernel(DistinctSpace s) {
  __shared__ uint4 s_or[kOrRows][kOrVecs];
  __shared__ int64_t s_scan[kThreads / kWave + 1];
  if (SECOND && !s.first[1]) return;
  const int64_t known = largest_of_list<kThreads>(s) / kSliceIds + 1;
  const int64_t slices = SECOND ? known : *s.slices;
  const int64_t slice = blockIdx.y;
  int64_t n = 0;
  if (slice < known && known <= kMaxSlices) {  // (the same for the whole workgroup)
    // the slice's bitmaps: of the first launch's workgroups, or of the second's
    const bool rest = slice >= slices;
    const FirstSlices f(slices);
    const int64_t step = known - slices;
    const int64_t rows = rest ? kBitBlocks / step : f.parts();
    const int g = threadIdx.x / kOrVecs, v = threadIdx.x % kOrVecs;
    const uint4* map = reinterpret_cast<const uint4*>(s.map) + static_cast<int64_t>(blockIdx.x) * kOrVecs + v;
    uint4 all = make_uint4(0, 0, 0, 0);
#pragma unroll 8
    for (int64_t r = g; r < rows; r += kOrRows) {
      const int64_t row = rest ? kBitBlocks + slice - slices + r * step : f.workgroup(slices, slice, r);
      const uint4 x = map[row * (kBitWords / 4)];
      all.x |= x.x; all.y |= x.y; all.z |= x.z; all.w |= x.w;
    }
    s_or[g][v] = all;
    __syncthreads();
    if (g == 0) {
      for (int r = 1; r < kOrRows; ++r) {
        const uint4 x = s_or[r][v];
        all.x |= x.x; all.y |= x.y; all.z |= x.z; all.w |= x.w;
      }
      n = __popc(all.x) + __popc(all.y) + __popc(all.z) + __popc(all.w);
    }
  }
  int64_t total;
  block_exclusive_scan<kThreads>(n, &total, s_scan);
  if (threadIdx.x == 0) s.partial[blockIdx.y * kOrBlocks + blockIdx.x] = total;
}

template <typename IdT>
void distinct_by_bits(const IdT* a, const IdT* b, int64_t E, const DistinctSpace& s, gs_mailbox* box,
                      int64_t ticket, hipStream_t st) {
  hipLaunchKernelGGL((guess_slices_kernel<IdT>), dim3(1), dim3(kGuessThreads), 0, st, a, b, E, s);
  const IdT* known = nullptr;
  const dim3 marks(kBitBlocks), counts(kOrBlocks, kMaxSlices);
  hipLaunchKernelGGL((mark_bits_kernel<IdT, false, false>), marks, dim3(kBitThreads), 0, st, a, b, E, s,
                     box, ticket);
  hipLaunchKernelGGL((mark_bits_kernel<IdT, true, false>), marks, dim3(kBitThreads), 0, st, a, b, E, s,
                     box, ticket);
  hipLaunchKernelGGL(count_bits_kernel<false>, counts, dim3(kThreads), 0, st, s);
  hipLaunchKernelGGL((mark_bits_kernel<IdT, false, true>), marks, dim3(kBitThreads), 0, st, b, known, E, s,
                     box, ticket);
  hipLaunchKernelGGL(count_bits_kernel<true>, counts, dim3(kThreads), 0, st, s);
}

// bytes per end of the list, a multiple of 16; ids of a graph with up to a million nodes always fit
inline int64_t mark_range(int64_t E) {
  const int64_t n = E > (int64_t(1) << 20) ? E : (int64_t(1) << 20);
  return (n + 4095) / 4096 * 4096;
}

// ---------------------------------------------------- binned scatter-add ----
// out[target[e]] += data[e]^powk without an atomic to memory: the edges of up to 1024 bins of
// targets are brought together, and a workgroup adds a bin's edges up in LDS and writes its sums
// with plain stores.  Atomics to memory run at some twenty-five per nanosecond on this part
// whatever the kernel does around them; edges that mostly hit different targets paid that price
// one by one.
//
// A bin is as many lines of 32 targets as the others, dealt out by a multiplication of the line
// number: a run of neighbouring targets as a bin held a third of a skewed graph's edges, which
// then took dozens of workgroups and their sums atomics to memory after all.
//
//   tiles    8192 edges are put in the order of their bins in LDS and written side by side, place in
//            the bin (2 bytes) and value, with the places where the bins' runs start
//   totals   edges of every bin
//   sums     a workgroup per bin (or share of one with many more than the average) reads its runs
//
// The sums in LDS are 64-bit ones: 64 additions to 32-bit floats in LDS take 81 ns on a compute
// unit, to 64-bit floats 8 (to 32-bit integers 2.3).
//
// 2 M edges over 2.45 M targets, uniform / skewed like R-MAT's rows: 56 / 58 us with bins of neighbours,
// made by a pass of the sort above, and 32-bit sums; 32 / 40 now (64-bit ids, one by one: 115 / 276).
constexpr int kBinThreads = 1024;
constexpr int kSumTileItems = 8;
constexpr int kSumTile = kBinThreads * kSumTileItems;
constexpr int kMaxBins = 1024;
constexpr int kBinMaxShift = 13;          // 2^13 sums = 64 KB of LDS
constexpr int kBinMinBits = 8;            // 256 bins at least, where there are as many targets
// The additions to one LDS word queue up, so a bin of more than 5/4 of the average (a hub's) and of
// two edges a sum is shared by several workgroups, which then add their sums to memory with atomics.  Shares by the average
// alone left a bin of twice as much to one workgroup, and, of three targets, each: 30 M edges,
// uniform / skewed, 3 targets 12900 / 7630 us, now 279 / 330; 40: 1090 / 1192, now 282 / 294; 256: 277 / 542,
// now 277 / 455; 30 k: 216 / 274, now 215 / 259.
constexpr int kBinParts = 256;           // workgroups that may share one bin
constexpr int64_t kBinPartItems = 4096;  // edges a share has at least
constexpr int64_t kBinPartMost = 16384;  // and at most, where 256 shares of the bin allow it
constexpr int kBinLineBits = 5;           // 32 targets, 128 bytes

// Target t is sum `place` of bin `place >> bin_shift`: its line number times an odd number.
struct BinOrder {
  uint32_t mult, inverse, mask;  // of the line number
  int line_bits, bin_shift, bins;
  __device__ __forceinline__ uint32_t place(uint32_t t) const {
    return ((((t >> line_bits) * mult) & mask) << line_bits) | (t & ((1u << line_bits) - 1u));
  }
  __device__ __forceinline__ uint32_t target(uint32_t place) const {
    return ((((place >> line_bits) * inverse) & mask) << line_bits) |
           (place & ((1u << line_bits) - 1u));
  }
};

inline BinOrder bin_order(int64_t num_targets) {
  BinOrder o;
  const int bits = bits_for(num_targets);
  o.bin_shift = bits > kBinMinBits ? bits - kBinMinBits : 0;
  if (o.bin_shift > kBinMaxShift) o.bin_shift = kBinMaxShift;
  o.bins = 1 << (bits - o.bin_shift);
  o.line_bits = o.bin_shift < kBinLineBits ? o.bin_shift : kBinLineBits;
  o.mask = static_cast<uint32_t>((int64_t(1) << (bits - o.line_bits)) - 1);
  o.mult = 0x9E3779B1u;
  o.inverse = o.mult;  // Newton: right in three more bits each time, from three
  for (int i = 0; i < 4; ++i) o.inverse *= 2u - o.mult * o.inverse;
  return o;
}

struct SumSpace {
  unsigned short* place;  // [E]: in the bin
  float* value;           // [E]
  unsigned short* start;  // [tiles][bins + 1]
  int64_t* totals;        // [bins]
};

template <typename IdT>
__global__ void __launch_bounds__(kBinThreads)
sum_tiles_kernel(const IdT* __restrict__ target, const float* __restrict__ data, int64_t E,
                 int64_t num_targets, int powk, BinOrder order, SumSpace s, float* __restrict__ clear) {
  static_assert(kBinThreads == kOneThreads && kMaxBins <= kBinThreads, "one_scan is over 1024 threads");
  __shared__ uint32_t s_cnt[kMaxBins];
  __shared__ float s_value[kSumTile];
  __shared__ unsigned short s_place[kSumTile];
  __shared__ int s_scan[2][kOneWaves];
  const int64_t base = static_cast<int64_t>(blockIdx.x) * kSumTile;
  const int n = static_cast<int>(E - base < kSumTile ? E - base : kSumTile);
  // (no read carries a condition: the last edge again past the end)
  IdT t[kSumTileItems];
  float x[kSumTileItems];
#pragma unroll
  for (int u = 0; u < kSumTileItems; ++u) {
    const int i = u * kBinThreads + static_cast<int>(threadIdx.x);
    t[u] = target[base + (i < n ? i : n - 1)];
  }
#pragma unroll
  for (int u = 0; u < kSumTileItems; ++u) {
    const int i = u * kBinThreads + static_cast<int>(threadIdx.x);
    x[u] = data[base + (i < n ? i : n - 1)];
  }
  const int bins = order.bins;
  s_cnt[threadIdx.x] = 0u;
  lds_barrier();
  uint32_t bin[kSumTileItems], rank[kSumTileItems], place[kSumTileItems];
#pragma unroll
  for (int u = 0; u < kSumTileItems; ++u) {
    const int i = u * kBinThreads + static_cast<int>(threadIdx.x);
    // (a target that is none of num_targets has no sum to go to: left out)
    const bool live = i < n && t[u] >= 0 && static_cast<int64_t>(t[u]) < num_targets;
    const uint32_t p = order.place(static_cast<uint32_t>(t[u]));
    bin[u] = live ? p >> order.bin_shift : kMaxBins;
    place[u] = p & ((1u << order.bin_shift) - 1u);
    rank[u] = live ? atomicAdd(&s_cnt[bin[u]], 1u) : 0u;
  }
  lds_barrier();
  unsigned short* __restrict__ start = s.start + static_cast<int64_t>(blockIdx.x) * (bins + 1);
  const int mine = static_cast<int>(s_cnt[threadIdx.x]);
  int total;
  const int at = one_scan(mine, &total, s_scan, 0);
  s_cnt[threadIdx.x] = static_cast<uint32_t>(at);
  if (static_cast<int>(threadIdx.x) < bins) start[threadIdx.x] = static_cast<unsigned short>(at);
  if (threadIdx.x == 0) start[bins] = static_cast<unsigned short>(total);
  lds_barrier();
#pragma unroll
  for (int u = 0; u < kSumTileItems; ++u) {
    if (bin[u] < kMaxBins) {
      const uint32_t to = s_cnt[bin[u]] + rank[u];
      s_value[to] = powk_f(x[u], powk);
      s_place[to] = static_cast<unsigned short>(place[u]);
    }
  }
  lds_barrier();
#pragma unroll
  for (int u = 0; u < kSumTileItems; ++u) {
    const int i = u * kBinThreads + static_cast<int>(threadIdx.x);
    if (i < total) {
      s.value[base + i] = s_value[i];
      s.place[base + i] = s_place[i];
    }
  }
  if (clear) {  // this workgroup's share of the sums
    const int64_t to = num_targets * (blockIdx.x + 1) / gridDim.x;
    for (int64_t i = num_targets * blockIdx.x / gridDim.x + threadIdx.x; i < to; i += kBinThreads) clear[i] = 0.0f;
  }
}

constexpr int kClearTile = 4 * kThreads;
__global__ void __launch_bounds__(kThreads) clear_sums_kernel(float* __restrict__ out, int64_t n) {
  const int64_t base = static_cast<int64_t>(blockIdx.x) * kClearTile + threadIdx.x;
#pragma unroll
  for (int u = 0; u < 4; ++u)
    if (base + u * kThreads < n) out[base + u * kThreads] = 0.0f;
}

__global__ void __launch_bounds__(kThreads) sum_totals_kernel(SumSpace s, int64_t tiles, int bins) {
  __shared__ int64_t s_scan[kThreads / kWave + 1];
  const unsigned short* __restrict__ start = s.start + blockIdx.x;
  int64_t mine = 0;
  for (int64_t t = threadIdx.x; t < tiles; t += kThreads)
    mine += start[t * (bins + 1) + 1] - start[t * (bins + 1)];
  int64_t total;
  block_exclusive_scan<kThreads>(mine, &total, s_scan);
  if (threadIdx.x == 0) s.totals[blockIdx.x] = total;
}

constexpr int kSumTrip = 8;  // pieces of runs, of up to 64 edges, that a wave asks for together

__global__ void __launch_bounds__(kBinThreads)
bin_sum_kernel(SumSpace s, int64_t tiles, int64_t alone, int64_t part_items, BinOrder order,
               int64_t num_targets, bool zero, float* __restrict__ out) {
  extern __shared__ double s_sum[];
  // Which bin, and which share of it, this workgroup takes: the launch has one workgroup per
  // share that can exist (a bin of n > alone edges has ceil(n / part_items) of them, 256 at most),
  // and every workgroup works the numbering out for itself from the bins' sizes.
  __shared__ int s_scan[2][kOneWaves];
  __shared__ int s_first[kMaxBins + 1];
  const int bins = order.bins;
  {
    int shares = 0, total;
    if (static_cast<int>(threadIdx.x) < bins) {
      const int64_t n = s.totals[threadIdx.x];
      const int64_t some = (n + part_items - 1) / part_items;
      shares = n > alone ? static_cast<int>(some < kBinParts ? some : kBinParts) : (n > 0 ? 1 : 0);
    }
    s_first[threadIdx.x] = one_scan(shares, &total, s_scan, 0);
    if (threadIdx.x == 0) s_first[kBinThreads] = total;
    __syncthreads();
  }
  if (static_cast<int>(blockIdx.x) >= s_first[bins]) return;
  int bin = 0;
  for (int step = kMaxBins / 2; step > 0; step >>= 1)
    if (bin + step <= bins && s_first[bin + step] <= static_cast<int>(blockIdx.x)) bin += step;
  const int part = static_cast<int>(blockIdx.x) - s_first[bin];
  const int parts = s_first[bin + 1] - s_first[bin];
  const int64_t tile_lo = tiles * part / parts, tile_hi = tiles * (part + 1) / parts;
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int width = 1 << order.bin_shift;
  for (int j = threadIdx.x; j < width; j += kBinThreads) s_sum[j] = 0.0;
  __syncthreads();
  // a wave takes every sixteenth tile, 64 at a time: a lane knows a tile's run
  for (int64_t t0 = tile_lo + wave; t0 < tile_hi; t0 += kOneWaves * kWave) {
    const int64_t tile = t0 + static_cast<int64_t>(lane) * kOneWaves;
    int start = 0, len = 0;
    if (tile < tile_hi) {
      start = s.start[tile * (bins + 1) + bin];
      len = static_cast<int>(s.start[tile * (bins + 1) + bin + 1]) - start;
    }
    const int ends = wave_inclusive_sum((len + kWave - 1) / kWave);
    const int pieces = __builtin_amdgcn_readlane(ends, kWave - 1);
    for (int p0 = 0; p0 < pieces; p0 += kSumTrip) {
      // (no read under a condition of its own, past the run's end its last edge again: a place that might be
      // none was cut to its 16 bits at once, and so waited for before the next read was asked for: 1.0 M edges
      // 26 -> 22 us)
      float v[kSumTrip];
      uint32_t at[kSumTrip];
      unsigned int held = 0u;
#pragma unroll
      for (int u = 0; u < kSumTrip; ++u) {
        if (p0 + u >= pieces) break;
        const int j = __popcll(__ballot(ends <= p0 + u));
        const int run = __builtin_amdgcn_readlane(len, j);
        const int i = (p0 + u - (__builtin_amdgcn_readlane(ends, j) - (run + kWave - 1) / kWave)) * kWave + lane;
        const int64_t from = (t0 + static_cast<int64_t>(j) * kOneWaves) * kSumTile +
                             __builtin_amdgcn_readlane(start, j) + (i < run ? i : run - 1);
        v[u] = s.value[from];
        at[u] = s.place[from];
        if (i < run) held |= 1u << u;
      }
#pragma unroll
      for (int u = 0; u < kSumTrip; ++u)
        if (held >> u & 1u) unsafeAtomicAdd(&s_sum[at[u]], static_cast<double>(v[u]));
    }
  }
  __syncthreads();
  const uint32_t first = static_cast<uint32_t>(bin) << order.bin_shift;
  if (parts > 1) {
    for (int j = threadIdx.x; j < width; j += kBinThreads) {
      const float x = static_cast<float>(s_sum[j]);
      const uint32_t t = order.target(first + j);
      if (x != 0.0f && t < num_targets) unsafeAtomicAdd(out + t, x);
    }
    return;
  }
  if (zero) {  // (and nothing to add to: plain writes)
    for (int j = threadIdx.x; j < width; j += kBinThreads) {
      const float x = static_cast<float>(s_sum[j]);
      const uint32_t t = order.target(first + j);
      if (x != 0.0f && t < num_targets) out[t] = x;
    }
    return;
  }
  // the bin is this workgroup's alone: plain read, add, write -- a thread's sums eight at a
  // time, the reads (of a word that is always there where the sum is zero) before the writes
  constexpr int kBatch = 8;
  for (int j0 = threadIdx.x; j0 < width; j0 += kBinThreads * kBatch) {
    float x[kBatch], was[kBatch];
    uint32_t t[kBatch];
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      const int j = j0 + u * kBinThreads;
      t[u] = order.target(first + j);
      x[u] = (j < width && t[u] < num_targets) ? static_cast<float>(s_sum[j]) : 0.0f;
    }
#pragma unroll
    for (int u = 0; u < kBatch; ++u) was[u] = out[x[u] != 0.0f ? t[u] : 0u];
#pragma unroll
    for (int u = 0; u < kBatch; ++u)
      if (x[u] != 0.0f) out[t[u]] = was[u] + x[u];
  }
}

// Whether the binned path takes the call: plain edge order, few enough targets for 1024 bins of
// 2^13, enough edges for three launches to pay.  Few targets meet in the plain kernel's LDS tables
// already; among very many, its atomics to memory cost less than clearing and writing all sums.
// Plain / binned, us, uniform and skewed targets, at the lines and beyond:
//   E x targets 2^23: 131 k edges, 10 targets  13/34  14/46, 100   28/16  29/33
//                     524 k        10          38/29  38/47,  40   66/19  66/38
//                       1 M         3          29/37  30/60,  10   73/28  75/49
//                     8.4 M         1         100/108 99/108,  3  174/100 176/104
//   32 targets an edge: 131 k, 8 M targets     16/26  27/28, 2.45 M 16/18 28/22; 262 k, 8 M 21/28 46/31
inline bool bin_sum_applies(const int64_t* e_ids, int64_t E, int64_t num_targets) {
  return !e_ids && E >= (int64_t(1) << 17) && num_targets > 0 &&
         num_targets <= (int64_t(kMaxBins) << kBinMaxShift) && E < (int64_t(1) << 31) &&
         E * num_targets > (int64_t(1) << 23) && num_targets <= 32 * E;
}

// Sums that a tile's workgroup clears along with its edges, 64 KB; with more a launch of its own spreads them.  Nothing
// is read then: 2.0 M edges into 2.45 M sums, a fill of 4.8 us, tiles 9.6 and bins 21.1, now 11.5 and 20.7 us, and the
// layer-wise minibatch around it 330 -> 324 with the gap between them.
constexpr int64_t kClearAlong = int64_t(1) << 14;

inline int64_t sum_tiles(int64_t E) { return (E + kSumTile - 1) / kSumTile; }

template <typename IdT>
int bin_sum_impl(const IdT* target, const float* data, int64_t E, int powk, int64_t num_targets,
                 bool fresh, float* out, void* workspace, size_t workspace_bytes, hipStream_t st) {
  const int64_t tiles = sum_tiles(E);
  Carver ws(workspace, workspace_bytes);
  SumSpace s;
  s.place = ws.take<unsigned short>(E);
  s.value = ws.take<float>(E);
  const BinOrder order = bin_order(num_targets);
  s.start = ws.take<unsigned short>(tiles * (order.bins + 1));
  s.totals = ws.take<int64_t>(order.bins);
  if (!ws.ok) {
    set_error_text("gs_coo_sum_binned: workspace needs %zu bytes, 256-byte aligned",
                   gs_coo_sum_workspace_bytes(E, num_targets));
    return GS_ERR_WORKSPACE;
  }
  // (per call: the attribute belongs to the device the call runs on)
  const hipError_t lds_allowed = hipFuncSetAttribute(
      reinterpret_cast<const void*>(bin_sum_kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
      static_cast<int>(sizeof(double) << kBinMaxShift));
  if (lds_allowed != hipSuccess) {
    set_error_text("gs_coo_sum_binned: %s", hipGetErrorString(lds_allowed));
    return GS_ERR_LAUNCH;
  }
  const bool along = fresh && num_targets <= kClearAlong * tiles;
  if (fresh && !along)
    hipLaunchKernelGGL(clear_sums_kernel, dim3(blocks_for(num_targets, kClearTile)), dim3(kThreads), 0, st, out,
                       num_targets);
  hipLaunchKernelGGL(sum_tiles_kernel<IdT>, dim3(static_cast<unsigned>(tiles)), dim3(kBinThreads), 0, st,
                     target, data, E, num_targets, powk, order, s, along ? out : nullptr);
  hipLaunchKernelGGL(sum_totals_kernel, dim3(order.bins), dim3(kThreads), 0, st, s, tiles, order.bins);
  // (few targets make few bins: the average is that of 256 then, so that every bin is shared.  A share
  // clears and writes all sums of its bin, so bins of many sums are shared for many edges only, in
  // larger shares: 2 M R-MAT edges into 2.45 M sums, call, 52 us by edges alone, 49 so; a tenth of them
  // on one target 45 and 41)
  const int64_t width = int64_t(1) << order.bin_shift;
  const int64_t average = std::max({E / std::max(order.bins, 1 << kBinMinBits), kBinPartItems, width});
  const int64_t part_items = std::min(average, kBinPartMost);
  const int64_t alone = std::max(average + average / 4, 2 * width);
  const int64_t shares = E / part_items + order.bins;  // at most: sum of ceil(n / part_items) over the bins
  hipLaunchKernelGGL(bin_sum_kernel, dim3(static_cast<unsigned>(shares)), dim3(kBinThreads),
                     sizeof(double) << order.bin_shift, st, s, tiles, alone, part_items, order,
                     num_targets, fresh, out);
  return check_launch("coo_sum_binned");
}

// fresh: `out` holds nothing yet
int coo_sum_any(const void* target, int id_bytes, const int64_t* e_ids, const float* data, int64_t E, int64_t powk,
                int64_t num_targets, bool fresh, float* out, void* workspace, size_t workspace_bytes, void* stream) {
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (E == 0 || !bin_sum_applies(e_ids, E, num_targets)) {
    if (fresh)
      hipLaunchKernelGGL(clear_sums_kernel, dim3(blocks_for(num_targets, kClearTile)), dim3(kThreads), 0, st, out,
                         num_targets);
    if (E == 0) return check_launch("coo_sum");
    return coo_sum_bounded(target, id_bytes, e_ids, data, E, powk, num_targets, out, stream);
  }
  if (id_bytes == 8)
    return bin_sum_impl(static_cast<const int64_t*>(target), data, E, static_cast<int>(powk), num_targets, fresh, out,
                        workspace, workspace_bytes, st);
  return bin_sum_impl(static_cast<const int32_t*>(target), data, E, static_cast<int>(powk), num_targets, fresh, out,
                      workspace, workspace_bytes, st);
}

}  // namespace
}  // namespace gs

using namespace gs;

extern "C" {

int gs_csc2coo(const int64_t* indptr, int64_t num_cols, int64_t nnz, void* col, int id_bytes,
               void* stream) {
  GS_REQUIRE(num_cols >= 0 && nnz >= 0 && num_cols < (int64_t(1) << 31),
             "gs_csc2coo: negative size or more than 2^31 columns");
  GS_REQUIRE(nnz == 0 || (indptr && col), "gs_csc2coo: null pointer");
  GS_REQUIRE(valid_id_bytes(id_bytes), "gs_csc2coo: id_bytes must be 4 or 8, got %d", id_bytes);
  if (nnz == 0) return GS_OK;
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (id_bytes == 8)
    launch_csc2coo<int64_t, false>(indptr, num_cols, nnz, nullptr, static_cast<int64_t*>(col), st);
  else
    launch_csc2coo<int32_t, false>(indptr, num_cols, nnz, nullptr, static_cast<int32_t*>(col), st);
  return check_launch("csc2coo");
}

int gs_dcsc2coo(const int64_t* indptr, int64_t num_cols, int64_t nnz, const void* ids, void* col,
                int id_bytes, void* stream) {
  GS_REQUIRE(num_cols >= 0 && nnz >= 0 && num_cols < (int64_t(1) << 31),
             "gs_dcsc2coo: negative size or more than 2^31 columns");
  GS_REQUIRE(nnz == 0 || (indptr && col && ids), "gs_dcsc2coo: null pointer");
  GS_REQUIRE(valid_id_bytes(id_bytes), "gs_dcsc2coo: id_bytes must be 4 or 8, got %d", id_bytes);
  if (nnz == 0) return GS_OK;
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (id_bytes == 8)
    launch_csc2coo<int64_t, true>(indptr, num_cols, nnz, static_cast<const int64_t*>(ids),
                              static_cast<int64_t*>(col), st);
  else
    launch_csc2coo<int32_t, true>(indptr, num_cols, nnz, static_cast<const int32_t*>(ids),
                              static_cast<int32_t*>(col), st);
  return check_launch("dcsc2coo");
}

size_t gs_csc_compress_workspace_bytes(int64_t num_cols) {
  if (num_cols < 0) num_cols = 0;
  return padded(static_cast<size_t>(num_cols + 1) * 8) + scan_workspace_bytes(num_cols);
}

int gs_csc_compress(const int64_t* indptr, int64_t num_cols, int id_bytes, void* val_ids,
                    int64_t* out_indptr, int64_t* num_valid, void* workspace,
                    size_t workspace_bytes, void* stream) {
  GS_REQUIRE(num_cols >= 0 && indptr && out_indptr && num_valid && (num_cols == 0 || val_ids),
             "gs_csc_compress: bad argument");
  GS_REQUIRE(valid_id_bytes(id_bytes), "gs_csc_compress: id_bytes must be 4 or 8, got %d", id_bytes);
  Carver ws(workspace, workspace_bytes);
  int64_t* prefix = ws.take<int64_t>(num_cols + 1);
  int64_t* tiles = ws.take<int64_t>(scan_num_tiles(num_cols) + 1);
  if (!ws.ok) {
    set_error_text("gs_csc_compress: workspace needs %zu bytes, 256-byte aligned",
                   gs_csc_compress_workspace_bytes(num_cols));
    return GS_ERR_WORKSPACE;
  }
  hipStream_t st = static_cast<hipStream_t>(stream);
  NonEmptyColumn f{indptr};
  GS_RETURN_IF_ERROR(exclusive_scan(f, num_cols, prefix, tiles, st));
  const dim3 grid(blocks_for(num_cols + 1, kThreads));
  if (id_bytes == 8)
    hipLaunchKernelGGL(compress_kernel<int64_t>, grid, dim3(kThreads), 0, st, indptr, num_cols,
                       prefix, static_cast<int64_t*>(val_ids), out_indptr, num_valid);
  else
    hipLaunchKernelGGL(compress_kernel<int32_t>, grid, dim3(kThreads), 0, st, indptr, num_cols,
                       prefix, static_cast<int32_t*>(val_ids), out_indptr, num_valid);
  return check_launch("csc_compress");
}

size_t gs_coo2csc_workspace_bytes(int64_t E, int64_t num_keys) {
  (void)num_keys;
  if (E < 0) E = 0;
  return sort_space_bytes(E);
}

size_t gs_distinct_ends_workspace_bytes(int64_t E) {
  if (E < 0) E = 0;
  size_t map = 2 * static_cast<size_t>(mark_range(E));
  const size_t bits = static_cast<size_t>(2 * kBitBlocks) * kBitWords * 4;
  if (E >= kBitMarkEdges && bits > map) map = bits;
  const size_t largest = 2 * static_cast<size_t>(blocks_for(E, kMarkTile)) + kBitBlocks;
  return padded(map) + padded(largest * 8) + padded(kOrBlocks * kMaxSlices * 8) + 256;
}

int gs_distinct_ends(const void* a, const void* b, int id_bytes, int64_t E, void* workspace,
                     size_t workspace_bytes, gs_mailbox* mailbox, int64_t ticket, void* stream) {
  const bool by_bits = !(id_bytes & GS_DISTINCT_BYTES) && E >= kBitMarkEdges;
  id_bytes &= ~GS_DISTINCT_BYTES;
  GS_REQUIRE(E > 0 && E < (int64_t(1) << 32) - 8192 && a && b && mailbox,
             "gs_distinct_ends: bad argument");
  GS_REQUIRE(valid_id_bytes(id_bytes), "gs_distinct_ends: id_bytes must be 4 or 8, got %d", id_bytes);
  const int64_t range = mark_range(E);
  const int blocks = blocks_for(E, kMarkTile);
  const size_t bits = static_cast<size_t>(2 * kBitBlocks) * kBitWords * 4;
  Carver ws(workspace, workspace_bytes);
  DistinctSpace s;
  s.map = ws.take<unsigned char>(by_bits ? bits : static_cast<size_t>(2 * range));
  s.largest = ws.take<int64_t>(2 * static_cast<size_t>(blocks) + kBitBlocks);
  s.num_partial = by_bits ? kOrBlocks * kMaxSlices : kCountBlocks;
  s.partial = ws.take<int64_t>(static_cast<size_t>(s.num_partial));
  s.first = ws.take<int64_t>(3);
  s.slices = s.first + 2;
  s.bits = by_bits;
  if (!ws.ok) {
    set_error_text("gs_distinct_ends: workspace needs %zu bytes, 256-byte aligned",
                   gs_distinct_ends_workspace_bytes(E));
    return GS_ERR_WORKSPACE;
  }
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (by_bits) {
    if (id_bytes == 8)
      distinct_by_bits(static_cast<const int64_t*>(a), static_cast<const int64_t*>(b), E, s, mailbox,
                       ticket, st);
    else
      distinct_by_bits(static_cast<const int32_t*>(a), static_cast<const int32_t*>(b), E, s, mailbox,
                       ticket, st);
  } else {
    const int64_t vecs = 2 * range / 16;
    hipLaunchKernelGGL(clear_marks_kernel, dim3(blocks_for(vecs, kThreads * 4)), dim3(kThreads), 0, st,
                       reinterpret_cast<uint4*>(s.map), vecs);
    auto both = [&](auto first, auto second, auto* pa, auto* pb) {
      hipLaunchKernelGGL(first, dim3(blocks, 2), dim3(kThreads), 0, st, pa, pb, E, range, s);
      hipLaunchKernelGGL(count_marks_kernel<true>, dim3(kCountBlocks), dim3(kThreads), 0, st, s, range);
      hipLaunchKernelGGL(decide_second_kernel, dim3(1), dim3(kDecideThreads), 0, st, s,
                         static_cast<int64_t>(2) * blocks);
      hipLaunchKernelGGL(second, dim3(blocks), dim3(kThreads), 0, st, pa, pb, E, range, s);
      hipLaunchKernelGGL(count_marks_kernel<false>, dim3(kCountBlocks), dim3(kThreads), 0, st, s, range);
    };
    if (id_bytes == 8)
      both(mark_ids_kernel<int64_t, true>, mark_ids_kernel<int64_t, false>,
           static_cast<const int64_t*>(a), static_cast<const int64_t*>(b));
    else
      both(mark_ids_kernel<int32_t, true>, mark_ids_kernel<int32_t, false>,
           static_cast<const int32_t*>(a), static_cast<const int32_t*>(b));
  }
  hipLaunchKernelGGL(post_distinct_kernel, dim3(1), dim3(kDecideThreads), 0, st, s, mailbox, ticket);
  return check_launch("distinct_ends");
}

int gs_coo2csc_values(const void* key, const void* value, int id_bytes, int64_t E, int64_t num_keys,
                      int64_t num_values, int sorted, int64_t* indptr, void* out_value, int64_t* perm,
                      void* workspace, size_t workspace_bytes, void* stream) {
  GS_REQUIRE(E >= 0 && num_keys >= 0 && num_values >= 0, "gs_coo2csc: negative size");
  GS_REQUIRE(indptr || !sorted, "gs_coo2csc: sorted keys and no indptr leave nothing to do");
  GS_REQUIRE(E == 0 || key, "gs_coo2csc: key is null");
  GS_REQUIRE(sorted || E == 0 || (value && out_value && perm),
             "gs_coo2csc: value/out_value/perm required when the keys are not sorted");
  GS_REQUIRE(valid_id_bytes(id_bytes), "gs_coo2csc: id_bytes must be 4 or 8, got %d", id_bytes);
  hipStream_t st = static_cast<hipStream_t>(stream);
  return id_bytes == 8
             ? coo2csc_impl<int64_t>(static_cast<const int64_t*>(key),
                                     static_cast<const int64_t*>(value), E, num_keys, num_values, sorted,
                                     indptr, static_cast<int64_t*>(out_value), perm, workspace,
                                     workspace_bytes, st)
             : coo2csc_impl<int32_t>(static_cast<const int32_t*>(key),
                                     static_cast<const int32_t*>(value), E, num_keys, num_values, sorted,
                                     indptr, static_cast<int32_t*>(out_value), perm, workspace,
                                     workspace_bytes, st);
}

int gs_coo2csc(const void* key, const void* value, int id_bytes, int64_t E, int64_t num_keys,
               int sorted, int64_t* indptr, void* out_value, int64_t* perm, void* workspace,
               size_t workspace_bytes, void* stream) {
  return gs_coo2csc_values(key, value, id_bytes, E, num_keys, num_keys, sorted, indptr, out_value, perm,
                           workspace, workspace_bytes, stream);
}

int gs_indptr_split(const int64_t* indptr, const int64_t* offsets, int64_t num_batches,
                    int64_t total, int64_t* out, void* stream) {
  return gs_indptr_split_cuts(indptr, offsets, num_batches, total, out, nullptr, stream);
}

int gs_indptr_split_cuts(const int64_t* indptr, const int64_t* offsets, int64_t num_batches,
                         int64_t total, int64_t* out, int64_t* cuts, void* stream) {
  GS_REQUIRE(num_batches >= 0 && total >= 0, "gs_indptr_split: negative size");
  if (num_batches == 0 || (total == 0 && !cuts)) return GS_OK;
  GS_REQUIRE(indptr && offsets && (out || total == 0), "gs_indptr_split: null pointer");
  const int64_t lanes = cuts && num_batches + 1 > total ? num_batches + 1 : total;
  hipLaunchKernelGGL(indptr_split_kernel, dim3(blocks_for(lanes, kThreads)), dim3(kThreads), 0,
                     static_cast<hipStream_t>(stream), indptr, offsets, num_batches, total, out,
                     cuts);
  return check_launch("indptr_split");
}

size_t gs_coo_sum_workspace_bytes(int64_t E, int64_t num_targets) {
  if (E < 0) E = 0;
  if (!bin_sum_applies(nullptr, E, num_targets)) return 256;
  return padded(static_cast<size_t>(E) * 2) + padded(static_cast<size_t>(E) * 4) +
         padded(static_cast<size_t>(sum_tiles(E)) * (bin_order(num_targets).bins + 1) * 2) +
         padded(static_cast<size_t>(bin_order(num_targets).bins) * 8);
}

int gs_coo_sum_binned(const void* target, int id_bytes, const int64_t* e_ids, const float* data,
                      int64_t E, int64_t powk, int64_t num_targets, float* out, void* workspace,
                      size_t workspace_bytes, void* stream) {
  GS_REQUIRE(E >= 0 && powk >= 1 && num_targets >= 0,
             "gs_coo_sum_binned: negative size or powk < 1");
  GS_REQUIRE(E == 0 || (target && data && out), "gs_coo_sum_binned: null pointer");
  GS_REQUIRE(valid_id_bytes(id_bytes), "gs_coo_sum_binned: id_bytes must be 4 or 8, got %d",
             id_bytes);
  if (E == 0) return GS_OK;
  return coo_sum_any(target, id_bytes, e_ids, data, E, powk, num_targets, false, out, workspace, workspace_bytes,
                     stream);
}

int gs_coo_sum_fresh(const void* target, int id_bytes, const int64_t* e_ids, const float* data, int64_t E,
                     int64_t powk, int64_t num_targets, float* out, void* workspace, size_t workspace_bytes,
                     void* stream) {
  GS_REQUIRE(E >= 0 && powk >= 1 && num_targets >= 0, "gs_coo_sum_fresh: negative size or powk < 1");
  GS_REQUIRE((E == 0 || (target && data)) && (num_targets == 0 || out), "gs_coo_sum_fresh: null pointer");
  GS_REQUIRE(valid_id_bytes(id_bytes), "gs_coo_sum_fresh: id_bytes must be 4 or 8, got %d", id_bytes);
  if (num_targets == 0) return GS_OK;
  return coo_sum_any(target, id_bytes, e_ids, data, E, powk, num_targets, true, out, workspace, workspace_bytes,
                     stream);
}

}  // extern "C"
