// Batched relabel without a memory-side atomic per item: bring the items of a batch together
// by hash class, find first occurrences per class in an LDS table, rank them by position.
//
// Same contract as the relabel on hash regions (gs_unique.hip: batch_relabel_impl; reference
// impl::BatchCSRRelabelCUDA, src/cuda/batch_relabel.cu:236-328): batch b owns seeds
// [seeds_ptr[b], seeds_ptr[b+1]) and ids [ids_ptr[b], ids_ptr[b+1]); its frontier is the
// distinct values of (its seeds, then its ids) in first-occurrence order; every id is renamed
// to its rank inside its own batch's frontier.
//
// The regions version pays one compare-and-swap on device memory per item, and those run at
// about 26 G/s on this machine whatever else happens.  Here there are no atomics on memory:
//
//   plan      every batch is cut into P_b classes of about 2 k items by its ids' hash times
//             P_b; a class of a batch is a "bucket", numbered batch by batch
//   tiles     8192 consecutive items of a batch are put in the order of their classes in LDS and
//             written side by side, with the places where the classes start: a "run" per class.
//             The order inside a run is whatever the atomics make it: nothing below depends
//             on it, first occurrences are decided by the positions the records carry
//   first     one workgroup per bucket: the runs of its class in all tiles of the batch, LDS
//             table id -> smallest position; that position is the id's first occurrence in
//             the batch, and is stored at the record's position
//   rank      chained scan over the positions that are their own first: per 64 positions a
//             mask and the number of first occurrences before them
//   rename    a pass in the order of the positions: the rank of an item's first position from
//             mask + count; first occurrences write the frontier, ids their new name
//
// 17 M items in 64 batches: plan 4 us, tiles 40, first 104, rank 24, rename 66; counted, scanned
// and scattered it was 43 + 9 + 92, first 99 and rename 86.  Batches of more than 2^20 items on average have so many
// classes that a tile's runs are a few records; they are counted, the buckets laid out by a scan
// and the records scattered to them, with a counter addition per (4096-item tile, class).
//
// A record is read once and never written again; of the three places an item touches at
// random (its first position's store, the rank it looks up, and before these passes were in
// the order of the positions its new name and its place in the frontier) two are left, and a
// first occurrence looks up nothing.
//
// Buckets are handed to workgroups so that consecutive buckets -- one batch's -- run on the
// same XCD one after the other (workgroup w runs on XCD w % 8): the positions a batch's
// buckets store to are a megabyte or two that stays in that XCD's L2 until its lines are
// full.
//
// The ids may come from a sampler that is still running when the relabel is queued, and whose
// total is then read from the offsets on the device.  A sampler that failed leaves a negative
// last offset: every pass then leaves at once and the call reports -1, as a look-back of its
// own that gave up would.
//
// An LDS table that fills up (a bucket with more than its slots' worth of distinct ids: only
// a batch beyond ~16 M distinct ids can do that) raises an error word and the call reports
// -4: the caller repeats it on hash regions (GS_RELABEL_REGIONS).
#include "gs_common.hpp"
#include "gs_batch_items.hpp"
#include "gs_one.hpp"

namespace gs {
namespace {

constexpr int kThreads = 256;
constexpr int kBucketItemsLog2 = 11;   // classes are sized for <= 2048 items on average
constexpr int kMaxClassesLog2 = 12;    // at most 4096 classes per batch
constexpr int kPartItems = 16;         // items of a thread in the count / scatter passes
constexpr int kPartTile = kThreads * kPartItems;
// LDS counters of a tile: the buckets of the batches it touches (two batches with all the
// classes there may be, and those wholly inside it: a class per 2048 items and one on top)
constexpr int counter_cap(int classes_log2) {
  return 2 * (1 << classes_log2) + (kPartTile >> (kBucketItemsLog2 - 1)) +
         2 * static_cast<int>(kStagedBatches) + 2;
}
constexpr int kCounterCap = counter_cap(kMaxClassesLog2);
// Batches of up to so many items on average go by tiles of runs: at 2^20 items a batch has 512
// classes and a tile's runs 16 records, at 2^22 of 2048 classes 4.  By counting / by runs (which are
// read a tenth faster since), us, ids skewed like R-MAT's rows of 2^14 | 2^17 | 2^21 nodes:
//    items a batch    one batch                      four
//    2^19          59/58   53/42   51/37       81/68   79/58   80/55
//    2^20          87/91   76/72   70/58      158/122 156/122 158/121
//    2^21         147/163 124/122 117/105     292/296 291/301 300/305
//    2^22         270/309 225/286 210/280     578/866 585/910 608/964
// An id that has 4 % of a batch's items fills a bucket that one workgroup reads, and runs
// are slower to read than records side by side: 2^20 items of 2^12 nodes in one batch 103/123.
constexpr int64_t kRunsItems = int64_t(1) << 20;
constexpr int kTileThreads = 1024;     // two such workgroups fill a compute unit's waves
constexpr int kTileItems = 8;          // items of a thread
constexpr int kTile = kTileThreads * kTileItems;
constexpr int kSlots = 4096;           // LDS table of a bucket (8-byte slots)
// 64 positions make a word of the rank pass; a wave takes 64 words, or 16 where there are few items:
// more workgroups, one trip each (0.5 M items: 10 -> 7 us).
constexpr int kRankWords = 64, kRankWordsFew = 16;
constexpr int64_t kRankFewItems = int64_t(1) << 22;
constexpr int rank_tile(int words) { return kThreads / kWave * words * kWave; }
// Threads of a bucket's workgroup: the table lets five of them share a compute unit, 20 waves
// of 256 threads, 32 of 512 (17 M items: 112 -> 104 us; 4.3 M: 39 -> 30).
constexpr int kBucketThreads = 512;
constexpr int kTrip = 5;  // records of a thread that are asked for together (a whole bucket nearly always)

struct Plan {
  uint32_t* bucket_base;  // [B + 1]: first bucket of every batch; [B] = number of buckets
  uint32_t* classes;      // [B]
  // by tiles of runs only
  uint32_t* tile_base;    // [B + 1]: first tile of every batch; [B] = number of tiles
  uint32_t* row_base;     // [B]: where the batch's tiles keep their runs' starts
  // [buckets bound]: what the pass over the buckets needs of a bucket, in one read: {the start of its
  // run in the batch's first tile, from one tile to the next, tiles, the batch's first item}
  uint4* bucket;
};

struct Bins {
  Plan plan;
  uint32_t* count;        // [buckets bound]: items per bucket
  uint32_t* fill;         // [buckets bound]: records placed so far
  int64_t* bucket_ptr;    // [buckets bound + 1]: first record of every bucket
  uint32_t* bucket_batch; // [buckets bound]: the batch of every bucket that holds records
  unsigned long long* records;  // [M]: id << 32 | position
  // by tiles of runs instead: the tiles' items in the order of their classes, ids and places in the
  // tile apart, and per tile the start of every class's run and the tile's number of items
  uint32_t* run_id;             // [M]
  unsigned short* run_pos;      // [M]
  unsigned short* run_start;    // [starts bound]
  uint32_t* first;        // [M]: position of the first occurrence of the item's id in its batch
  uint4* ranks;           // per 64 positions: {first occurrences as bits (x, y), how many before them (z), 0}
  unsigned int* error;    // the look-back state's error word: 2 = id too wide, 3 = a table filled up
};

inline int64_t buckets_bound(int64_t M, int64_t B) { return (M >> kBucketItemsLog2) + B + 8; }
inline int64_t rank_tiles(int64_t M) {
  return M / rank_tile(M < kRankFewItems ? kRankWordsFew : kRankWords) + 1;
}
inline int64_t tiles_bound(int64_t M, int64_t B) { return M / kTile + B; }
inline int64_t starts_bound(int64_t M, int64_t B) {
  const int64_t most = int64_t(1) << kMaxClassesLog2, classes = (M >> kBucketItemsLog2) + 1;
  return tiles_bound(M, B) * ((classes < most ? classes : most) + 1);
}
inline bool by_runs(int64_t M, int64_t B) { return M / B <= kRunsItems; }

// slot of an id in a bucket's table: other hash bits than the ones that chose the bucket
__device__ __forceinline__ uint32_t slot_of(uint32_t key) {
  return (key * 0x85EBCA6Bu) >> (32 - 12);
}
static_assert(kSlots == 1 << 12, "slot_of yields 12 bits");

__global__ void __launch_bounds__(kThreads)
bins_init_kernel(Bins s, int64_t buckets, LookbackState lb, int64_t tiles) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
  if (i < buckets) {
    s.count[i] = 0u;
    s.fill[i] = 0u;
  }
  if (i < tiles) lb.status[i] = 0ull;
  if (i == 0) *lb.error = 0u;
}

// one workgroup: classes per batch and the numbering of the buckets; by tiles of runs also the
// numbering of the tiles and the look-back state of the rank pass cleared
template <typename IdT, bool RUNS>
__global__ void __launch_bounds__(512)
bins_plan_kernel(BatchItems<IdT> x, Plan p, LookbackState lb, int64_t rank_tiles) {
  __shared__ int64_t s_scan[512 / kWave + 1];
  const int64_t b = threadIdx.x;
  const int64_t m = b < x.B && x.ids_ptr[x.B] >= 0 ? x.start(b + 1) - x.start(b) : 0;
  int64_t classes = 0, tiles = 0;
  if (b < x.B) {
    classes = (m + (int64_t(1) << kBucketItemsLog2) - 1) >> kBucketItemsLog2;
    if (classes < 1) classes = 1;
    if (classes > (int64_t(1) << kMaxClassesLog2)) classes = int64_t(1) << kMaxClassesLog2;
    p.classes[b] = static_cast<uint32_t>(classes);
    if (RUNS) tiles = (m + kTile - 1) / kTile;
  }
  int64_t total;
  const int64_t before = block_exclusive_scan<512>(classes << 32 | tiles, &total, s_scan);
  if (b < x.B) p.bucket_base[b] = static_cast<uint32_t>(before >> 32);
  if (b == 0) p.bucket_base[x.B] = static_cast<uint32_t>(total >> 32);
  if (!RUNS) return;
  if (b < x.B) p.tile_base[b] = static_cast<uint32_t>(before);
  if (b == 0) p.tile_base[x.B] = static_cast<uint32_t>(total);
  const int64_t row = block_exclusive_scan<512>(tiles * (classes + 1), &total, s_scan);
  if (b < x.B) {
    p.row_base[b] = static_cast<uint32_t>(row);
    // (the others are written by their batch's first tile)
    if (tiles == 0) p.bucket[before >> 32] = make_uint4(0u, 0u, 0u, 0u);
  }
  for (int64_t i = b; i < rank_tiles; i += 512) lb.status[i] = 0ull;
  if (b == 0) *lb.error = 0u;
}

// the last batch whose base is <= t (base[0] = 0; B <= 511); whole waves call this
__device__ __forceinline__ int64_t batch_at(const uint32_t* __restrict__ base, int64_t B, uint32_t t) {
  static_assert(kStagedBatches < 8 * kWave, "eight batches a lane");
  const int lane = threadIdx.x & (kWave - 1);
  const uint32_t far = 8 * lane < B ? base[8 * lane] : 0xFFFFFFFFu;
  const int64_t group = 8 * (__popcll(__ballot(far <= t)) - 1);
  const uint32_t near = group + lane < B && lane < 8 ? base[group + lane] : 0xFFFFFFFFu;
  return group + __popcll(__ballot(near <= t)) - 1;
}

// A tile: 8192 items of one batch, put in the order of their classes.
template <typename IdT>
__global__ void __launch_bounds__(kTileThreads) bins_tiles_kernel(BatchItems<IdT> x, Bins s) {
  constexpr int kMaxClasses = 1 << kMaxClassesLog2;
  constexpr int kPer = kMaxClasses / kTileThreads;  // consecutive classes of a thread in the scan
  static_assert(kTileThreads == kOneThreads, "one_scan is over 1024 threads");
  __shared__ uint32_t s_cnt[kMaxClasses];
  __shared__ uint32_t s_id[kTile];
  __shared__ unsigned short s_pos[kTile];
  __shared__ int s_scan[2][kOneWaves];
  const uint32_t tile = blockIdx.x;
  if (tile >= s.plan.tile_base[x.B]) return;
  const int64_t b = batch_at(s.plan.tile_base, x.B, tile);
  const int64_t in_batch = tile - s.plan.tile_base[b];
  const int64_t first_seed = x.seeds_ptr[b], n_seeds = x.seeds_ptr[b + 1] - first_seed;
  const int64_t first_id = x.ids_ptr[b];
  const int64_t left = n_seeds + x.ids_ptr[b + 1] - first_id - in_batch * kTile;
  const int n = static_cast<int>(left < kTile ? left : kTile);
  const int classes = static_cast<int>(s.plan.classes[b]);
  // an item is read through a chosen address, the last one again past the end, all at once
  IdT key[kTileItems];
#pragma unroll
  for (int u = 0; u < kTileItems; ++u) {
    const int i = u * kTileThreads + static_cast<int>(threadIdx.x);
    const int64_t off = in_batch * kTile + (i < n ? i : n - 1);
    key[u] = *(off < n_seeds ? x.seeds + first_seed + off : x.ids + first_id + off - n_seeds);
  }
  for (int c = threadIdx.x; c < classes; c += kTileThreads) s_cnt[c] = 0u;
  if (in_batch == 0) {
    const uint32_t tiles = s.plan.tile_base[b + 1] - s.plan.tile_base[b];
    for (int c = threadIdx.x; c < classes; c += kTileThreads)
      s.plan.bucket[s.plan.bucket_base[b] + c] =
          make_uint4(s.plan.row_base[b] + c, static_cast<uint32_t>(classes + 1), tiles,
                     static_cast<uint32_t>(first_seed + first_id));
  }
  lds_barrier();
  uint32_t cls[kTileItems], rank[kTileItems];
  bool wide = false;
#pragma unroll
  for (int u = 0; u < kTileItems; ++u) {
    const int i = u * kTileThreads + static_cast<int>(threadIdx.x);
    cls[u] = __umulhi(hash32(static_cast<uint32_t>(key[u])), static_cast<uint32_t>(classes));
    rank[u] = 0u;
    if (i < n) {
      wide |= !fits_slot(key[u]);
      rank[u] = atomicAdd(&s_cnt[cls[u]], 1u);
    }
  }
  if (wide) *s.error = 2u;  // 64-bit ids ride on 32-bit records: this one does not fit
  lds_barrier();
  // counts to starts, for the tile's own records and for the pass over the buckets
  unsigned short* __restrict__ starts = s.run_start + s.plan.row_base[b] + in_batch * (classes + 1);
  int mine[kPer], sum = 0;
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    const int c = static_cast<int>(threadIdx.x) * kPer + j;
    mine[j] = c < classes ? static_cast<int>(s_cnt[c]) : 0;
    sum += mine[j];
  }
  int total;
  int at = one_scan(sum, &total, s_scan, 0);
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    const int c = static_cast<int>(threadIdx.x) * kPer + j;
    if (c < classes) {
      s_cnt[c] = static_cast<uint32_t>(at);
      starts[c] = static_cast<unsigned short>(at);
    }
    at += mine[j];
  }
  if (threadIdx.x == 0) starts[classes] = static_cast<unsigned short>(n);
  lds_barrier();
#pragma unroll
  for (int u = 0; u < kTileItems; ++u) {
    const int i = u * kTileThreads + static_cast<int>(threadIdx.x);
    if (i < n) {
      const uint32_t to = s_cnt[cls[u]] + rank[u];
      s_id[to] = static_cast<uint32_t>(key[u]);
      s_pos[to] = static_cast<unsigned short>(i);
    }
  }
  lds_barrier();
  const int64_t out = first_seed + first_id + in_batch * kTile;
#pragma unroll
  for (int u = 0; u < kTileItems; ++u) {
    const int i = u * kTileThreads + static_cast<int>(threadIdx.x);
    if (i < n) {
      s.run_id[out + i] = s_id[i];
      s.run_pos[out + i] = s_pos[i];
    }
  }
}

// What the count and the scatter pass share: the tile's items, their batches and buckets.
template <typename IdT, int CAP>
struct TileWalk {
  int64_t lo, hi;          // batches of the tile's first and last item
  uint32_t first_bucket;   // bucket_base[lo]
  uint32_t span;           // buckets of batches lo..hi, cut to the LDS counters
  // M comes in as the caller's count of items, which may be a bound: the offsets hold the
  // true one.  False: the tile lies beyond the items (the whole workgroup leaves).
  __device__ __forceinline__ bool open(BatchItems<IdT>& x, const Plan& p, int64_t& M,
                                       int64_t* s_seeds_ptr, int64_t* s_ids_ptr,
                                       uint32_t* s_base, uint32_t* s_classes, int64_t* s_range,
                                       uint32_t* s_cnt) {
    x.stage_offsets(s_seeds_ptr, s_ids_ptr);
    const int64_t held = x.seeds_ptr[x.B] + x.ids_ptr[x.B];
    if (held < M) M = held;
    if (x.ids_ptr[x.B] < 0) return false;  // the producer of the ids failed
    if (static_cast<int64_t>(blockIdx.x) * kPartTile >= M) return false;
    for (int64_t b = threadIdx.x; b <= x.B; b += kThreads) {
      s_base[b] = p.bucket_base[b];
      s_classes[b] = b < x.B ? p.classes[b] : 1u;
    }
    const int64_t first = static_cast<int64_t>(blockIdx.x) * kPartTile;
    const int64_t last = first + kPartTile - 1 < M ? first + kPartTile - 1 : M - 1;
    x.block_range(first, last, s_range, &lo, &hi);  // (ends with a barrier: s_base is there)
    first_bucket = s_base[lo];
    const uint32_t all = s_base[hi + 1] - first_bucket;
    span = all < static_cast<uint32_t>(CAP) ? all : static_cast<uint32_t>(CAP);
    for (uint32_t c = threadIdx.x; c < span; c += kThreads) s_cnt[c] = 0u;
    __syncthreads();
    return true;
  }
};

// LDS of the two partition passes
template <int CAP>
struct PartShared {
  int64_t seeds_ptr[kStagedBatches + 1];
  int64_t ids_ptr[kStagedBatches + 1];
  uint32_t base[kStagedBatches + 1];
  uint32_t classes[kStagedBatches + 1];
  int64_t range[2];
  uint32_t cnt[CAP];
};

// count (SCATTER false): items per bucket.  scatter: the same walk, then the tile's share of
// every bucket it touches is reserved with one addition and the records are placed.  (Tiles
// of several rounds of 4096 items -- fewer additions to memory, longer runs of records side
// by side -- were slower: 64 / 143 us against 55 / 105 us over 17 M items; workgroups that
// stay and loop are the slower shape on this machine.)
template <typename IdT, bool SCATTER, int CAP>
__global__ void __launch_bounds__(kThreads)
bins_partition_kernel(BatchItems<IdT> x, int64_t M, Bins s) {
  __shared__ PartShared<CAP> sh;
  TileWalk<IdT, CAP> w;
  if (!w.open(x, s.plan, M, sh.seeds_ptr, sh.ids_ptr, sh.base, sh.classes, sh.range, sh.cnt)) return;
  const int64_t tile_first = static_cast<int64_t>(blockIdx.x) * kPartTile;
  // where every item is: all reads of the thread's items stand together, none behind a
  // condition of its own (the last item again past the end)
  const IdT* from[kPartItems];
  uint32_t batch[kPartItems];
#pragma unroll
  for (int k = 0; k < kPartItems; ++k) {
    const int64_t i = tile_first + k * kThreads + threadIdx.x;
    const int64_t ic = i < M ? i : M - 1;
    const int64_t b = x.batch_of(ic, w.lo, w.hi);
    batch[k] = static_cast<uint32_t>(b);
    from[k] = x.where_in(b, ic);
  }
  IdT key[kPartItems];
#pragma unroll
  for (int k = 0; k < kPartItems; ++k) key[k] = *from[k];
  uint32_t bucket[kPartItems], rank[kPartItems];
  bool wide = false;
#pragma unroll
  for (int k = 0; k < kPartItems; ++k) {
    const int64_t i = tile_first + k * kThreads + threadIdx.x;
    const uint32_t cls = __umulhi(hash32(static_cast<uint32_t>(key[k])), sh.classes[batch[k]]);
    bucket[k] = sh.base[batch[k]] + cls;
    rank[k] = 0u;
    if (i < M) {
      if (sizeof(IdT) == 8 && (static_cast<unsigned long long>(key[k]) >> 32) != 0ull) wide = true;
      const uint32_t c = bucket[k] - w.first_bucket;
      if (c < w.span) {
        rank[k] = atomicAdd(&sh.cnt[c], 1u);
      } else if (SCATTER) {  // beyond the LDS counters: straight to memory
        rank[k] = static_cast<uint32_t>(s.bucket_ptr[bucket[k]]) + atomicAdd(&s.fill[bucket[k]], 1u);
        s.bucket_batch[bucket[k]] = batch[k];
      } else {
        atomicAdd(&s.count[bucket[k]], 1u);
      }
    }
  }
  if (wide) *s.error = 2u;  // 64-bit ids ride on 32-bit records: this one does not fit
  __syncthreads();
  for (uint32_t c = threadIdx.x; c < w.span; c += kThreads) {
    const uint32_t n = sh.cnt[c];
    if (!n) continue;
    const uint32_t bucket_c = w.first_bucket + c;
    if (SCATTER) {
      // the counter turns into the place of the tile's first record in the bucket
      sh.cnt[c] = static_cast<uint32_t>(s.bucket_ptr[bucket_c]) + atomicAdd(&s.fill[bucket_c], n);
      int64_t lo = w.lo, hi = w.hi;  // the batch the bucket belongs to, for the later passes
      while (lo < hi) {
        const int64_t mid = (lo + hi + 1) >> 1;
        if (sh.base[mid] <= bucket_c) lo = mid; else hi = mid - 1;
      }
      s.bucket_batch[bucket_c] = static_cast<uint32_t>(lo);
    } else {
      atomicAdd(&s.count[bucket_c], n);
    }
  }
  if (!SCATTER) return;
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kPartItems; ++k) {
    const int64_t i = tile_first + k * kThreads + threadIdx.x;
    if (i < M) {
      const uint32_t c = bucket[k] - w.first_bucket;
      const uint32_t at = c < w.span ? sh.cnt[c] + rank[k] : rank[k];
      s.records[at] = (static_cast<unsigned long long>(static_cast<uint32_t>(key[k])) << 32) |
                      static_cast<unsigned long long>(static_cast<uint32_t>(i));
    }
  }
}

struct CountOf {
  const uint32_t* count;
  __device__ __forceinline__ int64_t operator()(int64_t i) const { return count[i]; }
};

// Bucket of workgroup w: XCD x = w % 8 takes the x-th eighth of the buckets, in order.
__device__ __forceinline__ int64_t bucket_of_workgroup(int64_t num_buckets) {
  const int64_t per = (num_buckets + kXcds - 1) / kXcds;
  const int64_t k = static_cast<int64_t>(blockIdx.x % kXcds) * per + blockIdx.x / kXcds;
  return blockIdx.x / kXcds < per && k < num_buckets ? k : -1;
}

// Enters a record (id << 32 | position) into the bucket's LDS table: slot = id << 32 | smallest
// position.  Raises the error word when the table is full.
__device__ __forceinline__ void table_enter(unsigned long long* __restrict__ tab,
                                            unsigned long long rec, unsigned int* error) {
  const uint32_t key = static_cast<uint32_t>(rec >> 32);
  uint32_t p = slot_of(key);
  int probes = 0;
  while (true) {
    // (read first: a hub's thousands of records would queue up at their slot)
    unsigned long long prev = __hip_atomic_load(&tab[p], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    if (prev == ~0ull) prev = atomicCAS(&tab[p], ~0ull, rec);
    if (prev == ~0ull) break;
    if (static_cast<uint32_t>(prev >> 32) == key) {
      if (prev > rec) atomicMin(&tab[p], rec);
      break;
    }
    p = (p + 1) & (kSlots - 1);
    if (++probes >= kSlots) {
      *error = 3u;
      break;
    }
  }
}
// the first position of the record's id
// (a table that was too small may lack the id: what is returned then is read by nobody)
__device__ __forceinline__ uint32_t table_first(const unsigned long long* __restrict__ tab,
                                                unsigned long long w, uint32_t key) {  // w: its slot
  uint32_t p = slot_of(key);
  int probes = 0;
  while (static_cast<uint32_t>(w >> 32) != key && ++probes < kSlots) {
    p = (p + 1) & (kSlots - 1);
    w = tab[p];
  }
  return static_cast<uint32_t>(w);
}

// One workgroup per bucket: every record's position gets the smallest position of its id.
// (A bucket of one trip, as most are, still holds its records in registers by then; the first
// trip's records are asked for before the table is cleared, so that the clearing hides under it.)
__global__ void __launch_bounds__(kBucketThreads) bins_first_kernel(Bins s, int64_t B) {
  __shared__ unsigned long long tab[kSlots];
  const int64_t k = bucket_of_workgroup(s.plan.bucket_base[B]);
  if (k < 0) return;
  const int64_t begin = s.bucket_ptr[k], end = s.bucket_ptr[k + 1];
  if (begin == end) return;
  unsigned long long rec[kTrip];
#pragma unroll
  for (int u = 0; u < kTrip; ++u) {
    const int64_t r = begin + u * kBucketThreads + threadIdx.x;
    rec[u] = s.records[r < end ? r : end - 1];
  }
  for (int c = threadIdx.x; c < kSlots; c += kBucketThreads) tab[c] = ~0ull;
  __syncthreads();
  for (int64_t r0 = begin; r0 < end; r0 += kTrip * kBucketThreads) {
#pragma unroll
    for (int u = 0; u < kTrip; ++u)
      if (r0 + u * kBucketThreads + threadIdx.x < end) table_enter(tab, rec[u], s.error);
    if (r0 + kTrip * kBucketThreads < end) {
#pragma unroll
      for (int u = 0; u < kTrip; ++u) {
        const int64_t r = r0 + (kTrip + u) * kBucketThreads + threadIdx.x;
        rec[u] = s.records[r < end ? r : end - 1];
      }
    }
  }
  __syncthreads();
  const int64_t trips = (end - begin + kTrip * kBucketThreads - 1) / (kTrip * kBucketThreads);
  for (int64_t t = trips - 1; t >= 0; --t) {  // (from the last trip backwards)
    const int64_t r0 = begin + t * (kTrip * kBucketThreads);
#pragma unroll
    for (int u = 0; u < kTrip; ++u)
      if (r0 + u * kBucketThreads + threadIdx.x < end) {
        const uint32_t key = static_cast<uint32_t>(rec[u] >> 32);
        s.first[static_cast<uint32_t>(rec[u])] = table_first(tab, tab[slot_of(key)], key);
      }
    if (t > 0) {
#pragma unroll
      for (int u = 0; u < kTrip; ++u) rec[u] = s.records[r0 - (kTrip - u) * kBucketThreads + threadIdx.x];
    }
  }
}

// The same over a class's runs.  64 tiles at a time: a lane knows a tile's run, and the runs' pieces
// of up to 64 records -- a run is 8192 / classes records long on average -- are dealt out to the
// waves in turn, a piece a read.
constexpr int kRunTrip = 16;  // pieces of a wave that are asked for together
constexpr int kBucketWaves = kBucketThreads / kWave;
constexpr int kLookTrip = 4;   // slots of a wave's lane that are looked up together

__global__ void __launch_bounds__(kBucketThreads, 8) bins_first_runs_kernel(Bins s, int64_t B) {
  __shared__ unsigned long long tab[kSlots];
  const int64_t k = bucket_of_workgroup(s.plan.bucket_base[B]);
  if (k < 0) return;
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const uint4 at_bucket = s.plan.bucket[k];
  const int64_t tiles = at_bucket.z, row = at_bucket.y, first_item = at_bucket.w;
  const unsigned short* __restrict__ starts = s.run_start + at_bucket.x;
  // The records as they come: put together where they are used (put together here, every read waited for
  // the one before: 17 M items 121 -> 104 us).
  uint32_t id[kRunTrip], in_tile[kRunTrip];
  unsigned int held = 0u;  // which of them are records
  int start = 0, len = 0, ends = 0, pieces = 0;
  // the runs of the 64 tiles from t0 on
  const auto open = [&](int64_t t0) {
    start = len = 0;
    if (t0 + lane < tiles) {
      start = starts[(t0 + lane) * row];
      len = static_cast<int>(starts[(t0 + lane) * row + 1]) - start;
    }
    ends = wave_inclusive_sum((len + kWave - 1) / kWave);
    pieces = __builtin_amdgcn_readlane(ends, kWave - 1);
  };
  // the first position of the tile that piece p is of
  const auto tile_of = [&](int64_t t0, int p) {
    return static_cast<uint32_t>(first_item + (t0 + __popcll(__ballot(ends <= p))) * kTile);
  };
  // the wave's pieces from number p0 on (in steps of the workgroup's waves)
  const auto read = [&](int64_t t0, int p0) {
    held = 0u;
#pragma unroll
    for (int u = 0; u < kRunTrip; ++u) {
      const int p = p0 + u * kBucketWaves;
      if (p >= pieces) break;
      const int j = __popcll(__ballot(ends <= p));
      const int run_len = __builtin_amdgcn_readlane(len, j);
      const int before = __builtin_amdgcn_readlane(ends, j) - (run_len + kWave - 1) / kWave;
      const int at = (p - before) * kWave + lane;
      const int64_t tile_at = first_item + (t0 + j) * kTile;
      // (past the run's end its last record again)
      const int64_t r = tile_at + __builtin_amdgcn_readlane(start, j) + (at < run_len ? at : run_len - 1);
      id[u] = s.run_id[r];
      in_tile[u] = s.run_pos[r];
      if (at < run_len) held |= 1u << u;
    }
  };
  open(0);
  const bool once = tiles <= kWave && pieces <= kRunTrip * kBucketWaves;
  read(0, wave);
  for (int c = threadIdx.x; c < kSlots; c += kBucketThreads) tab[c] = ~0ull;
  __syncthreads();
  for (int64_t t0 = 0; t0 < tiles; t0 += kWave) {
    if (t0 > 0) open(t0);
    for (int p0 = wave; p0 < pieces; p0 += kRunTrip * kBucketWaves) {
      if (t0 > 0 || p0 > wave) read(t0, p0);
#pragma unroll
      for (int u = 0; u < kRunTrip; ++u) {
        if (p0 + u * kBucketWaves >= pieces) break;
        const uint32_t tile_first = tile_of(t0, p0 + u * kBucketWaves);
        uint32_t key = id[u];
        asm volatile("" : "+v"(key));  // (the halves of a record side by side no earlier: 16 registers)
        if (held >> u & 1u)
          table_enter(tab, static_cast<unsigned long long>(key) << 32 | (tile_first + in_tile[u]), s.error);
      }
    }
  }
  __syncthreads();
  for (int64_t t0 = 0; t0 < tiles; t0 += kWave) {
    if (!once) open(t0);
    for (int p0 = wave; p0 < pieces; p0 += kRunTrip * kBucketWaves) {
      if (!once) read(t0, p0);
#pragma unroll
      for (int u0 = 0; u0 < kRunTrip; u0 += kLookTrip) {
        if (p0 + u0 * kBucketWaves >= pieces) break;
        unsigned long long w[kLookTrip];
#pragma unroll
        for (int u = 0; u < kLookTrip; ++u) w[u] = tab[held >> (u0 + u) & 1u ? slot_of(id[u0 + u]) : 0u];
#pragma unroll
        for (int u = 0; u < kLookTrip; ++u) {
          const uint32_t tile_first = tile_of(t0, p0 + (u0 + u) * kBucketWaves);
          if (held >> (u0 + u) & 1u)
            s.first[tile_first + in_tile[u0 + u]] = table_first(tab, w[u], id[u0 + u]);
        }
      }
    }
  }
}

// Positions that are their own first, 64 to a mask word; scan of the counts over all tiles.
// A wave takes WORDS times 64 consecutive positions, one read and one ballot each, and lane l
// keeps the mask of the l-th.
constexpr int kRankTrip = 16;

template <int WORDS>
__global__ void __launch_bounds__(kThreads)
bins_rank_kernel(Bins s, int64_t M, int64_t B, const int64_t* __restrict__ seeds_ptr,
                 const int64_t* __restrict__ ids_ptr, int64_t* __restrict__ num_unique,
                 int64_t* __restrict__ unique_ptr, LookbackState lb, gs_mailbox* box,
                 int64_t box_ticket) {
  __shared__ int64_t s_scan[kThreads / kWave + 1];
  __shared__ int64_t s_prefix;
  constexpr int kTileWords = kThreads / kWave * WORDS;
  __shared__ unsigned long long s_mask[kTileWords];
  __shared__ uint32_t s_before[kTileWords];
  const unsigned int tile = blockIdx.x;
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  const int64_t tile_first = static_cast<int64_t>(tile) * rank_tile(WORDS);
  {  // (M may be a bound: the offsets hold the true count; nothing was stored beyond it)
    const int64_t held = ids_ptr[B] < 0 ? 0 : seeds_ptr[B] + ids_ptr[B];
    if (held < M) M = held;
  }
  unsigned long long m = 0ull;
  const int64_t wave_first = tile_first + wave * (WORDS * kWave);
  if (wave_first < M) {  // (the same for a whole wave)
    for (int w0 = 0; w0 < WORDS; w0 += kRankTrip) {
      uint32_t f[kRankTrip];
#pragma unroll
      for (int u = 0; u < kRankTrip; ++u) {
        const int64_t p = wave_first + (w0 + u) * kWave + lane;
        f[u] = s.first[p < M ? p : M - 1];
      }
#pragma unroll
      for (int u = 0; u < kRankTrip; ++u) {
        const int64_t p = wave_first + (w0 + u) * kWave + lane;
        const unsigned long long own = __ballot(p < M && f[u] == static_cast<uint32_t>(p));
        if (lane == w0 + u) m = own;
      }
    }
  }
  const int64_t mine = __popcll(m);
  int64_t tile_total;
  const int64_t local = block_exclusive_scan<kThreads>(mine, &tile_total, s_scan);
  if (threadIdx.x == 0) lookback_publish_sum(lb, tile, tile_total);
  if (threadIdx.x < kWave) {
    const int64_t before = lookback_exclusive_prefix(lb, tile, tile_total);
    if (threadIdx.x == 0) s_prefix = before;
  }
  __syncthreads();
  const uint32_t before = static_cast<uint32_t>(s_prefix + local);
  if (lane < WORDS) {
    const int word = wave * WORDS + lane;
    s.ranks[static_cast<int64_t>(tile) * kTileWords + word] =
        make_uint4(static_cast<uint32_t>(m), static_cast<uint32_t>(m >> 32), before, 0u);
    // frontier offsets: the rank at every batch's first position, by the thread that owns it
    s_mask[word] = m;
    s_before[word] = before;
  }
  __syncthreads();
  for (int64_t b = threadIdx.x; b < B; b += kThreads) {
    const int64_t p = seeds_ptr[b] + ids_ptr[b] - tile_first;
    if (p >= 0 && p < rank_tile(WORDS))
      unique_ptr[b] = s_before[p >> 6] + __popcll(s_mask[p >> 6] & ((1ull << (p & 63)) - 1ull));
  }
  if (tile == gridDim.x - 1 && threadIdx.x == 0) {
    int64_t total = s_prefix + tile_total;
    const unsigned int err = __hip_atomic_load(lb.error, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (err) total = err == 2u ? -2 : (err == 3u ? -4 : -1);
    if (ids_ptr[B] < 0) total = -1;  // the producer of the ids failed: nothing was relabelled
    *num_unique = total;
    unique_ptr[B] = total;
    post_mailbox(box, total, box_ticket);
  }
}

// The last pass, in the order of the positions: the rank of an item's first position is the
// count before its 64 positions plus the bits below it.  First occurrences write the frontier
// (neighbours side by side), ids -- not seeds -- their rank in their batch.  Tiles of
// consecutive positions go to one XCD one after the other: the ranks a batch looks up are a
// few dozen kilobytes.
constexpr int kRenameItems = 8;
constexpr int kRenameTile = kThreads * kRenameItems;

struct RenameShared {
  int64_t seeds_ptr[kStagedBatches + 1];
  int64_t ids_ptr[kStagedBatches + 1];
  int64_t range[2];
};

template <typename IdT>
__global__ void __launch_bounds__(kThreads)
bins_rename_kernel(BatchItems<IdT> x, int64_t M, Bins s, IdT* __restrict__ unique,
                   IdT* __restrict__ out_ids, const int64_t* __restrict__ unique_ptr) {
  __shared__ RenameShared sh;
  // a table was too small: a stored position may be none
  if (__hip_atomic_load(s.error, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return;
  {  // (M may be a bound: the offsets hold the true count)
    const int64_t held = x.seeds_ptr[x.B] + x.ids_ptr[x.B];
    if (held < M) M = held;
    if (x.ids_ptr[x.B] < 0) return;  // the producer of the ids failed: no records were made
  }
  const int64_t chunks = (M + kRenameTile - 1) / kRenameTile;
  const int64_t per = (chunks + kXcds - 1) / kXcds;
  const int64_t chunk = static_cast<int64_t>(blockIdx.x % kXcds) * per + blockIdx.x / kXcds;
  if (blockIdx.x / kXcds >= per || chunk >= chunks) return;
  const int64_t tile_first = chunk * kRenameTile;
  const int64_t last = tile_first + kRenameTile - 1 < M ? tile_first + kRenameTile - 1 : M - 1;
  uint32_t at[kRenameItems];
#pragma unroll
  for (int u = 0; u < kRenameItems; ++u) {
    const int64_t i = tile_first + u * kThreads + threadIdx.x;
    at[u] = s.first[i < M ? i : M - 1];
  }
  x.stage_offsets(sh.seeds_ptr, sh.ids_ptr);
  // the entries of the first occurrences' positions: one 16-byte read each, all in flight
  uint4 e[kRenameItems];
#pragma unroll
  for (int u = 0; u < kRenameItems; ++u) e[u] = s.ranks[at[u] >> 6];
  int64_t lo, hi;
  x.block_range(tile_first, last, sh.range, &lo, &hi);
  // (reading the ids and the batches' ranks of all eight up front was slower: 94 against 88 us)
#pragma unroll
  for (int u = 0; u < kRenameItems; ++u) {
    const int64_t i = tile_first + u * kThreads + threadIdx.x;
    if (i < M) {
      const unsigned long long m = static_cast<unsigned long long>(e[u].y) << 32 | e[u].x;
      const uint32_t rank = e[u].z + __popcll(m & ((1ull << (at[u] & 63u)) - 1ull));
      const int64_t b = x.batch_of(i, lo, hi);
      const int64_t off = i - x.start(b);
      const int64_t n_seeds = x.seeds_ptr[b + 1] - x.seeds_ptr[b];
      if (at[u] == static_cast<uint32_t>(i)) unique[rank] = *x.where_in(b, i);
      if (off >= n_seeds)
        out_ids[x.ids_ptr[b] + off - n_seeds] =
            static_cast<IdT>(rank - static_cast<uint32_t>(unique_ptr[b]));
    }
  }
}

// The same where the batches are cut into tiles: four workgroups a tile, whose batch is found once
// and not for every item.
template <typename IdT>
__global__ void __launch_bounds__(kThreads, sizeof(IdT) == 8 ? 6 : 8)  // (what fits without spilling)
bins_rename_runs_kernel(BatchItems<IdT> x, Bins s, IdT* __restrict__ unique,
                        IdT* __restrict__ out_ids, const int64_t* __restrict__ unique_ptr) {
  constexpr int kParts = kTile / kRenameTile;
  // a table was too small: a stored position may be none
  if (__hip_atomic_load(s.error, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return;
  const int64_t chunks = static_cast<int64_t>(s.plan.tile_base[x.B]) * kParts;
  const int64_t per = (chunks + kXcds - 1) / kXcds;
  const int64_t chunk = static_cast<int64_t>(blockIdx.x % kXcds) * per + blockIdx.x / kXcds;
  if (blockIdx.x / kXcds >= per || chunk >= chunks) return;
  const uint32_t tile = static_cast<uint32_t>(chunk / kParts);
  const int64_t b = batch_at(s.plan.tile_base, x.B, tile);
  const int64_t first_seed = x.seeds_ptr[b], n_seeds = x.seeds_ptr[b + 1] - first_seed;
  const int64_t first_id = x.ids_ptr[b];
  const int64_t from = (tile - s.plan.tile_base[b]) * kTile + chunk % kParts * kRenameTile;
  const int64_t left = n_seeds + x.ids_ptr[b + 1] - first_id - from;
  if (left <= 0) return;
  const int n = static_cast<int>(left < kRenameTile ? left : kRenameTile);
  const uint32_t first_item = static_cast<uint32_t>(first_seed + first_id + from);
  uint32_t at[kRenameItems];
#pragma unroll
  for (int u = 0; u < kRenameItems; ++u) {
    const int i = u * kThreads + static_cast<int>(threadIdx.x);
    at[u] = s.first[first_item + (i < n ? i : n - 1)];
  }
  const uint32_t frontier = static_cast<uint32_t>(unique_ptr[b]);
  uint4 e[kRenameItems];
#pragma unroll
  for (int u = 0; u < kRenameItems; ++u) e[u] = s.ranks[at[u] >> 6];
  uint32_t rank[kRenameItems];
#pragma unroll
  for (int u = 0; u < kRenameItems; ++u) {
    const unsigned long long m = static_cast<unsigned long long>(e[u].y) << 32 | e[u].x;
    rank[u] = e[u].z + __popcll(m & ((1ull << (at[u] & 63u)) - 1ull));
  }
  // (the first occurrences' ids all asked for before one is written: 17 M items 68 -> 66 us, 4.5 M 16 -> 13,
  // 0.9 M 6.9 -> 4.9)
  IdT key[kRenameItems];
#pragma unroll
  for (int u = 0; u < kRenameItems; ++u) {
    const int i = u * kThreads + static_cast<int>(threadIdx.x);
    const int64_t off = from + i;
    if (at[u] == first_item + i)
      key[u] = *(off >= n_seeds ? x.ids + first_id + off - n_seeds : x.seeds + first_seed + off);
  }
  // (said once that all are there, or the stores, which are counted with the loads, wait for one another)
  __builtin_amdgcn_s_waitcnt(kLoadsDone);
#pragma unroll
  for (int u = 0; u < kRenameItems; ++u) {
    const int i = u * kThreads + static_cast<int>(threadIdx.x);
    if (i < n) {
      const int64_t off = from + i;
      if (at[u] == first_item + i) unique[rank[u]] = key[u];
      if (off >= n_seeds) out_ids[first_id + off - n_seeds] = static_cast<IdT>(rank[u] - frontier);
    }
  }
}

template <typename IdT>
int binned_impl(const void* seeds, const int64_t* seeds_ptr, const void* ids,
                const int64_t* ids_ptr, int64_t B, int64_t num_seeds, int64_t num_ids,
                void* unique, int64_t* unique_ptr, void* out_ids, int64_t* num_unique,
                void* workspace, size_t workspace_bytes, gs_mailbox* box, int64_t box_ticket,
                hipStream_t stream) {
  const int64_t M = num_seeds + num_ids;
  const int64_t nb = buckets_bound(M, B);
  const int64_t tiles = rank_tiles(M);
  const bool runs = by_runs(M, B);
  Carver ws(workspace, workspace_bytes);
  Bins s = {};
  s.plan.bucket_base = ws.take<uint32_t>(B + 1);
  s.plan.classes = ws.take<uint32_t>(B);
  s.first = ws.take<uint32_t>(M);
  const bool few = M < kRankFewItems;
  s.ranks = ws.take<uint4>(tiles * (rank_tile(few ? kRankWordsFew : kRankWords) / kWave));
  LookbackState lb = carve_lookback(ws, tiles, 1u);
  s.error = lb.error;
  int64_t* scan_ws = nullptr;
  if (runs) {
    s.plan.tile_base = ws.take<uint32_t>(B + 1);
    s.plan.row_base = ws.take<uint32_t>(B);
    s.plan.bucket = ws.take<uint4>(nb);
    s.run_id = ws.take<uint32_t>(M);
    s.run_pos = ws.take<unsigned short>(M);
    s.run_start = ws.take<unsigned short>(starts_bound(M, B));
  } else {
    s.count = ws.take<uint32_t>(nb);
    s.fill = ws.take<uint32_t>(nb);
    s.bucket_ptr = ws.take<int64_t>(nb + 1);
    s.bucket_batch = ws.take<uint32_t>(nb);
    scan_ws = ws.take<int64_t>(scan_num_tiles(nb) + 1);
    s.records = ws.take<unsigned long long>(M);
  }
  if (!ws.ok) {
    set_error_text("gs_batch_csr_relabel: workspace needs %zu bytes, 256-byte aligned",
                   binned_relabel_workspace_bytes(M, B));
    return GS_ERR_WORKSPACE;
  }
  BatchItems<IdT> x{static_cast<const IdT*>(seeds), seeds_ptr, static_cast<const IdT*>(ids), ids_ptr,
                    B};
  // a workgroup per bucket (the bound: the number of buckets is on the device), rounded up so
  // that every XCD's share is whole
  const unsigned bucket_grid = static_cast<unsigned>((nb + kXcds - 1) / kXcds * kXcds);
  if (runs) {
    {
      ProfileScope prof("bins_plan", stream);
      hipLaunchKernelGGL((bins_plan_kernel<IdT, true>), dim3(1), dim3(512), 0, stream, x, s.plan, lb,
                         tiles);
    }
    {
      ProfileScope prof("bins_tiles", stream);
      hipLaunchKernelGGL(bins_tiles_kernel<IdT>, dim3(static_cast<unsigned>(tiles_bound(M, B))),
                         dim3(kTileThreads), 0, stream, x, s);
    }
    ProfileScope prof("bins_first", stream);
    hipLaunchKernelGGL(bins_first_runs_kernel, dim3(bucket_grid), dim3(kBucketThreads), 0, stream, s, B);
  } else {
    const int64_t n_init = tiles > nb ? tiles : nb;
    {
      ProfileScope prof("bins_init", stream);
      hipLaunchKernelGGL(bins_init_kernel, dim3(blocks_for(n_init, kThreads)), dim3(kThreads), 0,
                         stream, s, nb, lb, tiles);
      hipLaunchKernelGGL((bins_plan_kernel<IdT, false>), dim3(1), dim3(512), 0, stream, x, s.plan,
                         lb, tiles);
    }
    const unsigned part_grid = static_cast<unsigned>(blocks_for(M, kPartTile));
    {
      ProfileScope prof("bins_count", stream);
      hipLaunchKernelGGL((bins_partition_kernel<IdT, false, kCounterCap>), dim3(part_grid),
                         dim3(kThreads), 0, stream, x, M, s);
    }
    GS_RETURN_IF_ERROR(exclusive_scan(CountOf{s.count}, nb, s.bucket_ptr, scan_ws, stream));
    {
      ProfileScope prof("bins_scatter", stream);
      hipLaunchKernelGGL((bins_partition_kernel<IdT, true, kCounterCap>), dim3(part_grid),
                         dim3(kThreads), 0, stream, x, M, s);
    }
    ProfileScope prof("bins_first", stream);
    hipLaunchKernelGGL(bins_first_kernel, dim3(bucket_grid), dim3(kBucketThreads), 0, stream, s, B);
  }
  {
    ProfileScope prof("bins_rank", stream);
    hipLaunchKernelGGL((few ? bins_rank_kernel<kRankWordsFew> : bins_rank_kernel<kRankWords>),
                       dim3(static_cast<unsigned>(tiles)), dim3(kThreads), 0, stream, s, M, B, seeds_ptr,
                       ids_ptr, num_unique, unique_ptr, lb, box, box_ticket);
  }
  ProfileScope prof("bins_rename", stream);
  if (runs) {
    const int64_t most = tiles_bound(M, B) * (kTile / kRenameTile);
    hipLaunchKernelGGL(bins_rename_runs_kernel<IdT>,
                       dim3(static_cast<unsigned>((most + kXcds - 1) / kXcds * kXcds)), dim3(kThreads),
                       0, stream, x, s, static_cast<IdT*>(unique), static_cast<IdT*>(out_ids),
                       static_cast<const int64_t*>(unique_ptr));
    return check_launch("batch_csr_relabel (binned)");
  }
  const int64_t chunks = (M + kRenameTile - 1) / kRenameTile;
  hipLaunchKernelGGL(bins_rename_kernel<IdT>,
                     dim3(static_cast<unsigned>((chunks + kXcds - 1) / kXcds * kXcds)), dim3(kThreads),
                     0, stream, x, M, s, static_cast<IdT*>(unique), static_cast<IdT*>(out_ids),
                     static_cast<const int64_t*>(unique_ptr));
  return check_launch("batch_csr_relabel (binned)");
}

}  // namespace

size_t binned_relabel_workspace_bytes(int64_t M, int64_t B) {
  if (M < 0) M = 0;
  if (B < 1) B = 1;
  const int64_t nb = buckets_bound(M, B);
  const int64_t tiles = rank_tiles(M);
  const size_t items = static_cast<size_t>(M > 0 ? M : 1);
  const size_t both = 2 * padded((B + 1) * 4) + 2 * padded(B * 4) + padded(items * 4) +
                      padded(tiles * kThreads * 16) + lookback_state_bytes(tiles);
  const size_t runs = padded(items * 4) + padded(items * 2) + padded(starts_bound(M, B) * 2) +
                      padded(nb * 16);
  const size_t scattered = 3 * padded(nb * 4) + padded((nb + 1) * 8) + scan_workspace_bytes(nb) +
                           padded(items * 8);
  // (the caller may have sized this for another number of batches, and with it the other form)
  return both + (runs > scattered ? runs : scattered);
}

bool binned_relabel_applies(int64_t M, int64_t B) {
  // Fewer items are quicker by the regions' four launches than by five.  Skewed ids of 2 M nodes,
  // us, regions / bins, in 1 | 4 | 64 batches: 64 k items 36/40 33/41 35/32, 128 k 46/40 42/41 40/40,
  // 256 k 70/46 54/41 50/45, 512 k 107/53 92/42 73/47, 2 M 178/127 220/67 223/64, 4 M 283/228
  // 337/136 402/88 (the last of one batch by counting and scattering).
  // Positions ride in 32 bits; the batch offsets must fit the kernels' LDS copies.
  return M >= (int64_t(1) << 17) && M < (int64_t(1) << 32) && B >= 1 &&
         B <= static_cast<int64_t>(kStagedBatches);
}

int batch_relabel_binned(const void* seeds, const int64_t* seeds_ptr, const void* ids,
                         const int64_t* ids_ptr, int64_t B, int64_t num_seeds, int64_t num_ids,
                         int id_bytes, void* unique, int64_t* unique_ptr, void* out_ids,
                         int64_t* num_unique, void* workspace, size_t workspace_bytes,
                         gs_mailbox* box, int64_t box_ticket, hipStream_t stream) {
  const auto impl = id_bytes == 8 ? binned_impl<int64_t> : binned_impl<int32_t>;
  return impl(seeds, seeds_ptr, ids, ids_ptr, B, num_seeds, num_ids, unique, unique_ptr, out_ids,
              num_unique, workspace, workspace_bytes, box, box_ticket, stream);
}

}  // namespace gs
