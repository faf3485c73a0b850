// Weighted neighbour sampling without replacement (A-Res) on gfx950.
//
// Replaces impl::CSCColSamplingProbsCUDA (reference
// src/cuda/sampling_probs.cu:268; kernel :25-110, which keeps a faiss
// WarpSelect heap per warp and is limited to fanout <= 32, :32).
//
// Every edge of a row with deg > k gets the key log2(u)/w (same order as the
// reference's u^(1/w), :71) and the k largest keys win, emitted in descending
// key order, ties by lower position.  Key and position travel as one 64-bit
// composite (ordered key << 32 | ~position): composites are distinct, so
// "largest k" is unambiguous and bit-reproducible.
//
// Selection is a top-k over at most 2048 edges held in registers, by a rough key first: the
// hardware's log2 and reciprocal instead of the exact recipe with its two divisions.  The k-th
// largest of a wave's 64 lane maxima is a floor that at least k edges reach, so an edge that
// stays below it by more than both keys can be off is dropped at once; the few survivors
// (typically about 2 k) are packed into LDS, get their exact keys, and each counts how many
// survivors beat it -- that count is its place in the output.
//
// Rows up to 256 edges are one wave each; longer ones are cut into chunks of 2048 edges, a
// workgroup each, so that a 10^5-edge hub is spread over fifty workgroups.  What bounds the fill
// is instructions, not bytes (a Philox block per four edges, the keys, the floors: that is why
// exact keys are left to the survivors), then the chain of dependent reads of a task (offsets,
// weights, the picks' ids).  So the chunks are found by a launch of their own that only reads
// offsets, and rows and chunks then go side by side; the last chunk of a row to finish merges
// the row's candidates.
#include <limits>

#include "gs_common.hpp"
#include "gs_one.hpp"

namespace gs {
namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / kWave;
constexpr int64_t kChunk = 2048;          // edges per workgroup task
constexpr int64_t kSmall = 4 * kWave;     // longest row of one wave: 4 edges a lane
constexpr int kMaxFanout = 96;
// Chunks of rows with several that the queue has room for (their candidates are 8 * fanout bytes
// each, whether there are any or not).  Rows beyond are a wave's work each, 256 edges at a time, and
// keep the chip as busy: fanout 10, 300 k rows of 4096 edges (600 k chunks) 4.9 ms, 5.3 with room
// for all; 70 k of 20000 (700 k chunks) 5.2 and 5.7.
constexpr int64_t kHubTasks = 1 << 19;
constexpr int kPlanRows = 1024;           // rows (threads) of a planning workgroup
constexpr int kQueueGrid = 2048;          // workgroups that take chunks

// A row of one chunk, or chunk number (index of this entry - base) of a longer one.
struct Task {
  int64_t row;  // -1: void
  int64_t start, deg, out;
  int64_t base;  // entry of the row's first chunk
};

template <typename IdT>
struct WArgs {
  const int64_t* indptr;
  const IdT* indices;
  const float* probs;
  const IdT* cols;
  int64_t num_cols;
  int64_t S;
  int k;
  uint64_t seed;
  const uint32_t* replay;
  const int64_t* replay_ptr;
  const int64_t* sub_indptr;
  IdT* sub_indices;
  int64_t* select_index;
  IdT* coo_col;
  // edge data that follows the samples: data_out[o] = edge_data[q] for the output o taken at
  // position q; data_out == nullptr: none
  const float* edge_data;
  float* data_out;
  unsigned long long* reserved;  // chunks of rows with several << 32 | rows of one chunk
  // hub_tasks entries of the former, then S of the latter: those with a merge behind them are
  // taken first
  Task* tasks;
  int64_t hub_tasks;
  int64_t* row_base;             // first entry of a row with several chunks
  unsigned int* done;            // [base]: chunks of the row that have left their candidates
  unsigned long long* cand;      // hub_tasks * k composites
};

__device__ __forceinline__ unsigned long long composite(float key, uint32_t pos) {
  return (static_cast<unsigned long long>(float_to_ordered(key)) << 32) | (0xFFFFFFFFu - pos);
}
__device__ __forceinline__ uint32_t composite_pos(unsigned long long c) {
  return 0xFFFFFFFFu - static_cast<uint32_t>(c);
}

// log2(u) / w as the hardware's one-instruction log2 and reciprocal give it.  Over all 2^24
// values of u the first is within 3.1e-7 of log2_u24, the second within 9.2e-8 (measured, gfx950;
// test_rough_keys_stay_within_half_the_slack);
// with the roundings of the product and of the exact quotient a rough key is within 5.3e-7 of the
// exact one.  Weights whose keys could leave the normal range take the exact key.
constexpr float kRoughSlack = 1.9073486e-6f;  // 2^-19: twice that, and some
__device__ __forceinline__ float rough_key(uint32_t x, float w) {
  constexpr uint32_t kLow = 27u << 23, kSpan = 200u << 23;  // 2^-100 <= w < 2^100
  if (__float_as_uint(w) - kLow >= kSpan) return ares_key(x, w);
  const float u = static_cast<float>((x >> 8) + 1u) * 5.9604644775390625e-08f;
  return __builtin_amdgcn_logf(u) * __builtin_amdgcn_rcpf(w);
}

__device__ __forceinline__ float float_from_ordered(uint32_t o) {
  return __uint_as_float(o & 0x80000000u ? o & 0x7FFFFFFFu : ~o);
}

// four edges a trip: draws, the weights' bits and rough keys (NaN where there is no edge); or composites,
// the upper halves in x, the lower ones in w
template <int TRIPS>
struct Edges {
  uint32_t x[4 * TRIPS], w[4 * TRIPS];
  float rough[4 * TRIPS];
  __device__ __forceinline__ float most() const {
    float m = -__builtin_inff();
#pragma unroll
    for (int u = 0; u < 4 * TRIPS; ++u) m = fmaxf(m, rough[u]);
    return m;
  }
};

// Edges lo + at .. lo + at + 3 of row r (lo a multiple of 4), those below lo + len: one Philox block.
// The weights are read without conditions, the last one again past the end, so that all are on
// their way at once.
template <int TRIPS, typename IdT>
__device__ __forceinline__ void load_edges(const WArgs<IdT>& a, int64_t r, int64_t start, int64_t lo,
                                           int len, int at, int trip, Edges<TRIPS>& e) {
  const int wave_at = __builtin_amdgcn_readfirstlane(at);
  if (wave_at >= len) {  // the whole wave is past the end
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      e.x[trip * 4 + j] = 0u;
      e.w[trip * 4 + j] = 0u;
      e.rough[trip * 4 + j] = __builtin_nanf("");
    }
    return;
  }
  const float* __restrict__ probs = a.probs + (start + lo);
  float w[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) w[j] = probs[at + j < len ? at + j : len - 1];
  U4 x;
  if (a.replay) {
    const uint32_t* rp = a.replay + a.replay_ptr[r] + lo;
#pragma unroll
    for (int j = 0; j < 4; ++j) x.v[j] = rp[at + j < len ? at + j : len - 1];
  } else {
    x = draw_block(a.seed, kTagWeighted, static_cast<uint64_t>(r),
                   static_cast<uint64_t>((lo + at) >> 2));
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    e.x[trip * 4 + j] = x.v[j];
    e.w[trip * 4 + j] = __float_as_uint(w[j]);
    e.rough[trip * 4 + j] = at + j < len ? rough_key(x.v[j], w[j]) : __builtin_nanf("");
  }
}

template <int CTRL, int ROWS>
__device__ __forceinline__ float max_step(float v) {
  return fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(v), __float_as_int(v),
                                                             CTRL, ROWS, 0xf, false)));
}
// the wave's largest value, in every lane
__device__ __forceinline__ float wave_most(float v) {
  v = max_step<0x111, 0xf>(v);  // row_shr:1
  v = max_step<0x112, 0xf>(v);
  v = max_step<0x114, 0xf>(v);
  v = max_step<0x118, 0xf>(v);
  v = max_step<0x142, 0xa>(v);  // row_bcast:15
  v = max_step<0x143, 0xc>(v);  // row_bcast:31
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), kWave - 1));
}

// A value that at least k lanes reach, -inf when fewer than k hold one above that: the k-th
// largest of the lanes' (of equal ones, one at a time).  Taking the largest away k times is ten
// instructions each, comparing every lane with every other 200.
__device__ __forceinline__ float wave_floor(float mine, int k) {
  constexpr int kRounds = 16;
  if (k <= kRounds) {
    float f = -__builtin_inff();
    for (int round = 0; round < k; ++round) {
      f = wave_most(mine);
      const unsigned long long holders = __ballot(mine == f);
      if (static_cast<int>(threadIdx.x & (kWave - 1)) == __ffsll(holders) - 1) mine = -__builtin_inff();
    }
    return f;
  }
  int reach = 0;
#pragma unroll 16
  for (int l = 0; l < kWave; ++l)
    reach += __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(mine), l)) >= mine ? 1 : 0;
  const unsigned long long holder = __ballot(reach == k);
  if (holder)
    return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(mine), __ffsll(holder) - 1));
  return wave_most(reach >= k ? mine : -__builtin_inff());  // equal maxima, or k above 64
}

// (keys are not positive)
__device__ __forceinline__ float floor_with_slack(float f) { return f + f * kRoughSlack; }

// how many of list[0..n) beat `mine`
__device__ __forceinline__ int beaten_by(const unsigned long long* list, int n,
                                         unsigned long long mine) {
  int place = 0;
#pragma unroll 8
  for (int x = 0; x < n; ++x) place += list[x] > mine ? 1 : 0;
  return place;
}

// survivors of a selection: draw << 32 | weight and the edge's place in its chunk, then the composite
struct Shared {
  unsigned long long list[kChunk];  // (a wave that is on its own has a quarter of it)
  unsigned short pos[kChunk];
  unsigned long long best[kMaxFanout];
  float floors[kWaves];
  int n, last;
};
constexpr int kWaveList = kChunk / kWaves;

// packs the edges whose rough key reaches `cut` from list[at] on, in the order (trip, item, lane);
// item j of trip t is edge first + t * step + j of the chunk
template <int TRIPS>
__device__ __forceinline__ void pack(const Edges<TRIPS>& e, float cut, int at, int first, int step,
                                     unsigned long long* list, unsigned short* pos) {
  const int lane = threadIdx.x & (kWave - 1);
  const unsigned long long lower = (1ull << lane) - 1ull;
#pragma unroll
  for (int u = 0; u < 4 * TRIPS; ++u) {
    const bool keep = e.rough[u] >= cut;
    const unsigned long long votes = __ballot(keep);
    if (keep) {
      const int slot = at + __popcll(votes & lower);
      list[slot] = (static_cast<unsigned long long>(e.x[u]) << 32) | e.w[u];
      pos[slot] = static_cast<unsigned short>(first + (u >> 2) * step + (u & 3));
    }
    at += __popcll(votes);
  }
}
template <int TRIPS>
__device__ __forceinline__ int count_kept(const Edges<TRIPS>& e, float cut) {
  int n = 0;
#pragma unroll
  for (int u = 0; u < 4 * TRIPS; ++u) n += __popcll(__ballot(e.rough[u] >= cut));
  return n;
}

__device__ __forceinline__ unsigned long long exact_composite(unsigned long long packed,
                                                              uint32_t pos) {
  return composite(ares_key(static_cast<uint32_t>(packed >> 32),
                            __uint_as_float(static_cast<uint32_t>(packed))),
                   pos);
}

// The k best of the wave's edges [lo, lo + 256) and of the k composites in `best` (null: none) go to
// emit(place, composite), called once per winner by the lane that holds it in the end.  `list`
// and `pos` are the wave's own.  Every lane of the wave calls this.
template <typename Emit>
__device__ __forceinline__ void wave_topk(const Edges<1>& e, int64_t lo,
                                          const unsigned long long* best,
                                          unsigned long long* list, unsigned short* pos, int k,
                                          Emit emit) {
  const int lane = threadIdx.x & (kWave - 1);
  const float cut = floor_with_slack(wave_floor(e.most(), k));
  int n = count_kept(e, cut);
  pack(e, cut, 0, 4 * lane, 0, list, pos);
  // the wave's own stores must have landed before other lanes read them back
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup", "local");
  for (int i = lane; i < n; i += kWave)
    list[i] = exact_composite(list[i], static_cast<uint32_t>(lo) + pos[i]);
  if (best) {
    for (int i = lane; i < k; i += kWave) list[n + i] = best[i];
    n += k;
  }
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup", "local");
  for (int i = lane; i < n; i += kWave) {
    const unsigned long long mine = list[i];
    const int place = beaten_by(list, n, mine);
    if (place < k) emit(place, mine);
  }
  // the list is free again only when every lane has finished reading it
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup", "local");
}

// The k best of a workgroup's edges [lo, lo + 2048), or composites; returns how many there were.
// Every thread calls this; item j of trip t is edge lo + 4 * (t * 256 + the thread's number) + j.
// Every lane of the first `full` waves holds items: ceil(k / full) in each of them reach the
// lowest of these waves' floors.
template <bool COMPOSITES, int TRIPS, typename Emit>
__device__ __forceinline__ int group_topk(const Edges<TRIPS>& e, int64_t lo, int full,
                                          Shared& s, int k, Emit emit) {
  static_assert(4 * TRIPS * kThreads <= kChunk, "the list holds every edge");
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  if (wave < full) {
    const float mine = wave_floor(e.most(), (k + full - 1) / full);
    if (lane == 0) s.floors[wave] = mine;
  }
  if (threadIdx.x == 0) s.n = 0;
  lds_barrier();
  float floor_all = full > 0 ? s.floors[0] : -__builtin_inff();
#pragma unroll
  for (int w = 1; w < kWaves; ++w)
    if (w < full) floor_all = fminf(floor_all, s.floors[w]);
  const float cut = floor_with_slack(floor_all);
  const int count = count_kept(e, cut);
  int at = 0;
  if (lane == 0 && count > 0) at = atomicAdd(&s.n, count);
  at = __builtin_amdgcn_readfirstlane(at);
  if (count > 0) pack(e, cut, at, 4 * static_cast<int>(threadIdx.x), 4 * kThreads, s.list, s.pos);
  lds_barrier();
  const int n = s.n;
  if (!COMPOSITES) {
    for (int i = threadIdx.x; i < n; i += kThreads)
      s.list[i] = exact_composite(s.list[i], static_cast<uint32_t>(lo) + s.pos[i]);
    lds_barrier();
  }
  for (int i = threadIdx.x; i < n; i += kThreads) {
    const unsigned long long one = s.list[i];
    const int place = beaten_by(s.list, n, one);
    if (place < k) emit(place, one);
  }
  lds_barrier();
  return n < k ? n : k;
}

// output o is the edge at position q, of row r
template <typename IdT, bool WITH_COO>
__device__ __forceinline__ void emit_edge(const WArgs<IdT>& a, int64_t r, int64_t o, int64_t q) {
  const IdT id = a.indices[q];
  if (a.data_out) a.data_out[o] = a.edge_data[q];
  a.sub_indices[o] = id;
  a.select_index[o] = q;
  if (WITH_COO) a.coo_col[o] = static_cast<IdT>(r);
}

// Lays out the chunks of the rows above 256 edges: an entry each, a row's one after the other.  A
// workgroup reserves for its 1024 rows at once (a single one does not need the counter, which
// is then not cleared before either).
template <typename IdT>
__global__ void __launch_bounds__(kPlanRows) weighted_plan_kernel(WArgs<IdT> a) {
  __shared__ int64_t s_scan[kPlanRows / kWave + 1];
  __shared__ int64_t s_base;
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t r = static_cast<int64_t>(blockIdx.x) * kPlanRows + threadIdx.x;
  int64_t start = 0, deg = 0, out = 0;
  if (r < a.S) {
    const int64_t col = a.cols ? static_cast<int64_t>(a.cols[r]) : r;
    out = a.sub_indptr[r];
    // an id outside [0, num_cols) is an empty column
    if (static_cast<uint64_t>(col) < static_cast<uint64_t>(a.num_cols)) {
      start = a.indptr[col];
      deg = a.indptr[col + 1] - start;
    }
  }
  const int64_t chunks = deg > kChunk ? (deg + kChunk - 1) / kChunk : 0;
  const bool single = deg > kSmall && chunks == 0;
  int64_t total;
  int64_t at = block_exclusive_scan<kPlanRows>((chunks << 32) | (single ? 1 : 0), &total, s_scan);
  if (threadIdx.x == 0) {
    if (gridDim.x == 1) {
      *a.reserved = static_cast<unsigned long long>(total);
      s_base = 0;
    } else {
      s_base = static_cast<int64_t>(atomicAdd(a.reserved, static_cast<unsigned long long>(total)));
    }
  }
  __syncthreads();
  at += s_base;
  if (single) {
    const int64_t e = a.hub_tasks + (at & 0xFFFFFFFF);
    a.tasks[e] = Task{r, start, deg, out, e};
  }
  at >>= 32;
  // a row whose chunks do not all fit is left to its wave of the fill (its entries are void)
  const Task t{at + chunks <= a.hub_tasks ? r : -1, start, deg, out, at};
  if (chunks > 0) {
    a.row_base[r] = at;
    if (at < a.hub_tasks) a.done[at] = 0u;
  }
  // a few entries are written by the row's lane, many by its whole wave
  constexpr int64_t kFew = 4;
  if (chunks <= kFew)
    for (int64_t e = at; e < at + chunks && e < a.hub_tasks; ++e) a.tasks[e] = t;
  unsigned long long hubs = __ballot(chunks > kFew);
  while (hubs) {
    const int l = __ffsll(hubs) - 1;
    hubs &= hubs - 1;
    const Task h{__shfl(t.row, l, kWave), __shfl(t.start, l, kWave), __shfl(t.deg, l, kWave),
                 __shfl(t.out, l, kWave), __shfl(t.base, l, kWave)};
    const int64_t n = __shfl(chunks, l, kWave);
    for (int64_t e = h.base + lane; e < h.base + n && e < a.hub_tasks; e += kWave) a.tasks[e] = h;
  }
}

// a chunk: its k largest go to the output when it is the row's only one, else to cand, and the
// row's last chunk to get there merges them
template <typename IdT, bool WITH_COO>
__device__ __forceinline__ void run_task(const WArgs<IdT>& a, const Task& e, int64_t t, Shared& s) {
  const auto emit_final = [&](int j, unsigned long long c) {
    emit_edge<IdT, WITH_COO>(a, e.row, e.out + j, e.start + composite_pos(c));
  };
  const int64_t lo = (t - e.base) * kChunk;
  const int len = static_cast<int>(kChunk < e.deg - lo ? kChunk : e.deg - lo);
  constexpr int kTrips = kChunk / (4 * kThreads);
  Edges<kTrips> edges;
#pragma unroll
  for (int trip = 0; trip < kTrips; ++trip)
    load_edges(a, e.row, e.start, lo, len, 4 * static_cast<int>(threadIdx.x + trip * kThreads), trip,
               edges);
  const int full_here = len >= kWaves * kSmall ? kWaves : len / static_cast<int>(kSmall);
  if (e.deg <= kChunk) {
    group_topk<false>(edges, lo, full_here, s, a.k, emit_final);
    return;
  }
  unsigned long long* out = a.cand + static_cast<size_t>(t) * a.k;
  const int found = group_topk<false>(edges, lo, full_here, s, a.k, [&](int j, unsigned long long c) { lb_store(&out[j], c); });
  for (int j = found + threadIdx.x; j < a.k; j += kThreads) lb_store(&out[j], 0ull);  // fewer than k edges
  const int64_t chunks = (e.deg + kChunk - 1) / kChunk;
  // The candidates are stored and read with device scope, past the caches, so all that the count
  // needs before it is that they have arrived: every thread waits for its OWN stores (the
  // vector-memory counter; neither a workgroup-scope release nor the barrier waits for it) and only
  // then meets the others.  (An L2 released per chunk: 52 us a fill, so 30.)
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __syncthreads();
  if (threadIdx.x == 0)
    s.last = __hip_atomic_fetch_add(&a.done[e.base], 1u, __ATOMIC_RELAXED,
                                    __HIP_MEMORY_SCOPE_AGENT) == static_cast<unsigned>(chunks - 1);
  __syncthreads();
  if (!s.last) return;
  // 2048 candidates at a time, from the second time on the k best so far in front of the next
  // ones (k of them: the row's first chunk is full)
  const int64_t m = chunks * a.k;
  const unsigned long long* src = a.cand + static_cast<size_t>(e.base) * a.k;
  int64_t taken = 0;
  int kept = 0, full = 0;
  while (true) {
#pragma unroll
    for (int u = 0; u < 4 * kTrips; ++u) {
      const int i = u * kThreads + static_cast<int>(threadIdx.x);
      const int64_t from = taken + i - kept;
      const unsigned long long c = i < kept ? s.best[i] : (from < m ? lb_load(&src[from]) : 0ull);
      edges.x[u] = static_cast<uint32_t>(c >> 32);
      edges.w[u] = static_cast<uint32_t>(c);
      edges.rough[u] = c ? float_from_ordered(edges.x[u]) : __builtin_nanf("");
    }
    const int64_t here = kept + (m - taken < kChunk - kept ? m - taken : kChunk - kept);
    full = here >= kThreads ? kWaves : static_cast<int>(here) / kWave;
    taken += kChunk - kept;
    kept = a.k;
    if (taken >= m) break;
    group_topk<true>(edges, 0, full, s, a.k, [&](int j, unsigned long long c) { s.best[j] = c; });
  }
  group_topk<true>(edges, 0, full, s, a.k, emit_final);
}

// Workgroups below kQueueGrid take chunks, the others four rows each, a wave a row: deg <= k: copy;
// deg <= 256: select here; longer: the row's chunks are somebody else's.
// 5000 columns of 233 k with 114.6 M edges, fanout 25 (2.6 M edges looked at): 26 us and 6 for the
// layout; as rows, chunks and merge one after the other, with exact keys for all, it was 51.
// A third of that is instructions, the rest the trips of a task: two rounds of workgroups.
template <typename IdT, bool WITH_COO>
__global__ void __launch_bounds__(kThreads) weighted_fill_kernel(WArgs<IdT> a) {
  __shared__ Shared s;
  const int64_t chunks = static_cast<int64_t>(*a.reserved >> 32);
  if (blockIdx.x < kQueueGrid) {
    const int64_t hubs = chunks < a.hub_tasks ? chunks : a.hub_tasks;
    const int64_t n = hubs + static_cast<int64_t>(*a.reserved & 0xFFFFFFFFu);
    for (int64_t i = blockIdx.x; i < n; i += kQueueGrid) {
      const int64_t t = i < hubs ? i : a.hub_tasks + i - hubs;
      const Task e = a.tasks[t];
      if (e.row >= 0) run_task<IdT, WITH_COO>(a, e, t, s);
    }
    return;
  }
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x / kWave;
  const int64_t r = static_cast<int64_t>(blockIdx.x - kQueueGrid) * kWaves + wave;
  if (r >= a.S) return;
  const int64_t c = a.cols ? static_cast<int64_t>(a.cols[r]) : r;
  if (static_cast<uint64_t>(c) >= static_cast<uint64_t>(a.num_cols)) return;
  const int64_t start = a.indptr[c];
  const int64_t deg = a.indptr[c + 1] - start;
  const int64_t out = a.sub_indptr[r];
  if (deg <= a.k) {
    for (int64_t j = lane; j < deg; j += kWave)
      emit_edge<IdT, WITH_COO>(a, r, out + j, start + j);
    return;
  }
  unsigned long long* list = s.list + wave * kWaveList;
  unsigned short* pos = s.pos + wave * kWaveList;
  const auto emit_final = [&](int j, unsigned long long cmp) {
    emit_edge<IdT, WITH_COO>(a, r, out + j, start + composite_pos(cmp));
  };
  Edges<1> edges;
  if (deg <= kSmall) {
    load_edges(a, r, start, 0, static_cast<int>(deg), 4 * lane, 0, edges);
    wave_topk(edges, 0, nullptr, list, pos, a.k, emit_final);
    return;
  }
  if (deg <= kChunk || chunks <= a.hub_tasks ||
      a.row_base[r] + (deg + kChunk - 1) / kChunk <= a.hub_tasks)
    return;
  // a row that found the queue full: 256 edges at a time, the k best so far beside them
  static_assert(kSmall + 2 * kMaxFanout <= kWaveList, "the quarter holds both and the best of them");
  unsigned long long* best = list + kSmall + kMaxFanout;
  for (int64_t lo = 0; lo < deg; lo += kSmall) {
    load_edges(a, r, start, lo, static_cast<int>(kSmall < deg - lo ? kSmall : deg - lo), 4 * lane, 0,
               edges);
    wave_topk(edges, lo, lo > 0 ? best : nullptr, list, pos, a.k,
              [&](int j, unsigned long long cmp) { best[j] = cmp; });
  }
  for (int j = lane; j < a.k; j += kWave) emit_final(j, best[j]);
}

__global__ void __launch_bounds__(kThreads)
weighted_keys_kernel(const uint32_t* __restrict__ draws, const float* __restrict__ weights, int64_t n,
                     float* __restrict__ exact, float* __restrict__ rough) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
  if (i >= n) return;
  exact[i] = ares_key(draws[i], weights[i]);
  rough[i] = rough_key(draws[i], weights[i]);
}

static __global__ void zero_kernel(unsigned long long* p) { *p = 0; }

template <typename IdT, bool WITH_COO>
int weighted_launch(const WArgs<IdT>& a, hipStream_t st) {
  const unsigned plan = static_cast<unsigned>((a.S + kPlanRows - 1) / kPlanRows);
  ProfileScope prof("sample_weighted", st);
  if (plan > 1) hipLaunchKernelGGL(zero_kernel, dim3(1), dim3(1), 0, st, a.reserved);
  hipLaunchKernelGGL((weighted_plan_kernel<IdT>), dim3(plan), dim3(kPlanRows), 0, st, a);
  hipLaunchKernelGGL((weighted_fill_kernel<IdT, WITH_COO>),
                     dim3(static_cast<unsigned>(kQueueGrid + (a.S + kWaves - 1) / kWaves)),
                     dim3(kThreads), 0, st, a);
  return check_launch("sample_weighted");
}

template <typename IdT>
int weighted_impl(const int64_t* indptr, int64_t num_cols, const void* indices, const float* probs,
                  const void* cols, int64_t S, int64_t k, uint64_t seed, const uint32_t* replay,
                  const int64_t* replay_ptr, const int64_t* sub_indptr, void* sub_indices,
                  int64_t* select_index, void* coo_col, const float* edge_data, float* data_out,
                  int64_t queue_chunks, void* workspace, size_t workspace_bytes, hipStream_t st) {
  Carver ws(workspace, workspace_bytes);
  WArgs<IdT> a;
  a.indptr = indptr;
  a.indices = static_cast<const IdT*>(indices);
  a.probs = probs;
  a.cols = static_cast<const IdT*>(cols);
  a.num_cols = num_cols;
  a.S = S;
  a.k = static_cast<int>(k);
  a.seed = seed;
  a.replay = replay;
  a.replay_ptr = replay_ptr;
  a.sub_indptr = sub_indptr;
  a.sub_indices = static_cast<IdT*>(sub_indices);
  a.select_index = select_index;
  a.coo_col = static_cast<IdT*>(coo_col);
  a.edge_data = edge_data;
  a.data_out = data_out;
  a.reserved = ws.take<unsigned long long>(1);
  a.hub_tasks = queue_chunks < kHubTasks ? queue_chunks : kHubTasks;
  a.tasks = ws.take<Task>(static_cast<size_t>(a.hub_tasks + S));
  a.row_base = ws.take<int64_t>(static_cast<size_t>(S));
  a.done = ws.take<unsigned int>(static_cast<size_t>(a.hub_tasks));
  a.cand = ws.take<unsigned long long>(static_cast<size_t>(a.hub_tasks) * k);
  if (!ws.ok) {
    set_error_text("gs_sample_weighted_fill: workspace needs %zu bytes, 256-byte aligned",
                   gs_sample_weighted_workspace_bytes(S, k));
    return GS_ERR_WORKSPACE;
  }
  return coo_col ? weighted_launch<IdT, true>(a, st) : weighted_launch<IdT, false>(a, st);
}

// ------------------------------------------------ with replacement (inverse CDF) ----
// Replaces _CSRRowWiseSampleReplaceKernel (reference src/cuda/sampling_probs.cu:112-183).
// The prefix sums of max(prob, 0) over a column are built 64 edges at a time with a
// Kogge-Stone scan over the wave (x[i] += x[i-d], d = 1..32; the running total enters the
// next chunk through its first element, as in the reference's WarpScan loop :147-160) and
// kept in the caller's scratch; then every lane draws picks and searches them.  That chain
// is sequential, so a column is cut into blocks of 2048 edges: each block is scanned from
// zero by a wave of its own, the blocks' totals are added up in order, and entry i of block
// b stands for (sum of the totals before b) + (its value inside the block).  Columns up to
// 2048 edges are one block and one wave; a hub of 300 k edges is 146 waves instead of one
// wave walking 4640 chunks.  The order of the float additions is fixed by that scheme, so a
// host evaluation of the same steps gives the same bits.
constexpr int64_t kCdfBlock = 2048;
constexpr int kMaxBases = 2048;  // block sums of a column kept in LDS: columns up to 4 M edges

// prefix sums of max(prob, 0) over edges [lo, hi) of a column, from zero; returns their total
__device__ __forceinline__ float scan_block(const float* __restrict__ prob, int64_t lo, int64_t hi,
                                            float* __restrict__ out, int lane) {
  float carry = 0.0f;
  for (int64_t base = lo; base < hi; base += kWave) {
    float x = base + lane < hi ? prob[base + lane] : 0.0f;
    if (lane == 0) x += carry;
    x = x > 0.0f ? x : 0.0f;
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
      const float y = __shfl_up(x, d, kWave);
      if (lane >= d) x += y;
    }
    carry = __shfl(x, kWave - 1, kWave);
    if (base + lane < hi) out[base + lane] = x;
  }
  return carry;
}

// pick number j of row r: position `at` of the column that starts at `start`
template <typename IdT, bool WITH_COO>
__device__ __forceinline__ void emit_pick(const IdT* __restrict__ indices, int64_t start, int64_t at,
                                          int64_t r, int64_t slot, IdT* __restrict__ sub_indices,
                                          int64_t* __restrict__ select_index,
                                          IdT* __restrict__ coo_col) {
  sub_indices[slot] = indices[start + at];
  select_index[slot] = start + at;
  if (WITH_COO) coo_col[slot] = static_cast<IdT>(r);
}

__device__ __forceinline__ float pick_point(uint64_t seed, const uint32_t* __restrict__ replay,
                                            int64_t r, int64_t k, int64_t j, float total) {
  const uint32_t xd = replay ? replay[r * k + j]
                             : draw_one(seed, kTagWeighted, static_cast<uint64_t>(r),
                                        static_cast<uint64_t>(j));
  const float u = static_cast<float>((xd >> 8) + 1u) * 5.9604644775390625e-08f;
  return u * total;
}

// One wave per column of at most 2048 edges: scan, then picks.
template <typename IdT, bool WITH_COO>
__global__ void __launch_bounds__(256)
weighted_replace_kernel(const int64_t* __restrict__ indptr, int64_t num_cols,
                        const IdT* __restrict__ indices, const float* __restrict__ probs,
                        const IdT* __restrict__ cols, int64_t S, int64_t k, uint64_t seed,
                        const uint32_t* __restrict__ replay, const int64_t* __restrict__ sub_indptr,
                        const int64_t* __restrict__ cdf_ptr, float* __restrict__ cdf,
                        IdT* __restrict__ sub_indices, int64_t* __restrict__ select_index,
                        IdT* __restrict__ coo_col) {
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t r = static_cast<int64_t>(blockIdx.x) * (blockDim.x / kWave) + threadIdx.x / kWave;
  if (r >= S) return;
  const int64_t c = cols ? static_cast<int64_t>(cols[r]) : r;
  if (c < 0 || c >= num_cols) return;
  const int64_t start = indptr[c];
  const int64_t deg = indptr[c + 1] - start;
  if (deg <= 0 || deg > kCdfBlock) return;  // longer columns: the two kernels below
  float* my_cdf = cdf + cdf_ptr[r];
  const float total = scan_block(probs + start, 0, deg, my_cdf, lane);
  // the wave's own stores must have landed before other lanes read them back
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
  const int64_t out_start = sub_indptr[r];
  for (int64_t j = lane; j < k; j += kWave) {
    const float rnd = pick_point(seed, replay, r, k, j, total);
    // first the block (here the only one) whose last entry exceeds rnd, then inside it: the
    // same steps as for the longer columns.  Prefix sums made by different addition trees
    // need not be monotone to the last bit, so the order of the probes is part of the result.
    int64_t lo = deg, hi = deg;
    if (total > rnd) lo = 0;
    while (lo < hi) {
      const int64_t mid = (lo + hi) >> 1;
      if (my_cdf[mid] <= rnd) lo = mid + 1; else hi = mid;
    }
    if (lo > deg - 1) lo = deg - 1;
    emit_pick<IdT, WITH_COO>(indices, start, lo, r, out_start + j, sub_indices, select_index, coo_col);
  }
}

// Blocks of the longer columns.  The scratch `cdf` is the columns' edges one after the
// other (cdf_ptr), so the work is found without a queue: a wave takes 2048 consecutive
// scratch positions, and at most two columns longer than that can touch them -- the one
// that holds the first position and the one that holds the last.  Of each, at most one
// block STARTS inside the wave's positions; that block is the wave's.
template <typename IdT>
__global__ void __launch_bounds__(256)
replace_blocks_kernel(const int64_t* __restrict__ indptr, const float* __restrict__ probs,
                      const IdT* __restrict__ cols, int64_t S, const int64_t* __restrict__ cdf_ptr,
                      float* __restrict__ cdf) {
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t waves = static_cast<int64_t>(gridDim.x) * (blockDim.x / kWave);
  const int64_t D = cdf_ptr[S];
  for (int64_t g = static_cast<int64_t>(blockIdx.x) * (blockDim.x / kWave) + threadIdx.x / kWave;
       g * kCdfBlock < D; g += waves) {
    const int64_t t0 = g * kCdfBlock;
    const int64_t t1 = t0 + kCdfBlock < D ? t0 + kCdfBlock : D;
    int64_t owner[2];
#pragma unroll
    for (int side = 0; side < 2; ++side) {
      const int64_t at = side == 0 ? t0 : t1 - 1;
      int64_t lo = 0, hi = S + 1;  // first r with cdf_ptr[r] > at
      while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if (cdf_ptr[mid] <= at) lo = mid + 1; else hi = mid;
      }
      owner[side] = lo - 1;
    }
#pragma unroll
    for (int side = 0; side < 2; ++side) {
      const int64_t r = owner[side];
      if (side == 1 && r == owner[0]) break;
      if (r < 0 || r >= S) continue;
      const int64_t region = cdf_ptr[r];
      const int64_t deg = cdf_ptr[r + 1] - region;
      if (deg <= kCdfBlock) continue;
      const int64_t from = (t0 > region ? t0 : region) - region;
      const int64_t p = (from + kCdfBlock - 1) / kCdfBlock * kCdfBlock;  // block start in the column
      if (region + p >= t1 || p >= deg) continue;
      const int64_t c = cols ? static_cast<int64_t>(cols[r]) : r;
      scan_block(probs + indptr[c], p, p + kCdfBlock < deg ? p + kCdfBlock : deg, cdf + region, lane);
    }
  }
}

// One wave per column longer than 2048 edges, after its blocks have been scanned: the
// blocks' totals are added up in order (LDS), then the picks search first the block, then
// inside it, comparing (sum before the block) + (value inside the block).
template <typename IdT, bool WITH_COO>
__global__ void __launch_bounds__(256)
replace_long_kernel(const int64_t* __restrict__ indptr, int64_t num_cols,
                    const IdT* __restrict__ indices, const IdT* __restrict__ cols, int64_t S,
                    int64_t k, uint64_t seed, const uint32_t* __restrict__ replay,
                    const int64_t* __restrict__ sub_indptr, const int64_t* __restrict__ cdf_ptr,
                    const float* __restrict__ cdf, IdT* __restrict__ sub_indices,
                    int64_t* __restrict__ select_index, IdT* __restrict__ coo_col) {
  __shared__ float s_base[256 / kWave][kMaxBases + 1];
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x / kWave;
  const int64_t r = static_cast<int64_t>(blockIdx.x) * (blockDim.x / kWave) + wave;
  if (r >= S) return;
  const int64_t c = cols ? static_cast<int64_t>(cols[r]) : r;
  if (c < 0 || c >= num_cols) return;
  const int64_t start = indptr[c];
  const int64_t deg = indptr[c + 1] - start;
  if (deg <= kCdfBlock) return;
  const float* my_cdf = cdf + cdf_ptr[r];
  const int64_t nblocks = (deg + kCdfBlock - 1) / kCdfBlock;
  const bool staged = nblocks <= kMaxBases;
  float* base = s_base[wave];  // base[b] = sum of the totals of blocks 0 .. b-1
  float total = 0.0f;
  if (staged) {
    for (int64_t b = lane; b < nblocks; b += kWave) {
      const int64_t end = (b + 1) * kCdfBlock < deg ? (b + 1) * kCdfBlock : deg;
      base[b + 1] = my_cdf[end - 1];
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
    if (lane == 0) {
      float acc = 0.0f;
      base[0] = 0.0f;
      for (int64_t b = 0; b < nblocks; ++b) {
        acc = acc + base[b + 1];
        base[b + 1] = acc;
      }
      total = acc;
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
  } else if (lane == 0) {
    for (int64_t b = 0; b < nblocks; ++b) {
      const int64_t end = (b + 1) * kCdfBlock < deg ? (b + 1) * kCdfBlock : deg;
      total = total + my_cdf[end - 1];
    }
  }
  total = __shfl(total, 0, kWave);
  const int64_t out_start = sub_indptr[r];
  for (int64_t j = lane; j < k; j += kWave) {
    const float rnd = pick_point(seed, replay, r, k, j, total);
    // first block whose last entry exceeds rnd, and the sum before it
    int64_t b = 0;
    float before = 0.0f;
    if (staged) {
      int64_t lo = 0, hi = nblocks;
      while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if (base[mid + 1] <= rnd) lo = mid + 1; else hi = mid;
      }
      b = lo;
      before = b < nblocks ? base[b] : 0.0f;
    } else {
      for (; b < nblocks; ++b) {
        const int64_t end = (b + 1) * kCdfBlock < deg ? (b + 1) * kCdfBlock : deg;
        const float next = before + my_cdf[end - 1];
        if (next > rnd) break;
        before = next;
      }
    }
    int64_t at = deg - 1;
    if (b < nblocks) {
      int64_t lo = b * kCdfBlock;
      int64_t hi = lo + kCdfBlock < deg ? lo + kCdfBlock : deg;
      while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if (before + my_cdf[mid] <= rnd) lo = mid + 1; else hi = mid;
      }
      at = lo > deg - 1 ? deg - 1 : lo;
    }
    emit_pick<IdT, WITH_COO>(indices, start, at, r, out_start + j, sub_indices, select_index, coo_col);
  }
}

template <typename IdT, bool WITH_COO>
int weighted_replace_launch(const int64_t* indptr, int64_t num_cols, const IdT* indices,
                            const float* probs, const IdT* cols, int64_t S, int64_t k, uint64_t seed,
                            const uint32_t* replay, const int64_t* sub_indptr, const int64_t* cdf_ptr,
                            float* cdf, IdT* sub_indices, int64_t* select_index, IdT* coo_col,
                            hipStream_t st) {
  const dim3 grid(static_cast<unsigned>((S + 3) / 4)), block(4 * kWave);
  hipLaunchKernelGGL((weighted_replace_kernel<IdT, WITH_COO>), grid, block, 0, st, indptr, num_cols,
                     indices, probs, cols, S, k, seed, replay, sub_indptr, cdf_ptr, cdf, sub_indices,
                     select_index, coo_col);
  hipLaunchKernelGGL((replace_blocks_kernel<IdT>), dim3(512), block, 0, st, indptr, probs, cols, S,
                     cdf_ptr, cdf);
  hipLaunchKernelGGL((replace_long_kernel<IdT, WITH_COO>), grid, block, 0, st, indptr, num_cols,
                     indices, cols, S, k, seed, replay, sub_indptr, cdf_ptr, cdf, sub_indices,
                     select_index, coo_col);
  return check_launch("sample_weighted_replace");
}

template <typename IdT>
int weighted_replace_impl(const int64_t* indptr, int64_t num_cols, const void* indices,
                          const float* probs, const void* cols, int64_t S, int64_t k, uint64_t seed,
                          const uint32_t* replay, const int64_t* sub_indptr, const int64_t* cdf_ptr,
                          float* cdf, void* sub_indices, int64_t* select_index, void* coo_col,
                          hipStream_t st) {
  const IdT* ind = static_cast<const IdT*>(indices);
  const IdT* cl = static_cast<const IdT*>(cols);
  IdT* si = static_cast<IdT*>(sub_indices);
  IdT* cc = static_cast<IdT*>(coo_col);
  return coo_col ? weighted_replace_launch<IdT, true>(indptr, num_cols, ind, probs, cl, S, k, seed,
                                                     replay, sub_indptr, cdf_ptr, cdf, si,
                                                     select_index, cc, st)
                 : weighted_replace_launch<IdT, false>(indptr, num_cols, ind, probs, cl, S, k, seed,
                                                      replay, sub_indptr, cdf_ptr, cdf, si,
                                                      select_index, cc, st);
}

}  // namespace
}  // namespace gs

using namespace gs;

extern "C" {

size_t gs_sample_weighted_workspace_bytes(int64_t S, int64_t fanout) {
  if (S < 0) S = 0;
  if (fanout < 1) fanout = 1;
  const size_t hubs = static_cast<size_t>(kHubTasks);
  return padded(8) + padded((hubs + static_cast<size_t>(S)) * sizeof(Task)) +
         padded(static_cast<size_t>(S) * 8) + padded(hubs * 4) +
         padded(hubs * static_cast<size_t>(fanout) * 8);
}

int gs_weighted_debug_keys(const uint32_t* draws, const float* weights, int64_t n, float* exact,
                           float* rough, void* stream) {
  GS_REQUIRE(n >= 0 && n < (int64_t(1) << 31) && (n == 0 || (draws && weights && exact && rough)),
             "gs_weighted_debug_keys: null pointer or size");
  if (n == 0) return GS_OK;
  hipLaunchKernelGGL(weighted_keys_kernel, dim3(static_cast<unsigned>(blocks_for(n, kThreads))),
                     dim3(kThreads), 0, static_cast<hipStream_t>(stream), draws, weights, n, exact, rough);
  return check_launch("weighted_debug_keys");
}

int gs_sample_weighted_fill_queue(const int64_t* indptr, int64_t num_cols, const void* indices,
                                  const float* probs, const void* column_ids, int id_bytes,
                                  int64_t S, int64_t fanout, uint64_t seed, const uint32_t* replay,
                                  const int64_t* replay_ptr, const int64_t* sub_indptr,
                                  void* sub_indices, int64_t* select_index, void* coo_col,
                                  const float* edge_data, float* data_out, int64_t queue_chunks,
                                  void* workspace, size_t workspace_bytes, void* stream) {
  GS_REQUIRE(indptr && sub_indptr && S >= 0 && fanout >= 0 && num_cols >= 0,
             "gs_sample_weighted_fill: null pointer or negative size");
  GS_REQUIRE(column_ids || S <= num_cols,
             "gs_sample_weighted_fill: S exceeds num_cols without column_ids");
  GS_REQUIRE(valid_id_bytes(id_bytes), "gs_sample_weighted_fill: id_bytes must be 4 or 8, got %d",
             id_bytes);
  GS_REQUIRE((replay == nullptr) == (replay_ptr == nullptr),
             "gs_sample_weighted_fill: replay and replay_ptr must be given together");
  if (S == 0 || fanout == 0) return GS_OK;
  GS_REQUIRE(indices && probs && sub_indices && select_index,
             "gs_sample_weighted_fill: null buffer");
  GS_REQUIRE((edge_data == nullptr) == (data_out == nullptr),
             "gs_sample_weighted_fill: edge_data and data_out go together");
  GS_REQUIRE(queue_chunks >= 1, "gs_sample_weighted_fill: a queue without room");
  if (fanout > kMaxFanout) {
    set_error_text("gs_sample_weighted_fill: fanout %lld above the supported %d "
                   "(the reference stops at 32)",
                   static_cast<long long>(fanout), kMaxFanout);
    return GS_ERR_UNSUPPORTED;
  }
  hipStream_t st = static_cast<hipStream_t>(stream);
  const auto impl = id_bytes == 8 ? weighted_impl<int64_t> : weighted_impl<int32_t>;
  return impl(indptr, num_cols, indices, probs, column_ids, S, fanout, seed, replay, replay_ptr,
              sub_indptr, sub_indices, select_index, coo_col, edge_data, data_out, queue_chunks,
              workspace, workspace_bytes, st);
}

int gs_sample_weighted_fill_data(const int64_t* indptr, int64_t num_cols, const void* indices,
                                 const float* probs, const void* column_ids, int id_bytes,
                                 int64_t S, int64_t fanout, uint64_t seed, const uint32_t* replay,
                                 const int64_t* replay_ptr, const int64_t* sub_indptr,
                                 void* sub_indices, int64_t* select_index, void* coo_col,
                                 const float* edge_data, float* data_out, void* workspace,
                                 size_t workspace_bytes, void* stream) {
  return gs_sample_weighted_fill_queue(indptr, num_cols, indices, probs, column_ids, id_bytes, S,
                                       fanout, seed, replay, replay_ptr, sub_indptr, sub_indices,
                                       select_index, coo_col, edge_data, data_out,
                                       std::numeric_limits<int64_t>::max(), workspace, workspace_bytes,
                                       stream);
}

int gs_sample_weighted_fill(const int64_t* indptr, int64_t num_cols, const void* indices,
                            const float* probs, const void* column_ids, int id_bytes, int64_t S,
                            int64_t fanout,
                            uint64_t seed, const uint32_t* replay, const int64_t* replay_ptr,
                            const int64_t* sub_indptr, void* sub_indices, int64_t* select_index,
                            void* coo_col, void* workspace, size_t workspace_bytes, void* stream) {
  return gs_sample_weighted_fill_data(indptr, num_cols, indices, probs, column_ids, id_bytes, S,
                                      fanout, seed, replay, replay_ptr, sub_indptr, sub_indices,
                                      select_index, coo_col, nullptr, nullptr, workspace,
                                      workspace_bytes, stream);
}

int gs_sample_weighted_replace(const int64_t* indptr, int64_t num_cols, const void* indices,
                               const float* probs, const void* column_ids, int id_bytes, int64_t S,
                               int64_t fanout, uint64_t seed, const uint32_t* replay,
                               const int64_t* sub_indptr, const int64_t* cdf_ptr, float* cdf,
                               void* sub_indices, int64_t* select_index, void* coo_col,
                               void* stream) {
  GS_REQUIRE(indptr && sub_indptr && cdf_ptr && S >= 0 && fanout >= 0 && num_cols >= 0,
             "gs_sample_weighted_replace: null pointer or negative size");
  GS_REQUIRE(column_ids || S <= num_cols,
             "gs_sample_weighted_replace: S exceeds num_cols without column_ids");
  GS_REQUIRE(valid_id_bytes(id_bytes),
             "gs_sample_weighted_replace: id_bytes must be 4 or 8, got %d", id_bytes);
  if (S == 0 || fanout == 0) return GS_OK;
  GS_REQUIRE(indices && probs && cdf && sub_indices && select_index,
             "gs_sample_weighted_replace: null buffer");
  hipStream_t st = static_cast<hipStream_t>(stream);
  return id_bytes == 8
             ? weighted_replace_impl<int64_t>(indptr, num_cols, indices, probs, column_ids, S,
                                              fanout, seed, replay, sub_indptr, cdf_ptr, cdf,
                                              sub_indices, select_index, coo_col, st)
             : weighted_replace_impl<int32_t>(indptr, num_cols, indices, probs, column_ids, S,
                                              fanout, seed, replay, sub_indptr, cdf_ptr, cdf,
                                              sub_indices, select_index, coo_col, st);
}

}  // extern "C"
