// A whole small GraphSAGE minibatch -- every layer's column slice + uniform sample + relabel --
// by ONE workgroup: what gs_layer_sample / gs_layer_relabel do per layer (the reference's calls
// src/cuda/fusion/slice_sampling.cu:157 and src/cuda/tensor_ops.cu:46 per layer, each with a read
// of a size by the host), with the hash table, the frontier and the sizes in LDS.
//
// A minibatch of a few hundred items has no work for more than a few workgroups, and layer by
// layer it is a chain of launches that hand one another counts, table slots and ranks through
// memory: 32 seeds x [10, 5] took five launches, 29 us of kernels, 42 us the call; this is one of
// 12.5 us, 27 us the call.  Only the graph is read from memory, in dependent trips that bound it
// (two a layer: offsets; neighbours, edge data beside them).
//
// One table serves all layers.  A slot is (id << 32 | number), the number of a node being its rank
// in the frontier once it has one, and until then the smallest item number it was met at; layer
// l + 1's items are the frontier (numbers = ranks, already in the table) and then its samples,
// numbered from the frontier's length on, so ranks are smaller than every new item's number and
// one atomic minimum keeps both.  Nothing is entered twice, and a layer needs no pass over the
// nodes of the earlier ones.
#include "gs_one.hpp"
#include "gs_select.hpp"
#include "gs_table.hpp"

namespace gs {
namespace {

constexpr int kOneMaxLayers = 8;
constexpr int64_t kOneMaxItems = 8192;     // seeds and samples of the last layer, at their bound
constexpr int kOneMaxSlots = 2 * kOneMaxItems;  // load <= 1/2: 128 KB
constexpr int64_t kOneMaxColumns = 2048;   // of the last layer, at their bound

struct OneLayer {
  uint64_t seed;
  int64_t* offsets;
  void* out_ids;
  void* frontier;
  float* data_out;
  gs_mailbox* edge_box;
  int64_t edge_ticket;
  gs_mailbox* unique_box;
  int64_t unique_ticket;
  int fanout;
};

struct OneArgs {
  const int64_t* indptr;
  const void* indices;
  const void* seeds;
  int64_t num_cols;
  const float* edge_data;
  const int64_t* edge_ids;
  int64_t* counts;  // [2 * num_layers]: edges, frontier length of every layer
  int num_seeds;
  int num_layers;
  int slots;    // of the table, a power of two
  int columns;  // room for the columns of a later layer
  OneLayer layer[kOneMaxLayers];
};

struct OneShared {
  int scan[2][kOneWaves];
  int counts[2 * kOneMaxLayers];
  int too_wide;
};

// The table's word of a node is its final one, (id << 32 | rank), for the items that are the
// first of theirs: those take the next ranks, in the order of the items, and enter the frontier.
// `flags`: bit u = the lane's item u is the first; key[u], slot[u]: where.
template <typename IdT, int N>
__device__ __forceinline__ void give_ranks(unsigned int flags, const uint32_t (&key)[N],
                                           const uint32_t (&slot)[N], unsigned long long* s_table,
                                           uint32_t* s_cols, int columns, IdT* frontier,
                                           int* unique, OneShared& s, int which) {
  int total;
  int rank = *unique + one_scan(__popc(flags), &total, s.scan, which);
#pragma unroll
  for (int u = 0; u < N; ++u) {
    if (flags >> u & 1u) {
      s_table[slot[u]] = (static_cast<unsigned long long>(key[u]) << 32) | static_cast<uint32_t>(rank);
      if (rank < columns) s_cols[rank] = key[u];
      frontier[rank] = static_cast<IdT>(key[u]);
      ++rank;
    }
  }
  *unique += total;
}

// Layer `l`: columns 0..S-1, whose ids s_from holds, sampled kRows at a time, G lanes a column;
// *unique = the frontier's length so far.  The samples of one such pass are all entered before any
// of them is ranked, and a later pass's items have larger numbers than every item and rank before
// them, so what a pass finds to be a first occurrence is one.
template <typename IdT, int G, bool REPLACE>
__device__ __forceinline__ void one_layer(const OneArgs& a, int l, int S, int* unique,
                                          const PackedTable& t, const uint32_t* s_from,
                                          uint32_t* s_cols, OneShared& s) {
  constexpr int kRows = kOneThreads / G;
  const OneLayer& y = a.layer[l];
  const IdT* __restrict__ indices = static_cast<const IdT*>(a.indices);
  const int k = y.fanout;
  const int sub = threadIdx.x & (G - 1);
  int E = 0;
  for (int r0 = 0; r0 < S; r0 += kRows) {
    const int row = r0 + static_cast<int>(threadIdx.x) / G;
    int64_t start = 0, deg = 0;
    if (row < S) {
      const int64_t c = static_cast<int64_t>(static_cast<IdT>(s_from[row]));
      if (valid_col(c, a.num_cols)) {
        start = a.indptr[c];
        deg = a.indptr[c + 1] - start;
      }
    }
    const int cnt = REPLACE ? (deg > 0 ? k : 0) : static_cast<int>(deg < k ? deg : k);
    uint32_t mine[4] = {0u, 0u, 0u, 0u};
    if (cnt > 0) {
      if (REPLACE) {
        const U4 blk = draw_block(y.seed, kTagUniform, static_cast<uint64_t>(row),
                                  static_cast<uint64_t>(sub));
#pragma unroll
        for (int u = 0; u < 4; ++u) mine[u] = blk.v[u] % static_cast<uint32_t>(deg);
      } else {
        floyd_picks<G>(y.seed, row, sub, k, deg, nullptr, mine);
      }
    }
    // the lane's four reads go out together (its first pick again where it has fewer)
    bool live[4];
    int64_t q[4];
    IdT v[4] = {IdT(0), IdT(0), IdT(0), IdT(0)};
    float w[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      live[u] = 4 * sub + u < cnt;
      q[u] = start + (live[u] ? mine[u] : mine[0]);
    }
    if (live[0]) {
#pragma unroll
      for (int u = 0; u < 4; ++u) v[u] = indices[q[u]];
      if (a.edge_data) {
        if (a.edge_ids) {
#pragma unroll
          for (int u = 0; u < 4; ++u) q[u] = a.edge_ids[q[u]];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) w[u] = a.edge_data[q[u]];
      }
    }
    int total;
    const int ex = one_scan(sub == 0 ? cnt : 0, &total, s.scan, 0);
    const int out = E + (sub == 0 ? ex : ex - cnt);  // the column's first output
    if (row < S && sub == 0) y.offsets[row] = out;
    uint32_t key[4], item[4], at[4];
    unsigned long long seen[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (live[u] && !fits_slot(v[u])) {
        s.too_wide = 1;
        live[u] = false;
      }
      key[u] = live[u] ? static_cast<uint32_t>(v[u]) : 0u;
      item[u] = static_cast<uint32_t>(S + out + 4 * sub + u);
      at[u] = t.home(key[u]);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (live[u]) seen[u] = t.probe(key[u], item[u], at[u]);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (live[u]) {
        while (!t.landed(key[u], item[u], at[u], seen[u])) {
          at[u] = (at[u] + 1) & t.mask;
          seen[u] = t.probe(key[u], item[u], at[u]);
        }
      }
    }
    lds_barrier();
    unsigned int flags = 0u;
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (live[u] && static_cast<uint32_t>(t.slots[at[u]]) == item[u]) flags |= 1u << u;
    // (the scan inside has a barrier: every word has been looked at before one is replaced)
    give_ranks<IdT>(flags, key, at, t.slots, s_cols, a.columns, static_cast<IdT*>(y.frontier), unique,
                    s, 1);
    lds_barrier();
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (4 * sub + u < cnt) {
        const int o = out + 4 * sub + u;
        static_cast<IdT*>(y.out_ids)[o] =
            live[u] ? static_cast<IdT>(static_cast<uint32_t>(t.slots[at[u]])) : IdT(-1);
        if (a.edge_data) y.data_out[o] = w[u];
      }
    }
    E += total;
  }
  if (threadIdx.x == 0) {
    y.offsets[S] = E;
    s.counts[2 * l] = E;
    s.counts[2 * l + 1] = *unique;
  }
}

template <typename IdT, bool REPLACE>
__global__ void __launch_bounds__(kOneThreads) one_minibatch_kernel(OneArgs a) {
  extern __shared__ unsigned long long s_dynamic[];
  __shared__ OneShared s;
  PackedTable t;
  t.slots = s_dynamic;
  t.mask = static_cast<uint32_t>(a.slots - 1);
  t.shift = 64 - (31 - __clz(a.slots));
  uint32_t* s_cols = reinterpret_cast<uint32_t*>(s_dynamic + a.slots);
  uint32_t* s_seeds = s_cols + a.columns;  // the first layer's columns, as they were given
  for (int i = threadIdx.x; i < a.slots; i += kOneThreads) t.slots[i] = ~0ull;
  if (threadIdx.x == 0) s.too_wide = 0;
  lds_barrier();
  // the seeds, 1024 at a time: items 0 .. num_seeds - 1 of the first layer
  const IdT* __restrict__ seeds = static_cast<const IdT*>(a.seeds);
  int unique = 0;
  for (int i0 = 0; i0 < a.num_seeds; i0 += kOneThreads) {
    const int i = i0 + static_cast<int>(threadIdx.x);
    uint32_t key[1] = {0u}, at[1] = {0u};
    bool live = i < a.num_seeds;
    if (live) {
      const IdT id = seeds[i];
      key[0] = static_cast<uint32_t>(id);
      s_seeds[i] = key[0];
      if (!fits_slot(id)) {
        s.too_wide = 1;
        live = false;
      }
    }
    if (live) at[0] = t.template insert<false>(key[0], static_cast<uint32_t>(i));
    lds_barrier();
    const unsigned int first =
        live && static_cast<uint32_t>(t.slots[at[0]]) == static_cast<uint32_t>(i) ? 1u : 0u;
    // the first layer's frontier starts with them; a later layer's is the one before and more
    give_ranks<IdT>(first, key, at, t.slots, s_cols, a.columns,
                    static_cast<IdT*>(a.layer[0].frontier), &unique, s, (i0 / kOneThreads) & 1);
  }
  int S = a.num_seeds;
  for (int l = 0; l < a.num_layers; ++l) {
    lds_barrier();  // ranks and columns of the layer before are there for every wave
    if (l > 0) {
      IdT* frontier = static_cast<IdT*>(a.layer[l].frontier);
      for (int r = threadIdx.x; r < S; r += kOneThreads) frontier[r] = static_cast<IdT>(s_cols[r]);
    }
    const uint32_t* s_from = l == 0 ? s_seeds : s_cols;
    const int k = a.layer[l].fanout;
    if (k <= 4)
      one_layer<IdT, 1, REPLACE>(a, l, S, &unique, t, s_from, s_cols, s);
    else if (k <= 8)
      one_layer<IdT, 2, REPLACE>(a, l, S, &unique, t, s_from, s_cols, s);
    else if (k <= 16)
      one_layer<IdT, 4, REPLACE>(a, l, S, &unique, t, s_from, s_cols, s);
    else
      one_layer<IdT, 8, REPLACE>(a, l, S, &unique, t, s_from, s_cols, s);
    S = unique;
  }
  lds_barrier();
  // every count by a lane of its own: -2 for the frontiers when an id does not fit its slot
  const int i = threadIdx.x;
  if (i < 2 * a.num_layers) {
    const OneLayer& y = a.layer[i >> 1];
    const int64_t n = (i & 1) && s.too_wide ? int64_t(-2) : int64_t(s.counts[i]);
    if (a.counts) a.counts[i] = n;
    post_mailbox(i & 1 ? y.unique_box : y.edge_box, n, i & 1 ? y.unique_ticket : y.edge_ticket);
  }
}

// bounds of a layer's columns: S_0 = seeds, S_l+1 = S_l * (1 + fanout)
bool one_bounds(int64_t num_seeds, int num_layers, const int64_t* fanouts, int64_t* columns,
                int64_t* items) {
  if (num_seeds < 0 || num_seeds > kOneMaxItems || num_layers < 1 || num_layers > kOneMaxLayers)
    return false;
  int64_t S = num_seeds;
  for (int l = 0; l < num_layers; ++l) {
    if (fanouts[l] < 0 || fanouts[l] > GS_FUSED_MAX_FANOUT) return false;
    *columns = S;
    S *= 1 + fanouts[l];
    if (S > kOneMaxItems) return false;
  }
  *items = S;
  return *columns <= kOneMaxColumns;
}

}  // namespace
}  // namespace gs

using namespace gs;

extern "C" {

int gs_minibatch_applies(int64_t num_seeds, int num_layers, const int64_t* fanouts) {
  int64_t columns, items;
  return fanouts && one_bounds(num_seeds, num_layers, fanouts, &columns, &items);
}

int gs_minibatch_sample(const int64_t* indptr, int64_t num_cols, const void* indices,
                        const void* seeds, int id_bytes, int64_t num_seeds, int num_layers,
                        const int64_t* fanouts, int replace, const uint64_t* layer_seeds,
                        const float* edge_data, const int64_t* edge_ids, int64_t* const* sub_indptr,
                        void* const* out_ids, void* const* frontier, float* const* data_out,
                        int64_t* counts, gs_mailbox* const* mailboxes, const int64_t* tickets,
                        void* stream) {
  GS_REQUIRE(valid_id_bytes(id_bytes), "gs_minibatch_sample: id_bytes must be 4 or 8, got %d", id_bytes);
  GS_REQUIRE(fanouts && layer_seeds && sub_indptr && out_ids && frontier && num_cols >= 0,
             "gs_minibatch_sample: null pointer or negative size");
  int64_t columns = 0, items = 0;
  GS_REQUIRE(one_bounds(num_seeds, num_layers, fanouts, &columns, &items),
             "gs_minibatch_sample: sizes beyond gs_minibatch_applies");
  GS_REQUIRE(indptr && (num_seeds == 0 || (seeds && indices)), "gs_minibatch_sample: null pointer");
  GS_REQUIRE(!edge_data || data_out, "gs_minibatch_sample: edge data without data_out");
  GS_REQUIRE(!mailboxes || tickets, "gs_minibatch_sample: mailboxes without tickets");
  OneArgs a{};
  a.indptr = indptr;
  a.indices = indices;
  a.seeds = seeds;
  a.num_cols = num_cols;
  a.edge_data = edge_data;
  a.edge_ids = edge_ids;
  a.counts = counts;
  a.num_seeds = static_cast<int>(num_seeds);
  a.num_layers = num_layers;
  a.slots = 1024;
  while (a.slots < 2 * items) a.slots <<= 1;
  a.columns = static_cast<int>(columns);
  int64_t S = num_seeds;
  for (int l = 0; l < num_layers; ++l) {
    const int64_t cap = S * fanouts[l];
    GS_REQUIRE(sub_indptr[l] && (cap == 0 || (out_ids[l] && (!edge_data || data_out[l]))) &&
                   (S + cap == 0 || frontier[l]),
               "gs_minibatch_sample: null buffer of layer %d", l);
    OneLayer& y = a.layer[l];
    y.seed = layer_seeds[l];
    y.offsets = sub_indptr[l];
    y.out_ids = out_ids[l];
    y.frontier = frontier[l];
    y.data_out = edge_data ? data_out[l] : nullptr;
    if (mailboxes) {
      y.edge_box = mailboxes[2 * l];
      y.edge_ticket = tickets[2 * l];
      y.unique_box = mailboxes[2 * l + 1];
      y.unique_ticket = tickets[2 * l + 1];
    }
    y.fanout = static_cast<int>(fanouts[l]);
    S += cap;
  }
  const size_t lds = static_cast<size_t>(a.slots) * 8 + padded(static_cast<size_t>(columns + num_seeds) * 4);
  auto* kernel = id_bytes == 8 ? (replace ? one_minibatch_kernel<int64_t, true>
                                          : one_minibatch_kernel<int64_t, false>)
                               : (replace ? one_minibatch_kernel<int32_t, true>
                                          : one_minibatch_kernel<int32_t, false>);
  if (lds > 48 * 1024) {  // (per call: the attribute belongs to the device the call runs on)
    const hipError_t allowed =
        hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                            hipFuncAttributeMaxDynamicSharedMemorySize,
                            kOneMaxSlots * 8 + 2 * static_cast<int>(kOneMaxColumns) * 4);
    if (allowed != hipSuccess) {
      set_error_text("gs_minibatch_sample: %s", hipGetErrorString(allowed));
      return GS_ERR_LAUNCH;
    }
  }
  hipStream_t st = static_cast<hipStream_t>(stream);
  ProfileScope prof("minibatch", st);
  hipLaunchKernelGGL(kernel, dim3(1), dim3(kOneThreads), lds, st, a);
  return check_launch("minibatch_sample");
}

}  // extern "C"
