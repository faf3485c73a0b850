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

// Neighbour arrays from this size on, of so many nodes, are read as streams (the line is the first to
// leave the L2) by walkers enough: hardly one of their lines is met again, and the offsets, which are, stay
// longer.  Arrays that the L2s and the memory-side cache hold in good part lose by it, and so do few
// walkers, and graphs of few nodes, however long their lists: the offsets need no room there, and the hubs' lists are
// met again.  With a packed table of the offsets (below) arrays are read plainly.  R-MAT graphs, 32-bit ids, plain / as a
// stream, us, by walkers x steps:
//                                 131 k x 10   131 k x 30   300 k x 8   300 k x 30   1 M x 4   1 M x 80
//   0.13 M nodes x 492 (258 MB)     27.5/32.2    78/93        49/64       178/233      80/105   1467/2039
//   0.13 M x 700 (367 MB)           28.6/32.1    80/94        51/64       183/237      82/106   1482/2084
//   0.23 M x 492 (459 MB)           29.1/32.0    81/94        52/64       184/235      87/106   1501/2058
//   0.5 M x 360 (720 MB)            30.2/30.7    81/92        55/62       187/228      93/104   1563/1995
//   1 M x 100 (419 MB)              28.0/28.0    76/82        51/55       174/194      90/92    1387/1650
//   1 M x 250 (1.0 GB)              30.7/29.4    82/90        56/59       192/217      98/101   1630/1901
//   2.1 M x 25 (210 MB)             23.2/23.9                 42/43       134/139      77/75    1005/1087
//   2.1 M x 50 (419 MB)             26.9/25.7                 49/49       162/169      88/84    1306/1374
//   2.1 M x 100 (839 MB)            29.8/27.7                 54/53       184/191      97/92    1514/1627
//   4.2 M x 25 (419 MB)             24.8/24.0                 45/43       142/138      83/78    1048/1062
//   4.2 M x 50 (839 MB)             28.5/27.3                 52/48       170/165      93/86    1321/1344
//   8.4 M x 16 (537 MB)             23.3/22.5                 42/40                    78/74     888/858
//   16.8 M x 16 (1.1 GB)            24.6/23.4                 46/43                    82/77    1021/856
// (most of the long walks of the last column have a table).  66 k walkers, 30 steps: 2.4 M nodes of 35 edges
// 46.6/48.8, 1 M nodes of 80 48.2/50.9.  64-bit ids: 0.23 M nodes x 492 (917 MB), 300 k x 30 204/241, 4 M x 25 (839 MB)
// 154/142.
constexpr int64_t kStreamBytes = int64_t(5) << 26;
constexpr int64_t kStreamNodes = int64_t(1) << 21;
constexpr int64_t kStreamWalkers = 120'000;
// The same for a relation of a metapath, when the path has two such (of half as many nodes: they share the L2s),
// by any number of walkers.  Three relations, 32-bit ids, plain / as streams, us:
//                                  50 k x 64   100 k x 40   131 k x 30   400 k x 8   1 M x 4   1 M x 10
//   0.3 M nodes x 250 (300 MB)       85/94        99/110                    79/88
//   1 M x 80 (335 MB)                80/80        86/93        82/82        72/74      94/92
//   1 M x 160 (671 MB)               86/84        98/99        88/88        79/79     103/98
//   2.1 M x 50 (419 MB)              80/78        82/81        79/74        71/70      91/87     205/195
//   4.2 M x 25 (419 MB)              77/75        68/67        70/65        67/65      89/85     191/176
// and a path over one relation alone, which takes the line above:
//   1 M x 80 (335 MB)                69/80        75/92                     68/75
//   2.1 M x 50 (419 MB)              71/77        73/80        70/73        68/69      88/85
//   4.2 M x 25 (419 MB)              70/74        63/67        63/60        63/61      84/78     175/166
constexpr int64_t kStreamRelationBytes = int64_t(256) << 20;
constexpr int64_t kStreamRelationNodes = int64_t(1) << 20;
// A metapath's relations have to be looked up for it in front of the first step, which only long work earns
// back: three of 400 MB, 64-bit / 32-bit ids, 131 k walkers, 30 steps 71 -> 66 / 72 -> 66 us, 1 M walkers, 4 steps
// 87 -> 85 / 87 -> 83, but 200 k walkers, 10 steps 42.6 -> 44.5 / 42 -> 43, 18 k walkers, 30 steps 28 -> 34 / 31 -> 37.
constexpr int64_t kStreamSteps = int64_t(3) << 20;

// Draw t of a walker, in a block of four.  (An index would put the block into scratch memory, 20 bytes a
// lane written every four steps and read in every one; the values are named or the compiler picks an address.)
__device__ __forceinline__ uint32_t draw_of(const U4& x, int64_t t) {
  const uint32_t a = x.v[0], b = x.v[1], c = x.v[2], d = x.v[3];
  const uint32_t low = t & 1 ? b : a, high = t & 1 ? d : c;
  return t & 2 ? high : low;
}

// The neighbour that draw x takes of `deg` ones from `start` on; -1: there are none.
template <typename Indices>
__device__ __forceinline__ int64_t neighbour(Indices indices, int64_t start, int64_t deg, uint32_t x,
                                             bool stream) {
  if (deg <= 0) return -1;
  int64_t at = start + static_cast<int64_t>(x % static_cast<uint32_t>(deg));
  int64_t next;
  if (stream) {
    // (held apart from the other by two empty statements, or the compiler makes one plain load
    // of the two)
    asm volatile("" : "+v"(at));
    next = __builtin_nontemporal_load(indices + at);
    asm volatile("" : "+v"(next));
  } else {
    next = indices[at];
  }
  return next;
}

// The offsets of kRecordNodes nodes in 16 bytes: the first node's start in 32 bits, then every node's
// end as its distance from that start, in 16 bits each and in order.  Where that cannot be said (a
// hub among the nodes), the first distance is larger than the last and the offsets themselves are
// read instead.  A step reads a record at once, and what the L2s (4 MB a die) have to hold of the offsets
// is a third: 1 M walkers, 80 steps, 4 M nodes of 50 edges 1321 -> 1148 us with the making of the table
// (11).  60 nodes to a line of 128 bytes, start and two ends read apart, are a fifth smaller and were no better (both
// in the kernel as it was with the draws in scratch memory and the store in front of the offsets): 1 M nodes 1132 us
// against 1166, but 200 k walkers 266 against 263, 4 M nodes of 8 edges 673 against 668.
constexpr int kRecordNodes = 6;

// Whether a table of the offsets is made in front of a walk: where they outgrow an L2 by far or by a little, the
// walkers fill the chip (fewer wait for the longer step instead: 66 k walkers, 38 steps 47 -> 59 us) and the steps earn
// the table back.  Offsets as they are / table, us, 20 to 35 edges a node, walkers x steps:
//                  200 k x 30   300 k x 10   300 k x 20   300 k x 80    1 M x 4      1 M x 10     1 M x 80
//   131 k nodes      70/69        34/34        63/62       217/211       45/44       106/101       701/678
//   262 k            79/76        38/39        72/70       246/237       54/50       124/116       818/774
//   500 k            95/91        46/46        87/83       307/287       67/61       152/140      1018/947
//     2 M           110/101       52/51       100/93       346/307       80/73       174/156      1140/989
//     8 M            93/103       50/62        91/99       286/281       76/86       157/162       954/869
//    16 M            98/120       54/77        96/115      303/308       81/102      167/180       965/904
// The more nodes, the more walkers a table wants, however many steps they take (table_walkers); 16 edges a node, the
// steps from where the line lies, and twice as many:
//                  131 k walkers          300 k                500 k                1 M                  4 M
//     4.2 M        112/120 (25 edges)    138/134 (x 30)
//     8.4 M        152/188               176/188, 296/306     198/207, 345/349     209/221, 380/367     279/272, 464/455
//    16.8 M        256/349               294/307, 452/476     335/346, 551/548     371/367, 646/613     461/434, 806/754
//    33.6 M                              467/505, 687/774     573/563, 852/831     669/651, 1087/1025   845/782, 1481/1340
//    67 M                                697/853, 1084/1296   867/908, 1197/1284   1117/1121, 1669/1650 1445/1394, 2594/2418
// and graphs of more nodes than that want their walks not to end early: 111 M nodes of 8 edges 915/1131 us by 1 M
// walkers, 1551/1733 by 4 M, of 14 edges 1589/1529, 2419/2200 (kWideNodes, kWideDegree; no larger one was measured).
// A record with a hub among its nodes costs three reads one behind the other, and in dense graphs of many
// edges many steps meet one.  As above, by edges a node (kDenseEdges, kDenseDegree):
//                        131 k x 30   300 k x 30    1 M x 4     1 M x 8     1 M x 80
//   262 k nodes x 250      76/75        172/167      82/78       160/151     1428/1346
//   262 k x 492            80/82        183/181      87/82       165/157     1485/1482
//   262 k x 600            80/86        185/192      87/85       164/164     1542/1584
//   262 k x 1000           87/96        208/220      90/95       180/189     1798/1869
//   524 k x 300            80/83        183/182      91/83       170/157     1528/1476
//   524 k x 492            85/94        202/211      94/92       176/181     1725/1768
//     1 M x 160            80/81        183/174      95/84       173/155     1460/1396
//     1 M x 250            82/90        192/199      98/91       178/173     1630/1646
//     1 M x 320            86/95        204/212      99/95       181/185     1739/1774
//     1 M x 492            92/102       219/230     102/101      192/200     1898/1944
//   2.1 M x 200           114/122       209/208                  189/184     1823/1719
//   2.1 M x 300           118/132       218/224                  196/197     1911/1875
//   4.2 M x 200           182/198       205/217                  209/218     1797/1788
constexpr int64_t kMostNodes = int64_t(1) << 27, kWideNodes = int64_t(1) << 26, kWideDegree = 12;
constexpr int64_t kDenseEdges = int64_t(1) << 27, kDenseDegree = 320;

// a walker for so many nodes, 2^17 at the least; a million are enough for any
inline int64_t table_walkers(int64_t num_nodes, int64_t nodes_a_walker) {
  const int64_t n = num_nodes / nodes_a_walker < 1'000'000 ? num_nodes / nodes_a_walker : 1'000'000;
  return n > (int64_t(1) << 17) ? n : int64_t(1) << 17;
}
inline bool steps_pay(int64_t num_nodes, int64_t n, int64_t length) {
  return length > 0 && n > ((int64_t(1) << 21) + num_nodes * 3 / 2 - 1) / length;
}
bool packed_pays(int64_t num_nodes, int64_t nnz, int64_t n, int64_t length) {
  return num_nodes >= (int64_t(1) << 18) && num_nodes <= kMostNodes && nnz < (int64_t(1) << 32) &&
         (num_nodes <= kWideNodes || nnz >= kWideDegree * num_nodes) &&
         (nnz < kDenseEdges || nnz < kDenseDegree * num_nodes) && n >= table_walkers(num_nodes, 16) &&
         steps_pay(num_nodes, n, length);
}
// The same for a metapath; num_nodes: of all relations given together, each of which is packed (the graph gives those
// that the path takes: 1 M walkers, ten steps over a relation of 30 k nodes beside one of 4 M 57 -> 53 us, 131 k walkers,
// 120 steps 85 -> 64; few of them: a record's thread goes through them in turn).  Offsets as they are / table, us, three relations:
//                            200 k x 10   200 k x 20   200 k x 30   400 k x 20   1 M x 4   1 M x 10   1 M x 30
//   44 k nodes, 1 M edges      25/27        46/47        67/66        83/81       39/39      96/91     271/253
//   100 k, 2 M                 29/31        55/54        76/74        96/91       49/46     118/107    321/292
//   300 k, 5 M, 64-bit ids     36/38        69/68        96/92       127/119      72/66     164/147    440/395
//   1 M, 10 M                  30/34        52/55        73/72        99/94       63/60     134/122    338/305
//   2 M, 20 M                  32/40        55/62        77/84       109/109      68/70     145/139    363/326
//   2 M, 50 M, 64-bit ids      43/52        83/91       116/119      146/150      85/91     181/183    496/465
//   4 M, 100 M                 42/63        80/98       110/128      143/157      83/101    179/192    471/466
// A walker for every 32 nodes, the steps from where the line lies, and twice as many:
//                            131 k             200 k             300 k             500 k             1 M
//   2.1 M, 25 M              116/135, 205/233  144/146, 222/219  142/143, 235/226  161/157, 282/262  174/168, 313/292
//   2.1 M, 52 M              166/183, 277/320  200/192, 351/319  190/188, 343/312  205/194, 377/345  217/200, 408/361
//   4.2 M, 50 M              205/260, 360/434  222/235, 349/380  231/235, 359/356  274/263, 448/418  294/288, 522/486
//   4.2 M, 105 M             249/308, 427/535  309/317, 493/506  302/317, 510/517  326/337, 586/561  347/343, 632/606
//   8.4 M, 67 M              314/405, 543/654  282/352, 459/555  268/317, 432/492  320/358, 449/506  390/426, 606/644
//   8.4 M, 134 M             372/492, 653/807  381/443, 617/708  398/439, 592/650  475/486, 731/734  533/545, 914/900
// (from 400 MB a relation on, as streams).  No more nodes were measured.
constexpr int64_t kMostRelationNodes = int64_t(1) << 25;
bool packed_relations_pay(int64_t num_relations, int64_t num_nodes, int64_t n, int64_t length) {
  return num_relations > 0 && num_relations <= 16 && num_nodes >= (int64_t(1) << 18) &&
         num_nodes <= kMostRelationNodes && n >= table_walkers(num_nodes, 32) && steps_pay(num_nodes, n, length);
}
size_t tables_bytes(int64_t num_relations, int64_t num_nodes) {
  return padded(static_cast<size_t>(num_relations) * 8) +
         padded(static_cast<size_t>(num_nodes / kRecordNodes + num_relations + 1) * sizeof(uint4));
}
size_t table_bytes(int64_t num_nodes) {
  return padded(static_cast<size_t>((num_nodes + kRecordNodes - 1) / kRecordNodes) * sizeof(uint4));
}

__device__ __forceinline__ void pack_record(const int64_t* __restrict__ indptr, int64_t num_nodes, int64_t r,
                                            uint4* __restrict__ to) {
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
  *to = fits ? make_uint4(static_cast<uint32_t>(at[0]), end[1] << 16 | end[0],
                          end[3] << 16 | end[2], end[5] << 16 | end[4])
             : make_uint4(0u, 1u, 0u, 0u);
}

__global__ void __launch_bounds__(kThreads)
pack_offsets_kernel(const int64_t* __restrict__ indptr, int64_t num_nodes, int64_t records,
                    uint4* __restrict__ table) {
  const int64_t r = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
  if (r < records) pack_record(indptr, num_nodes, r, table + r);
}

// What a step reads of its node's offsets, and what it makes of it.
template <bool PACKED>
struct Offsets {
  int64_t start, end;
  template <typename Indptr>
  __device__ __forceinline__ void read(Indptr indptr, const uint4* __restrict__, int64_t v) {
    start = indptr[v];
    end = indptr[v + 1];
  }
  template <typename Indptr>
  __device__ __forceinline__ int64_t degree(Indptr, int64_t, int64_t* first) const {
    *first = start;
    return end - start;
  }
};
template <>
struct Offsets<true> {
  uint4 r;
  template <typename Indptr>
  __device__ __forceinline__ void read(Indptr, const uint4* __restrict__ table, int64_t v) {
    r = table[static_cast<uint32_t>(v) / kRecordNodes];
  }
  template <typename Indptr>
  __device__ __forceinline__ int64_t degree(Indptr indptr, int64_t v, int64_t* first) const {
    if ((r.y & 0xFFFFu) > r.w >> 16) {
      *first = indptr[v];
      return indptr[v + 1] - *first;
    }
    const uint32_t j = static_cast<uint32_t>(v) % kRecordNodes, half = j >> 1;
    const uint32_t here = half == 0 ? r.y : half == 1 ? r.z : r.w;
    const uint32_t left = half == 0 ? 0u : half == 1 ? r.y : r.z;
    const uint32_t begin = j & 1 ? here & 0xFFFFu : left >> 16;
    const uint32_t end = j & 1 ? here >> 16 : here & 0xFFFFu;
    *first = static_cast<int64_t>(r.x) + begin;
    return static_cast<int64_t>(end - begin);
  }
};

// The steps are ordered for the loads' sake: the node's offsets are asked for, then the node is stored and
// the draw made, while they come.  (Loads and stores are counted together and in order: with the store in
// front, the offsets waited for it.)  With the block of draws out of scratch memory, 4 M nodes and 200 M edges:
// 18 k walkers, 40 steps 60 -> 45 us, 66 k 70 -> 55, 300 k, 20 steps 120 -> 114, 1 M, 80 steps 1240 -> 1155
// (packed); 131 k nodes 1 M walkers 833 -> 704.
// PACKED: the offsets come from `table`, made for this call from indptr.  REPLAY: draws come from `replay`.
// A node outside [0, num_nodes) has no neighbours (the walker dies there), so a stray seed can never turn
// into a wild read.
template <typename IdT, bool PACKED, bool REPLAY>
__global__ void __launch_bounds__(kThreads)
random_walk_kernel(const int64_t* __restrict__ indptr, const uint4* __restrict__ table,
                   const IdT* __restrict__ indices,
                   int64_t num_nodes, const IdT* __restrict__ seeds, int64_t n, int64_t length, uint64_t seed,
                   const uint32_t* __restrict__ replay, IdT* __restrict__ trace) {
  const int64_t w = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
  if (w >= n) return;
  int64_t curr = static_cast<int64_t>(seeds[w]);
  const bool stream = !PACKED && n >= kStreamWalkers && num_nodes >= kStreamNodes &&
                      indptr[num_nodes] >= kStreamBytes / static_cast<int64_t>(sizeof(IdT));
  U4 x;
  for (int64_t t = 0; t < length; ++t) {
    const bool alive = static_cast<uint64_t>(curr) < static_cast<uint64_t>(num_nodes);
    Offsets<PACKED> off;
    if (alive) off.read(indptr, table, curr);
    trace[t * n + w] = static_cast<IdT>(curr);
    if (!REPLAY && (t & 3) == 0)
      x = draw_block(seed, kTagWalk, static_cast<uint64_t>(w), static_cast<uint64_t>(t >> 2));
    int64_t pick = -1;
    if (alive) {
      const uint32_t xv = REPLAY ? replay[t * n + w] : draw_of(x, t);
      int64_t start;
      const int64_t deg = off.degree(indptr, curr, &start);
      pick = neighbour(indices, start, deg, xv, stream);
    }
    curr = pick;
  }
  trace[length * n + w] = static_cast<IdT>(curr);
}

// The same for the relations of a metapath, one after the other: table_at[r] is where relation r's records
// begin, `capacity` where they have no room or its nodes no 32 bits.
__global__ void __launch_bounds__(kThreads)
pack_relations_kernel(const int64_t* const* __restrict__ all_indptr,
                      const int64_t* __restrict__ all_num_nodes, int64_t num_relations, int64_t capacity,
                      int64_t* __restrict__ table_at, uint4* __restrict__ table) {
  const int64_t r = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
  if (r == capacity) table[r] = make_uint4(0u, 1u, 0u, 0u);
  int64_t base = 0;
  for (int64_t rel = 0; rel < num_relations; ++rel) {
    const int64_t nodes = all_num_nodes[rel];
    const int64_t records = (nodes + kRecordNodes - 1) / kRecordNodes;
    const bool packed = nodes < (int64_t(1) << 32) && records <= capacity - base;
    if (r == 0) table_at[rel] = packed ? base : capacity;
    if (!packed) continue;
    if (r >= base && r - base < records) pack_record(all_indptr[rel], nodes, r - base, table + r);
    base += records;
  }
}

// (Said to be in global memory: a load through an address that was itself loaded is otherwise one that
// LDS might answer, and waits for everything in flight.)
template <typename T>
using GlobalPtr = const T __attribute__((address_space(1)))*;
template <typename IdT>
struct Relation {
  GlobalPtr<int64_t> indptr;
  GlobalPtr<IdT> indices;
  int64_t num_nodes;
  int64_t table_at;  // of its records
  bool packed;       // it has some
};

// LONG_WORK: large neighbour arrays are looked for and read as streams.  PACKED: the offsets come from a
// table, made for this call.  REPLAY: draws come from `replay`.
// A step's relation is looked up while the step before is under way, and its number a step earlier still.  With the
// order above, three relations of 2 M nodes and 50 M edges, 64-bit ids: 18 k walkers, 30 steps 38 -> 30 us, 200 k 119.6
// -> 114, 1 M 532 -> 512; packed 465.
template <typename IdT, bool LONG_WORK, bool PACKED, bool REPLAY>
__global__ void __launch_bounds__(kThreads)
metapath_walk_kernel(const int64_t* const* __restrict__ all_indptr,
                     const IdT* const* __restrict__ all_indices,
                     const int64_t* __restrict__ all_num_nodes, const int64_t* __restrict__ table_at,
                     const uint4* __restrict__ table, int64_t capacity,
                     const int64_t* __restrict__ metapath, int64_t length,
                     const IdT* __restrict__ seeds, int64_t n, uint64_t seed,
                     const uint32_t* __restrict__ replay, IdT* __restrict__ trace) {
  const int64_t w = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
  if (w >= n) return;
  int64_t curr = static_cast<int64_t>(seeds[w]);
  if (length == 0) {
    trace[w] = static_cast<IdT>(curr);
    return;
  }
  auto relation = [&](int64_t rel) {
    Relation<IdT> r{(GlobalPtr<int64_t>)all_indptr[rel], (GlobalPtr<IdT>)all_indices[rel],
                    all_num_nodes[rel], PACKED ? table_at[rel] : 0, true};
    if (PACKED) r.packed = r.table_at != capacity;
    return r;
  };
  U4 x;
  unsigned long long streams = 0ull;  // bit t: the relation of step t (mod 64) is read as a stream
  Relation<IdT> here = relation(metapath[0]);
  int64_t ahead = metapath[length > 1 ? 1 : 0];
  for (int64_t t = 0; t < length; ++t) {
    if (LONG_WORK && (t & (kWave - 1)) == 0) {  // a lane per step of the next 64
      const int64_t step = t + (threadIdx.x & (kWave - 1));
      const int64_t rel = metapath[step < length ? step : length - 1];
      const int64_t nodes = all_num_nodes[rel];
      const int64_t bytes = all_indptr[rel][nodes] * static_cast<int64_t>(sizeof(IdT));
      const bool one_of_two = bytes >= kStreamRelationBytes && nodes >= kStreamRelationNodes;
      const unsigned long long large = __ballot(one_of_two);
      const int64_t one = __shfl(rel, large ? __ffsll(static_cast<long long>(large)) - 1 : 0, kWave);
      const bool two = __ballot(one_of_two && rel != one) != 0ull;
      streams = two ? large : __ballot(n >= kStreamWalkers && bytes >= kStreamBytes && nodes >= kStreamNodes);
    }
    const bool alive = static_cast<uint64_t>(curr) < static_cast<uint64_t>(here.num_nodes);
    Offsets<PACKED> off;
    // (a relation without records: the one behind the last, which says to read the offsets)
    if (alive) off.read(here.indptr, table + (PACKED ? here.table_at : 0), !PACKED || here.packed ? curr : 0);
    const Relation<IdT> next = relation(ahead);
    ahead = metapath[t + 2 < length ? t + 2 : length - 1];
    trace[t * n + w] = static_cast<IdT>(curr);
    if (!REPLAY && (t & 3) == 0)
      x = draw_block(seed, kTagWalk, static_cast<uint64_t>(w), static_cast<uint64_t>(t >> 2));
    int64_t pick = -1;
    if (alive) {
      const uint32_t xv = REPLAY ? replay[t * n + w] : draw_of(x, t);
      int64_t start;
      const int64_t deg = off.degree(here.indptr, curr, &start);
      pick = neighbour(here.indices, start, deg, xv,
                       LONG_WORK && ((streams >> (t & (kWave - 1))) & 1ull));
    }
    curr = pick;
    here = next;
  }
  trace[length * n + w] = static_cast<IdT>(curr);
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
  if (workspace_bytes > 0 && num_nodes > 0 && !replay) {
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
  auto by_id = [&](auto id) {
    using IdT = decltype(id);
    if (replay)
      go(random_walk_kernel<IdT, false, true>, id);
    else
      go(table ? random_walk_kernel<IdT, true, false> : random_walk_kernel<IdT, false, false>, id);
  };
  if (id_bytes == 8)
    by_id(int64_t());
  else
    by_id(int32_t());
  return check_launch("random_walk");
}

int gs_random_walk(const int64_t* indptr, int64_t num_nodes, const void* indices, int id_bytes,
                   const void* seeds, int64_t n, int64_t length, uint64_t seed, const uint32_t* replay,
                   void* trace, void* stream) {
  return gs_random_walk_workspace(indptr, num_nodes, indices, id_bytes, seeds, n, length, seed, replay,
                                  trace, nullptr, 0, stream);
}

size_t gs_metapath_walk_workspace_bytes(int64_t num_relations, int64_t num_nodes, int64_t n, int64_t length) {
  return packed_relations_pay(num_relations, num_nodes, n, length)
             ? tables_bytes(num_relations, num_nodes) : 0;
}

int gs_metapath_walk_workspace(const int64_t* const* all_indptr, const void* const* all_indices,
                               const int64_t* all_num_nodes, int64_t num_relations, int64_t num_nodes,
                               int id_bytes, const int64_t* metapath, int64_t length, const void* seeds,
                               int64_t n, uint64_t seed, const uint32_t* replay, void* trace,
                               void* workspace, size_t workspace_bytes, void* stream) {
  GS_REQUIRE(n >= 0 && length >= 0 && num_relations >= 0 && num_nodes >= 0,
             "gs_metapath_walk: negative size");
  GS_REQUIRE(n == 0 || (seeds && trace), "gs_metapath_walk: null pointer");
  GS_REQUIRE(n == 0 || length == 0 || (all_indptr && all_indices && all_num_nodes && metapath),
             "gs_metapath_walk: null relation tables");
  GS_REQUIRE(valid_id_bytes(id_bytes), "gs_metapath_walk: id_bytes must be 4 or 8, got %d", id_bytes);
  if (n == 0) return GS_OK;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const dim3 grid(blocks_for(n, kThreads));
  const bool long_work = length > 0 && n >= (kStreamSteps + length - 1) / length;
  int64_t* table_at = nullptr;
  uint4* table = nullptr;
  const int64_t capacity = num_nodes / kRecordNodes + num_relations;
  if (workspace_bytes > 0 && length > 0 && num_relations > 0 && !replay) {
    Carver ws(workspace, workspace_bytes);
    table_at = ws.take<int64_t>(static_cast<size_t>(num_relations));
    table = ws.take<uint4>(static_cast<size_t>(capacity + 1));
    if (!ws.ok) {
      set_error_text("gs_metapath_walk: workspace needs %zu bytes, 256-byte aligned",
                     tables_bytes(num_relations, num_nodes));
      return GS_ERR_WORKSPACE;
    }
  }
  ProfileScope prof("metapath_walk", st);
  if (table)
    hipLaunchKernelGGL(pack_relations_kernel, dim3(blocks_for(capacity + 1, kThreads)), dim3(kThreads), 0, st,
                       all_indptr, all_num_nodes, num_relations, capacity, table_at, table);
  auto go = [&](auto kernel, auto id) {
    using IdT = decltype(id);
    hipLaunchKernelGGL(kernel, grid, dim3(kThreads), 0, st, all_indptr,
                       reinterpret_cast<const IdT* const*>(all_indices), all_num_nodes, table_at, table, capacity,
                       metapath, length, static_cast<const IdT*>(seeds), n, seed, replay,
                       static_cast<IdT*>(trace));
  };
  auto by_id = [&](auto id) {
    using IdT = decltype(id);
    if (replay)
      go(metapath_walk_kernel<IdT, false, false, true>, id);
    else if (table)
      go(metapath_walk_kernel<IdT, false, true, false>, id);
    else
      go(long_work ? metapath_walk_kernel<IdT, true, false, false>
                   : metapath_walk_kernel<IdT, false, false, false>, id);
  };
  if (id_bytes == 8)
    by_id(int64_t());
  else
    by_id(int32_t());
  return check_launch("metapath_walk");
}

int gs_metapath_walk(const int64_t* const* all_indptr, const void* const* all_indices,
                     const int64_t* all_num_nodes, int id_bytes, const int64_t* metapath, int64_t length, const void* seeds,
                     int64_t n, uint64_t seed, const uint32_t* replay, void* trace,
                     void* stream) {
  return gs_metapath_walk_workspace(all_indptr, all_indices, all_num_nodes, 0, 0, id_bytes, metapath, length,
                                    seeds, n, seed, replay, trace, nullptr, 0, stream);
}

}  // extern "C"
