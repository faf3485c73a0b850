"""GPU parity: random walks and metapath walks through the C ABI vs the CPU oracle."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from graph_sampling_amd import capi
from tests.util import rmat_csc_np, to_dev, u32_draws

pytestmark = pytest.mark.gpu


def _tables(indptrs, indicess, dev, idt):
    d_ip = [to_dev(a, dev) for a in indptrs]
    d_ix = [to_dev(a, dev, idt) for a in indicess]
    ip_tab = torch.tensor([t.data_ptr() for t in d_ip], dtype=torch.int64, device=dev)
    ix_tab = torch.tensor([t.data_ptr() for t in d_ix], dtype=torch.int64, device=dev)
    nn_tab = torch.tensor([t.numel() - 1 for t in d_ip], dtype=torch.int64, device=dev)
    return d_ip, d_ix, ip_tab, ix_tab, nn_tab


def test_metapath_reference_unique_path(dev):
    # reference tests/test_hetero_random_walk.cc:29-71: every hop has exactly one choice
    indptr1, indices1 = np.array([0, 0, 1, 2, 3]), np.array([0, 1, 2])   # "follow"
    indptr2, indices2 = np.array([0, 1, 2, 3]), np.array([0, 1, 2])      # "view"
    keep = _tables([indptr1, indptr2], [indices1, indices2], dev, torch.int64)
    metapath = np.array([1, 0, 0], dtype=np.int64)  # view, follow, follow
    seeds = np.array([2, 1], dtype=np.int64)
    trace = capi.metapath_walk(keep[2], keep[3], keep[4], torch.int64, to_dev(metapath, dev), to_dev(seeds, dev),
                               seed=3)
    expected = np.array([2, 1, 2, 1, 1, 0, 0, -1], dtype=np.int64)  # step-major [4][2]
    assert np.array_equal(trace.cpu().numpy(), expected)
    assert np.array_equal(O.metapath_walk([indptr1, indptr2], [indices1, indices2], metapath, seeds,
                                          seed=3), expected)


def test_metapath_reference_multi_path_edges_exist(dev):
    # reference tests/test_hetero_random_walk.cc:74-120
    indptr1, indices1 = np.array([0, 0, 1, 2, 3]), np.array([0, 1, 2])
    indptr2, indices2 = np.array([0, 1, 3, 5]), np.array([0, 0, 1, 2, 3])
    graphs = {0: (indptr1, indices1), 1: (indptr2, indices2)}
    keep = _tables([indptr1, indptr2], [indices1, indices2], dev, torch.int64)
    metapath = np.array([1, 0, 0], dtype=np.int64)
    seeds = np.array([2, 2, 1, 1, 0], dtype=np.int64)
    trace = capi.metapath_walk(keep[2], keep[3], keep[4], torch.int64, to_dev(metapath, dev), to_dev(seeds, dev),
                               seed=11).cpu().numpy().reshape(4, 5)
    for w in range(5):
        for t in range(3):
            src, dst = trace[t, w], trace[t + 1, w]
            if dst == -1:
                continue
            ip, ix = graphs[int(metapath[t])]
            assert dst in ix[ip[src]:ip[src + 1]]
        dead = np.where(trace[:, w] == -1)[0]
        if dead.size:
            assert (trace[dead[0]:, w] == -1).all()  # -1 is absorbing
    want = O.metapath_walk([indptr1, indptr2], [indices1, indices2], metapath, seeds, seed=11)
    assert np.array_equal(trace.reshape(-1), want)


@pytest.mark.parametrize("idt", [torch.int64, torch.int32])
@pytest.mark.parametrize("length", [0, 1, 7, 80])
def test_random_walk_matches_oracle(dev, idt, length):
    indptr, indices = rmat_csc_np(1 << 12, 1 << 15, seed=9)  # avg degree 8, plenty of dead ends
    seeds = np.random.default_rng(length).integers(0, 1 << 12, size=5000).astype(np.int64)
    got = capi.random_walk(to_dev(indptr, dev), to_dev(indices, dev, idt), to_dev(seeds, dev, idt),
                           length, seed=21)
    want = O.random_walk(indptr, indices, seeds, length, seed=21)
    assert np.array_equal(got.cpu().numpy().astype(np.int64), want)
    if length:
        assert (want == -1).any()
    # layout: flat [L+1][n]; row 0 is the seeds
    assert np.array_equal(want[:seeds.size], seeds)


def test_random_walk_replay(dev):
    indptr, indices = rmat_csc_np(1 << 12, 1 << 16, seed=10)
    n, L = 3000, 12
    seeds = np.random.default_rng(0).integers(0, 1 << 12, size=n).astype(np.int64)
    replay = u32_draws(n * L, 5)
    got = capi.random_walk(to_dev(indptr, dev), to_dev(indices, dev), to_dev(seeds, dev), L,
                           replay=to_dev(replay, dev))
    want = O.random_walk(indptr, indices, seeds, L, replay=replay)
    assert np.array_equal(got.cpu().numpy(), want)
    # closed form for one live step: indices[indptr[c] + r % deg]
    c = seeds
    deg = indptr[c + 1] - indptr[c]
    step1 = np.where(deg > 0, indices[np.minimum(indptr[c] + replay[:n] % np.maximum(deg, 1), indices.size - 1)], -1)
    assert np.array_equal(want[n:2 * n], step1)


@pytest.mark.parametrize("idt", [torch.int64, torch.int32])
def test_metapath_walk_rmat(dev, idt):
    rels = [rmat_csc_np(1 << 11, 1 << 14, seed=s) for s in (1, 2, 3)]
    indptrs, indicess = [r[0] for r in rels], [r[1] for r in rels]
    keep = _tables(indptrs, indicess, dev, idt)
    metapath = np.array([0, 1, 2, 1] * 4, dtype=np.int64)
    seeds = np.random.default_rng(3).integers(0, 1 << 11, size=4096).astype(np.int64)
    got = capi.metapath_walk(keep[2], keep[3], keep[4], idt, to_dev(metapath, dev), to_dev(seeds, dev, idt), seed=8)
    want = O.metapath_walk(indptrs, indicess, metapath, seeds, seed=8)
    assert np.array_equal(got.cpu().numpy().astype(np.int64), want)


def test_walk_next_hop_chi_square(dev):
    """Next hop of a degree-d node is uniform over its d neighbours."""
    d, n = 16, 64000
    indptr = np.array([0, d] + [d] * d, dtype=np.int64)  # node 0 has d neighbours 1..d, others none
    indices = np.arange(1, d + 1, dtype=np.int64)
    seeds = np.zeros(n, dtype=np.int64)
    got = capi.random_walk(to_dev(indptr, dev), to_dev(indices, dev), to_dev(seeds, dev), 1, seed=77)
    hop = got.cpu().numpy()[n:]
    counts = np.bincount(hop, minlength=d + 1)[1:].astype(np.float64)
    chi2 = ((counts - n / d) ** 2 / (n / d)).sum()
    assert chi2 < (d - 1) + 5 * np.sqrt(2 * (d - 1)), chi2


def test_walk_out_of_range_seeds_die(dev):
    indptr, indices = rmat_csc_np(1 << 10, 1 << 14, seed=13)
    seeds = np.array([5, -1, 1 << 10, 7, (1 << 10) + 999, -7], dtype=np.int64)
    got = capi.random_walk(to_dev(indptr, dev), to_dev(indices, dev), to_dev(seeds, dev), 4, seed=1)
    want = O.random_walk(indptr, indices, seeds, 4, seed=1)
    assert np.array_equal(got.cpu().numpy(), want)
    tr = want.reshape(5, 6)
    assert (tr[1:, [1, 2, 4, 5]] == -1).all()


@pytest.mark.parametrize("idt", [torch.int32, torch.int64])
@pytest.mark.parametrize("less", [0, 1])
def test_few_walkers_over_large_neighbour_arrays(dev, idt, less):
    """Neighbour arrays of 256 MB and of one edge less, alone and as one relation beside a small one,
    over more than 64 steps; each node has 64 neighbours, the last fewer.  (Too few walkers for streams.)"""
    E = (1 << 28) // (4 if idt == torch.int32 else 8) - less
    N = (E + 63) // 64
    rng = np.random.default_rng(less)
    indptr = np.minimum(np.arange(N + 1, dtype=np.int64) * 64, E)
    indices = rng.integers(0, N, E).astype(np.int32 if idt == torch.int32 else np.int64)
    small_ptr = np.arange(N + 1, dtype=np.int64)
    small_ix = rng.permutation(N)
    seeds = rng.integers(0, N, 300)
    big = indices.astype(np.int64)
    keep = _tables([indptr, small_ptr], [indices, small_ix], dev, idt)
    got = capi.random_walk(keep[0][0], keep[1][0], to_dev(seeds, dev, idt), 9, seed=5)
    assert np.array_equal(got.cpu().numpy().astype(np.int64), O.random_walk(indptr, big, seeds, 9, seed=5))
    path = np.array([0, 0, 1] * 22 + [0], dtype=np.int64)
    got = capi.metapath_walk(keep[2], keep[3], keep[4], idt, to_dev(path, dev), to_dev(seeds, dev, idt),
                             seed=6)
    want = O.metapath_walk([indptr, small_ptr], [big, small_ix], path, seeds, seed=6)
    assert np.array_equal(got.cpu().numpy().astype(np.int64), want)


def _even_offsets(nodes, edges):
    return np.arange(nodes + 1, dtype=np.int64) * edges // nodes


@pytest.mark.parametrize("idt", [torch.int32, torch.int64])
@pytest.mark.parametrize("less_edges,less_walkers,less_nodes", [(0, 0, 0), (1, 0, 0), (0, 1, 0), (0, 0, 1)])
def test_long_metapath_work_over_one_large_relation(dev, idt, less_edges, less_walkers, less_nodes):
    """A path's only large relation is read as a stream from 320 MB of neighbours, 2^21 nodes and
    120 000 walkers on; a small relation beside it is not."""
    E = (5 << 26) // (4 if idt == torch.int32 else 8) - less_edges
    N, n = (1 << 21) - less_nodes, 120_000 - less_walkers
    gen = torch.Generator(device=dev)
    gen.manual_seed(1)
    indices = torch.randint(0, N, (E,), generator=gen, device=dev, dtype=idt)
    rng = np.random.default_rng(1)
    small_ix = rng.permutation(N)
    indptr, small_ptr = _even_offsets(N, E), np.arange(N + 1, dtype=np.int64)
    keep = _tables([indptr, small_ptr], [np.zeros(1, np.int64), small_ix], dev, idt)
    keep[3][0] = indices.data_ptr()
    seeds, path = rng.integers(0, N, n), np.array([0, 0, 1] * 9, dtype=np.int64)  # 3.24 M steps: long work
    got = capi.metapath_walk(keep[2], keep[3], keep[4], idt, to_dev(path, dev), to_dev(seeds, dev, idt), seed=6)
    want = O.metapath_walk([indptr, small_ptr], [indices.cpu().numpy().astype(np.int64), small_ix], path, seeds,
                           seed=6)
    assert np.array_equal(got.cpu().numpy().astype(np.int64), want)


# 67 steps of each: 3 * 2**20 in all, less 11 and more 56
@pytest.mark.parametrize("walkers,relations,less_edges,less_nodes",
                         [(46_951, 2, 0, 0), (46_952, 2, 0, 0), (46_952, 1, 0, 0), (46_952, 2, 1, 0),
                          (46_952, 2, 0, 1)])
def test_long_metapath_work_over_streams(dev, walkers, relations, less_edges, less_nodes):
    """From 3 * 2**20 steps in all, the neighbour arrays of a metapath's relations are read as streams
    when two of them have 256 MB and 2^20 nodes."""
    E, N = (1 << 28) // 4 - less_edges, (1 << 20) - less_nodes
    rng = np.random.default_rng(walkers)
    ptr, small_ptr = _even_offsets(N, E), np.arange(N + 1, dtype=np.int64)
    indices = [rng.integers(0, N, E).astype(np.int32) for _ in range(relations)]
    small_ix = rng.permutation(N).astype(np.int32)
    seeds = rng.integers(0, N, walkers)
    ptrs = [ptr] * relations + [small_ptr]
    keep = _tables(ptrs, indices + [small_ix], dev, torch.int32)
    path = np.array([0, relations - 1, relations] * 22 + [0], dtype=np.int64)
    got = capi.metapath_walk(keep[2], keep[3], keep[4], torch.int32, to_dev(path, dev),
                             to_dev(seeds, dev, torch.int32), seed=6)
    want = O.metapath_walk(ptrs, [i.astype(np.int64) for i in indices + [small_ix]], path, seeds, seed=6)
    assert np.array_equal(got.cpu().numpy().astype(np.int64), want)


@pytest.mark.parametrize("idt", [torch.int32, torch.int64])
@pytest.mark.parametrize("nodes,hub", [(1, 3), (5, 65535), (6, 65535), (7, 65536), (601, 65530), (4096, 70000)])
def test_random_walk_with_packed_offsets(dev, idt, nodes, hub):
    """Records of six nodes: the last one part empty, ends up to 16 bits behind the start and beyond."""
    rng = np.random.default_rng(nodes)
    degree = rng.integers(0, 9, nodes)
    degree[min(nodes - 1, 3)] = hub
    indptr = np.concatenate([[0], np.cumsum(degree)]).astype(np.int64)
    indices = rng.integers(0, nodes, indptr[-1])
    seeds = np.concatenate([rng.integers(0, nodes, 700), [-1, nodes, nodes + 5]])
    got = capi.random_walk(to_dev(indptr, dev), to_dev(indices, dev, idt), to_dev(seeds, dev, idt), 13, seed=5,
                           packed=True)
    want = O.random_walk(indptr, indices, seeds, 13, seed=5)
    assert np.array_equal(got.cpu().numpy().astype(np.int64), want)


@pytest.mark.parametrize("less", [0, 1])
def test_random_walk_at_the_line_of_packed_offsets(dev, less):
    """2^18 walkers over 2^18 nodes for ten steps make a table, over one node less they make none."""
    nodes, n, length = (1 << 18) - less, 1 << 18, 10
    size = capi.lib().gs_random_walk_workspace_bytes
    import ctypes
    assert (size(*(ctypes.c_int64(v) for v in (nodes, 3 * nodes, n, length))) > 0) == (less == 0)
    rng = np.random.default_rng(less)
    degree = rng.integers(1, 6, nodes)
    indptr = np.concatenate([[0], np.cumsum(degree)]).astype(np.int64)
    indices = rng.integers(0, nodes, indptr[-1])
    seeds = rng.integers(0, nodes, n)
    got = capi.random_walk(to_dev(indptr, dev), to_dev(indices, dev, torch.int32),
                           to_dev(seeds, dev, torch.int32), length, seed=9)
    want = O.random_walk(indptr, indices, seeds, length, seed=9)
    assert np.array_equal(got.cpu().numpy().astype(np.int64), want)


@pytest.mark.parametrize("idt", [torch.int32, torch.int64])
@pytest.mark.parametrize("less_edges,less_walkers,less_nodes", [(0, 0, 0), (1, 0, 0), (0, 1, 0), (0, 0, 1)])
def test_random_walk_at_the_lines_of_streams(dev, idt, less_edges, less_walkers, less_nodes):
    """320 MB of neighbours, 2^21 nodes and 120 000 walkers are read as streams, one of any less is not."""
    E = (5 << 26) // (4 if idt == torch.int32 else 8) - less_edges
    N, n = (1 << 21) - less_nodes, 120_000 - less_walkers
    gen = torch.Generator(device=dev)
    gen.manual_seed(1)
    indices = torch.randint(0, N, (E,), generator=gen, device=dev, dtype=idt)
    indptr = _even_offsets(N, E)
    seeds = np.random.default_rng(1).integers(0, N, n)
    got = capi.random_walk(to_dev(indptr, dev), indices, to_dev(seeds, dev, idt), 6, seed=4, packed=False)
    want = O.random_walk(indptr, indices.cpu().numpy().astype(np.int64), seeds, 6, seed=4)
    assert np.array_equal(got.cpu().numpy().astype(np.int64), want)


@pytest.mark.parametrize("idt", [torch.int32, torch.int64])
@pytest.mark.parametrize("path", [[0], [2, 1], [0, 1, 2, 1, 0]])
@pytest.mark.parametrize("room", ["all", "two", "none"])
def test_metapath_walk_with_packed_offsets(dev, idt, path, room):
    """Records of three relations one behind the other, a hub in each; where they have no room the offsets
    are read.  Relations of different sizes: walkers that leave one die."""
    rng = np.random.default_rng(len(path))
    sizes, hubs = [601, 7, 3000], [65536, 65535, 70000]
    indptrs, indicess = [], []
    for nodes, hub in zip(sizes, hubs):
        degree = rng.integers(0, 9, nodes)
        degree[3] = hub
        indptrs.append(np.concatenate([[0], np.cumsum(degree)]).astype(np.int64))
        indicess.append(rng.integers(0, rng.choice([7, 700]), indptrs[-1][-1]))
    keep = _tables(indptrs, indicess, dev, idt)
    seeds = np.concatenate([rng.integers(0, 3001, 700), [-1, 3, 3, 3]])
    num_nodes = {"all": sum(sizes), "two": sizes[0] + sizes[1], "none": 0}[room]
    got = capi.metapath_walk(keep[2], keep[3], keep[4], idt, to_dev(np.array(path), dev), to_dev(seeds, dev, idt),
                             seed=8, num_nodes=num_nodes, packed=True)
    want = O.metapath_walk(indptrs, indicess, np.array(path), seeds, seed=8)
    assert np.array_equal(got.cpu().numpy().astype(np.int64), want)


def test_metapath_walk_replay(dev):
    rels = [rmat_csc_np(1 << 11, 1 << 14, seed=s) for s in (1, 2)]
    indptrs, indicess = [r[0] for r in rels], [r[1] for r in rels]
    keep = _tables(indptrs, indicess, dev, torch.int64)
    path, n = np.array([0, 1, 1, 0, 1, 0, 0]), 1000
    seeds = np.random.default_rng(0).integers(0, 1 << 11, size=n).astype(np.int64)
    replay = u32_draws(n * path.size, 5)
    got = capi.metapath_walk(keep[2], keep[3], keep[4], torch.int64, to_dev(path, dev), to_dev(seeds, dev),
                             replay=to_dev(replay, dev))
    want = O.metapath_walk(indptrs, indicess, path, seeds, replay=replay)
    assert np.array_equal(got.cpu().numpy(), want)


@pytest.mark.parametrize("less", [0, 1])
def test_metapath_walk_at_the_line_of_packed_offsets(dev, less):
    """Two relations of 2^17 nodes, 2^17 walkers and twenty steps make tables, a walker less makes none."""
    import ctypes
    nodes, n, length = 1 << 17, (1 << 17) - less, 20
    size = capi.lib().gs_metapath_walk_workspace_bytes
    assert (size(*(ctypes.c_int64(v) for v in (2, 2 * nodes, n, length))) > 0) == (less == 0)
    rng = np.random.default_rng(less)
    indptrs, indicess = [], []
    for _ in range(2):
        degree = rng.integers(1, 6, nodes)
        indptrs.append(np.concatenate([[0], np.cumsum(degree)]).astype(np.int64))
        indicess.append(rng.integers(0, nodes, indptrs[-1][-1]))
    keep = _tables(indptrs, indicess, dev, torch.int32)
    path, seeds = np.array([0, 1] * 10), rng.integers(0, nodes, n)
    got = capi.metapath_walk(keep[2], keep[3], keep[4], torch.int32, to_dev(path, dev),
                             to_dev(seeds, dev, torch.int32), seed=9, num_nodes=2 * nodes)
    want = O.metapath_walk(indptrs, indicess, path, seeds, seed=9)
    assert np.array_equal(got.cpu().numpy().astype(np.int64), want)
