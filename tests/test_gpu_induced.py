"""Induced subgraphs of a node set that fits a compute unit's LDS, against the oracle: set sizes
around the limits, duplicate nodes, tiles with one column and with thousands, edge data."""
import numpy as np
import pytest
import torch

import graph_sampling_amd as gs
from oracle import oracle as O
from graph_sampling_amd import capi
from util import to_dev

pytestmark = pytest.mark.gpu


def _graph(n, hubs, hub_degree, small, seed, wide=False):
    """n columns: `hubs` of them hub_degree edges long, the others 0 .. small edges."""
    rng = np.random.default_rng(seed)
    degree = rng.integers(0, small + 1, n)
    degree[rng.permutation(n)[:hubs]] = hub_degree
    indptr = np.concatenate([[0], np.cumsum(degree)]).astype(np.int64)
    indices = rng.integers(0, n, indptr[-1]).astype(np.int64)
    if wide:  # ids that agree in their low 32 bits
        indices[::3] += 1 << 40
    return indptr, indices, rng


@pytest.mark.parametrize("idt", [torch.int32, torch.int64])
@pytest.mark.parametrize("n_ids", [1, 300, 8192, 8193, 16383, 16384])
@pytest.mark.parametrize("weights", [False, True])
def test_set_sizes(dev, n_ids, weights, idt):
    indptr, indices, rng = _graph(30_000, 40, 90_001, 60, n_ids)
    wide = idt == torch.int64 and n_ids == 300
    if wide:
        indptr, indices, rng = _graph(30_000, 40, 90_001, 60, n_ids, wide=True)
    cols = rng.integers(0, 30_000, 20_000).astype(np.int64)
    rows = rng.integers(0, 30_000, n_ids).astype(np.int64)      # (some ids twice)
    if wide:
        rows[::2] += 1 << 40
    g = gs.Graph(False)
    g._CAPI_LoadCSC(to_dev(indptr, dev), to_dev(indices, dev, idt))
    if weights:
        w = rng.random(indices.size).astype(np.float32)
        g._CAPI_SetData(to_dev(w, dev))
    sub = g._CAPI_FusionSlicing(to_dev(cols, dev, idt), to_dev(rows, dev, idt))
    ptr, idx, _ = sub._CAPI_GetCSC()
    want = O.col_row_slice(indptr, indices, cols, rows)
    assert idx.dtype == idt
    assert np.array_equal(ptr.cpu().numpy(), want[0])
    assert np.array_equal(idx.cpu().numpy(), want[1])
    if weights:
        assert np.array_equal(sub._CAPI_GetData("default").cpu().numpy(), w[want[3]])


@pytest.mark.parametrize("hubs,hub_degree,small,n", [(1, 1_100_000, 0, 5000),      # empty columns between
                                                     (130, 8192, 0, 60_000),      # thousands of them a tile
                                                     (3, 400_000, 20, 4000),
                                                     (64, 16_385, 0, 64),
                                                     (8, 200_000, 9, 500_000),    # larger bitmaps:
                                                     (40, 90_000, 1, 2_000_000)])  # one a unit, none
def test_columns_per_tile(dev, hubs, hub_degree, small, n):
    indptr, indices, rng = _graph(n, hubs, hub_degree, small, n)
    hub = np.flatnonzero(np.diff(indptr) == hub_degree)
    cols = np.concatenate([hub, rng.permutation(n)])[:100_000].astype(np.int64)
    rows = rng.permutation(n)[: min(n // 2, 9000)].astype(np.int64)
    at = cols.size // 3
    cols[at] = n + 7                                             # no such column: empty
    g = gs.Graph(False)
    g._CAPI_LoadCSC(to_dev(indptr, dev), to_dev(indices, dev))
    ptr, idx, _ = g._CAPI_FusionSlicing(to_dev(cols, dev), to_dev(rows, dev))._CAPI_GetCSC()
    cols = np.delete(cols, at)
    want = O.col_row_slice(indptr, indices, cols, rows)
    assert np.array_equal(np.delete(ptr.cpu().numpy(), at), want[0])
    assert np.array_equal(idx.cpu().numpy(), want[1])


@pytest.mark.parametrize("coo", [False, True])        # (from an edge list: data by edge id)
@pytest.mark.parametrize("hub_degree", [20, 90_001])  # the general slice, and the set in LDS
def test_data_that_is_followed(dev, hub_degree, coo):
    """Edge data that require a gradient, or carry a forward-mode tangent, keep it in the subgraph,
    whichever way the slice goes."""
    n = 3000
    indptr, indices, rng = _graph(n, 20, hub_degree, 30, 5)
    indices[:n] = rng.permutation(n)  # every node is there
    order = np.arange(indices.size)
    if coo:  # the edges in another order; inside a column they come as in the list
        shuffle = rng.permutation(indices.size)
        col, row = np.repeat(np.arange(n), np.diff(indptr))[shuffle], indices[shuffle]
        order = np.argsort(col, kind="stable")
        indices = row[order]
    cols, rows = rng.permutation(n).astype(np.int64), rng.permutation(n)[:900].astype(np.int64)
    at = torch.from_numpy(order[O.col_row_slice(indptr, indices, cols, rows)[3]]).to(dev)
    w = torch.rand(indices.size, device=dev)

    def cut(data):
        g = gs.Graph(False)
        if coo:
            g._CAPI_LoadCOO(to_dev(row, dev), to_dev(col, dev))
        else:
            g._CAPI_LoadCSC(to_dev(indptr, dev), to_dev(indices, dev))
        g._CAPI_SetData(data)
        return g._CAPI_FusionSlicing(to_dev(cols, dev), to_dev(rows, dev))._CAPI_GetData("default")

    r = torch.rand(at.numel(), device=dev)
    x = w.clone().requires_grad_(True)
    (cut(x) * r).sum().backward()
    assert torch.equal(x.grad, torch.zeros_like(w).index_put_((at,), r))
    with torch.no_grad():
        assert torch.equal(cut(x), w[at])
    t = torch.rand_like(w)
    with torch.autograd.forward_ad.dual_level():
        got = torch.autograd.forward_ad.unpack_dual(cut(torch.autograd.forward_ad.make_dual(w, t)))
        assert torch.equal(got.primal, w[at]) and torch.equal(got.tangent, t[at])


@pytest.mark.parametrize("coo", [False, True])
def test_data_of_the_first_edges_only(dev, coo):
    """Data that end before the edges do serve a subgraph whose kept edges all have theirs."""
    indptr = np.array([0, 1_200_000, 2_400_000], dtype=np.int64)
    indices = np.zeros(2_400_000, dtype=np.int64)
    indices[::3] = 1
    indices[2_000_000:] = 7  # no node of the subgraph
    g = gs.Graph(False)
    if coo:  # (with a map from its edges to the data)
        col = np.repeat(np.arange(8), np.diff(np.append(indptr, [indptr[-1]] * 6)))
        g._CAPI_LoadCOO(to_dev(indices, dev), to_dev(col, dev))
    else:
        g._CAPI_LoadCSC(to_dev(indptr, dev), to_dev(indices, dev))
    w = torch.rand(2_000_000, device=dev)
    g._CAPI_SetData(w)
    ids = torch.tensor([0, 1], device=dev)
    sub = g._CAPI_FusionSlicing(ids, ids)
    assert torch.equal(sub._CAPI_GetData("default"), w)
    assert np.array_equal(sub._CAPI_GetCSC()[1].cpu().numpy(), indices[:2_000_000])


@pytest.mark.parametrize("weights", [False, True])
def test_more_edges_than_32_bits_count(dev, weights):
    """Columns at the end of a neighbour array of more than 2**32 edges."""
    n, degree = 1 << 16, (1 << 16) + 1
    gen = torch.Generator(device=dev)
    gen.manual_seed(2)
    indices = torch.randint(0, n, (n * degree,), generator=gen, device=dev, dtype=torch.int32)
    g = gs.Graph(False)
    g._CAPI_LoadCSC(torch.arange(n + 1, device=dev) * degree, indices)
    if weights:
        w = torch.empty(n * degree, device=dev)
        w[-20 * degree:] = torch.rand(20 * degree, device=dev)
        g._CAPI_SetData(w)
    cols = torch.arange(n - 20, n, device=dev, dtype=torch.int32)
    rows = torch.randperm(n, generator=gen, device=dev)[:5000].to(torch.int32)
    sub = g._CAPI_FusionSlicing(cols, rows)
    place = torch.full((n,), -1, dtype=torch.int32, device=dev)
    place[rows.long()] = torch.arange(5000, dtype=torch.int32, device=dev)
    want = place[indices[-20 * degree:].long()]
    ptr, idx, _ = sub._CAPI_GetCSC()
    assert torch.equal(idx, want[want >= 0])
    assert torch.equal(ptr[1:], torch.cumsum((want >= 0).view(20, degree).sum(1), 0))
    if weights:
        assert torch.equal(sub._CAPI_GetData("default"), w[-20 * degree:][want >= 0])


@pytest.mark.parametrize("hubs,hub_degree,small,n,columns", [(130, 8192, 0, 60_000, 60_000),  # mostly empty
                                                             (8, 200_000, 9, 500_000, 100_000),
                                                             (40, 60_000, 20, 700_000, 37_000)])
@pytest.mark.parametrize("weights", [False, True])
def test_short_columns(dev, hubs, hub_degree, small, n, columns, weights):
    """Columns on both sides of 64 edges on average, with data and without (the general slice)."""
    indptr, indices, rng = _graph(n, hubs, hub_degree, small, n)
    hub = np.flatnonzero(np.diff(indptr) == hub_degree)
    cols = np.concatenate([hub, rng.permutation(n)])[:columns].astype(np.int64)
    rows = rng.permutation(n)[: min(n // 2, 9000)].astype(np.int64)
    g = gs.Graph(False)
    g._CAPI_LoadCSC(to_dev(indptr, dev), to_dev(indices, dev))
    w = rng.random(indices.size).astype(np.float32)
    if weights:
        g._CAPI_SetData(to_dev(w, dev))
    sub = g._CAPI_FusionSlicing(to_dev(cols, dev), to_dev(rows, dev))
    want = O.col_row_slice(indptr, indices, cols, rows)
    assert np.array_equal(sub._CAPI_GetCSC()[0].cpu().numpy(), want[0])
    assert np.array_equal(sub._CAPI_GetCSC()[1].cpu().numpy(), want[1])
    if weights:
        assert np.array_equal(sub._CAPI_GetData("default").cpu().numpy(), w[want[3]])


@pytest.mark.parametrize("n", [31, 32, 2016, 2047, 2048, 70_001])
@pytest.mark.parametrize("map", [False, True])
def test_bitmap_rows_and_data_from_the_parent(dev, n, map):
    """Bounds at the ends of the bitmap's words and of its rows of 64 words, every id at the bound's edge; data found
    word by word in words of one column, of several and of more columns than are staged, by position and by a
    map."""
    rng = np.random.default_rng(n)
    degree = np.concatenate([[700_001, 0, 511, 1, 64, 63, 65], np.zeros(130, int), [448_000, 3, 2, 1, 1]])
    degree = np.resize(degree, n) if n < degree.size else np.concatenate([degree, np.ones(n - degree.size, int)])
    degree[0] += max(0, (1 << 20) - degree.sum())
    indptr = np.concatenate([[0], np.cumsum(degree)]).astype(np.int64)
    E = int(indptr[-1])
    indices = rng.integers(0, n, E).astype(np.int64)
    rows = np.concatenate([[n - 1, 0], rng.permutation(n)[: min(n, 3000)]]).astype(np.int64)  # (two ids twice)
    order = np.arange(E)
    g = gs.Graph(False)
    if map:
        shuffle = rng.permutation(E)
        col, row = np.repeat(np.arange(n), degree)[shuffle], indices[shuffle]
        order = np.argsort(col, kind="stable")
        indices = row[order]
        g._CAPI_LoadCOO(to_dev(row, dev), to_dev(col, dev))
    else:
        g._CAPI_LoadCSC(to_dev(indptr, dev), to_dev(indices, dev))
    w = rng.random(E).astype(np.float32)
    g._CAPI_SetData(to_dev(w, dev))
    cols = np.arange(n).astype(np.int64)
    sub = g._CAPI_FusionSlicing(to_dev(cols, dev), to_dev(rows, dev))
    want = O.col_row_slice(indptr, indices, cols, rows)
    assert np.array_equal(sub._CAPI_GetCSC()[0].cpu().numpy(), want[0])
    assert np.array_equal(sub._CAPI_GetCSC()[1].cpu().numpy(), want[1])
    assert np.array_equal(sub._CAPI_GetData("default").cpu().numpy(), w[order][want[3]])


# more bytes of ids and data than are read through the caches; both forms of the set
@pytest.mark.parametrize("idt", [torch.int32, torch.int64])
@pytest.mark.parametrize("n", [60_000, 2_000_000])
@pytest.mark.parametrize("data", ["none", "by position", "by edge id"])
def test_streamed_positions(dev, data, n, idt):
    S, degree = 20, 3_400_001
    gen = torch.Generator(device=dev)
    gen.manual_seed(n)
    row = torch.randint(0, n, (S * degree,), generator=gen, device=dev, dtype=idt)
    w = torch.rand(S * degree, generator=gen, device=dev)
    g = gs.Graph(False)
    if data == "by edge id":  # the columns from the last to the first
        col = torch.arange(S - 1, -1, -1, device=dev, dtype=idt).repeat_interleave(degree)
        g._CAPI_LoadCOO(row, col)
        row, order = row.view(S, degree).flip(0).reshape(-1), w.view(S, degree).flip(0).reshape(-1)
    else:
        ptr = torch.full((n + 1,), S * degree, device=dev)
        ptr[:S + 1] = torch.arange(S + 1, device=dev) * degree
        g._CAPI_LoadCSC(ptr, row)
        order = w
    if data != "none":
        g._CAPI_SetData(w)
    cols = torch.arange(S, device=dev, dtype=idt)
    rows = torch.randperm(n, generator=gen, device=dev)[:7001].to(idt)
    sub = g._CAPI_FusionSlicing(cols, rows)
    place = torch.full((n,), -1, dtype=idt, device=dev)
    place[rows.long()] = torch.arange(7001, dtype=idt, device=dev)
    want = place[row.long()]
    ptr, idx, _ = sub._CAPI_GetCSC()
    assert torch.equal(idx, want[want >= 0])
    assert torch.equal(ptr[1:], torch.cumsum((want >= 0).view(S, degree).sum(1), 0))
    if data != "none":
        assert torch.equal(sub._CAPI_GetData("default"), order[want >= 0])


@pytest.mark.parametrize("idt", [torch.int32, torch.int64])
@pytest.mark.parametrize("data", ["none", "by position", "by map"])
@pytest.mark.parametrize("n", [60_000, 2_000_000])  # both forms of the set
def test_the_pair_whose_second_call_knows_no_data(dev, n, data, idt):
    """gs_induced_slice_mark and _compact as they were before the forms that keep the arrays: no mailbox, and the data are
    read by the first call; a row id at the bound on them is reported as a total of -1."""
    indptr, indices, rng = _graph(n, 30, 50_001, 40, n)
    cols, rows = rng.integers(0, n, 30_000).astype(np.int64), rng.integers(0, n, 5000).astype(np.int64)
    cols[::100] = np.flatnonzero(np.diff(indptr) == 50_001)[0]
    order = rng.permutation(indices.size)
    w = rng.random(indices.size).astype(np.float32)
    args = [to_dev(indptr, dev), to_dev(indices, dev, idt), to_dev(cols, dev, idt), to_dev(rows, dev, idt)]
    e_ids = to_dev(order, dev) if data == "by map" else None
    t_w = None if data == "none" else to_dev(w, dev)
    ptr, idx, got = capi.induced_slice(*args, n, t_w, e_ids)
    want = O.col_row_slice(indptr, indices, cols, rows)
    assert np.array_equal(ptr.cpu().numpy(), want[0]) and np.array_equal(idx.cpu().numpy(), want[1])
    if data != "none":
        assert np.array_equal(got.cpu().numpy(), (w[order] if data == "by map" else w)[want[3]])
    if n == 60_000:
        assert int(capi.induced_slice(*args, int(rows.max()), t_w, e_ids)[-1]) == -1


@pytest.mark.parametrize("data", ["by position", "by map"])
@pytest.mark.parametrize("idt", [torch.int32, torch.int64])
@pytest.mark.parametrize("lens", [[17], [40, 1, 0, 60, 0], [300, 20, 9, 700], [511, 1], [64, 64, 65, 63]])
def test_data_of_tiles_of_several_columns(dev, lens, idt, data):
    """Tiles whose words are all of several columns, and some of them; as many of their edges kept as a lane takes at once
    (64, 192) and one more and less, none and all; a column id that is none stands first."""
    rng = np.random.default_rng(len(lens))
    degree = np.resize(lens, (1_100_000 // sum(lens) + 1) * len(lens))
    cols = rng.permutation(degree.size)
    parent = np.zeros_like(degree)
    parent[cols] = degree
    indptr = np.concatenate([[0], np.cumsum(parent)]).astype(np.int64)
    D, n = int(indptr[-1]), 70_000
    kept = np.zeros((D + 511) // 512 * 512, bool)
    for t, k in zip(range(0, D, 512), np.resize([0, 1, 63, 64, 65, 191, 192, 193, 384, 385, 511, 512], D // 512 + 1)):
        kept[t + rng.permutation(512)[:k]] = True
    start = np.repeat(indptr[cols], degree)
    offset = np.concatenate([[0], np.cumsum(degree)])
    at = start + np.arange(D) - np.repeat(offset[:-1], degree)  # where the slice's positions are in the parent
    ids = np.where(kept[:D], rng.integers(0, 3000, D) * 2, rng.integers(0, 3000, D) * 2 + 1)
    indices = np.empty(D, np.int64)
    indices[at] = ids
    cols = np.concatenate([[-1], cols]).astype(np.int64)
    rows = rng.permutation(3000).astype(np.int64) * 2
    g = gs.Graph(False)
    w, order = rng.random(D).astype(np.float32), np.arange(D)
    if data == "by map":
        order = rng.permutation(D)
        ptr, idx, got = capi.induced_slice(to_dev(indptr, dev), to_dev(indices, dev, idt), to_dev(cols, dev, idt),
                                           to_dev(rows, dev, idt), n, to_dev(w, dev), to_dev(order, dev))
    else:
        g._CAPI_LoadCSC(to_dev(indptr, dev), to_dev(indices, dev, idt))
        g._CAPI_SetData(to_dev(w, dev))
        sub = g._CAPI_FusionSlicing(to_dev(cols, dev, idt), to_dev(rows, dev, idt))
        (ptr, idx, _), got = sub._CAPI_GetCSC(), sub._CAPI_GetData("default")
    want = O.col_row_slice(indptr, indices, cols, rows)
    assert np.array_equal(ptr.cpu().numpy(), want[0]) and np.array_equal(idx.cpu().numpy(), want[1])
    assert np.array_equal(got.cpu().numpy(), w[order][want[3]])


@pytest.mark.parametrize("n", [70_000, 2_000_000])  # both forms of the set
@pytest.mark.parametrize("data", ["by position", "by map"])
@pytest.mark.parametrize("idt", [torch.int32, torch.int64])
@pytest.mark.parametrize("more", [0, 1])
def test_data_on_both_sides_of_long_columns(dev, more, idt, data, n):
    """512 positions a column, where the copy reads the data from the parent, and one less, where the marks do: one
    column has most of them, between tiles whose words are of several; few, some and all edges of a tile kept."""
    rng = np.random.default_rng(n + more)
    short = np.concatenate([np.resize(np.array(lens), 800) for lens in ([17], [40, 1, 0, 60, 0], [300, 20, 9, 90], [511, 1])])
    S = short.size + 1
    degree = np.concatenate([short[:S // 2], [0], short[S // 2:]])
    degree[S // 2] = 512 * S - short.sum() - more
    cols = rng.permutation(S)
    parent = np.zeros_like(degree)
    parent[cols] = degree
    indptr = np.concatenate([[0], np.cumsum(parent)]).astype(np.int64)
    D = int(indptr[-1])
    assert D == 512 * S - more and D >= 1 << 20
    kept = np.zeros((D + 511) // 512 * 512, bool)
    for t, k in zip(range(0, D, 512), np.resize([0, 1, 5, 63, 64, 65, 192, 193, 511, 512], D // 512 + 1)):
        kept[t + rng.permutation(512)[:k]] = True
    offset = np.concatenate([[0], np.cumsum(degree)])
    at = np.repeat(indptr[cols], degree) + np.arange(D) - np.repeat(offset[:-1], degree)
    indices = np.empty(D, np.int64)
    indices[at] = np.where(kept[:D], rng.integers(0, 3000, D) * 2, rng.integers(0, 3000, D) * 2 + 1)
    rows = rng.permutation(3000).astype(np.int64) * 2
    w = rng.random(D).astype(np.float32)
    order = rng.permutation(D) if data == "by map" else np.arange(D)
    want = O.col_row_slice(indptr, indices, cols, rows)
    args = [to_dev(indptr, dev), to_dev(indices, dev, idt), to_dev(cols, dev, idt), to_dev(rows, dev, idt), n,
            to_dev(w, dev), to_dev(order, dev) if data == "by map" else None]
    for stays in (False, True):
        ptr, idx, got = capi.induced_slice(*args, kept=stays)
        assert np.array_equal(ptr.cpu().numpy(), want[0]) and np.array_equal(idx.cpu().numpy(), want[1])
        assert np.array_equal(got.cpu().numpy(), w[order][want[3]])
