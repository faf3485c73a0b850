"""GPU parity: a small minibatch by one workgroup in one launch (gs_minibatch_sample, behind
Graph.SampleLayers) against the CPU oracle layer by layer, and against the layer-by-layer calls for
the samples' edge data."""
import ctypes

import numpy as np
import pytest
import torch

import graph_sampling_amd as gs
from graph_sampling_amd import capi
from oracle import oracle as O
from tests.util import rmat_csc_np, to_dev

pytestmark = pytest.mark.gpu


def _one_launch(num_seeds, fanouts):
    f = (ctypes.c_int64 * len(fanouts))(*fanouts)
    return bool(capi.lib().gs_minibatch_applies(ctypes.c_int64(num_seeds), len(fanouts), f))


def _check(dev, indptr, indices, seeds, fanouts, replace, idt, seed):
    assert _one_launch(seeds.size, fanouts)
    g = gs.Graph(False)
    g._CAPI_LoadCSC(to_dev(indptr, dev), to_dev(indices, dev, idt))
    gs.set_seed(seed)
    out = g._CAPI_SampleLayers(to_dev(seeds, dev, idt), list(fanouts), replace)
    cols = seeds
    for l, k in enumerate(fanouts):
        sp, _, si, _ = O.sample_uniform(indptr, indices, cols, k, replace, seed=seed + l, with_coo=False)
        frontier, (renamed,) = O.relabel([cols, si], [si])
        for got, want in zip(out[3 * l:3 * l + 3], (frontier, sp, renamed)):
            # (an id of all ones is -1 in either width)
            assert np.array_equal(got.cpu().numpy().astype(np.int64), want.astype(np.int64)), (l, k)
        cols = frontier


# sizes: one column a layer, columns that fill a round of 1024 lanes and go past it for every
# number of lanes a column (1, 2, 4, 8; behind a layer that takes nothing, as one layer alone goes
# the other way from 2048 items on), the limits on items, columns and layers, no seed at all
@pytest.mark.parametrize("idt", [torch.int32, torch.int64])
@pytest.mark.parametrize("num_seeds,fanouts,replace", [
    (1, (1,), False), (32, (10, 5), False), (32, (10, 5), True), (0, (4, 4), False), (7, (15, 10, 5), False),
    (1024, (0, 4), False), (1025, (0, 4), True), (512, (0, 8), False), (513, (0, 5), False), (256, (0, 16), False),
    (257, (0, 16), True), (128, (0, 32), False), (129, (0, 17), True), (2048, (0, 3), False),
    (31, (10, 5, 3), False), (1, (2, 2, 2, 2, 2, 2, 1, 1), False), (50, (0, 7), False), (300, (3, 0), True)])
def test_one_launch_equals_the_oracle(dev, idt, num_seeds, fanouts, replace):
    n = 1 << 13
    indptr, indices = rmat_csc_np(n, 1 << 17, seed=num_seeds % 5)
    rng = np.random.default_rng(num_seeds)
    _check(dev, indptr, indices, rng.permutation(n)[:num_seeds].astype(np.int64), fanouts, replace, idt, 40)
    if num_seeds > 16:  # repeats, and hubs with their neighbours
        seeds = rng.integers(0, n, num_seeds).astype(np.int64)
        seeds[:8] = np.argsort(np.diff(indptr))[-8:]
        seeds[8:16] = seeds[0]
        _check(dev, indptr, indices, seeds, fanouts, replace, idt, 50)


@pytest.mark.parametrize("case", range(16))
def test_one_launch_on_seeded_random_shapes(dev, case):
    rng = np.random.default_rng(4000 + case)
    n = int(rng.choice([64, 1 << 10, 1 << 15]))
    indptr, indices = rmat_csc_np(n, int(n * rng.choice([1, 4, 30])), seed=case)
    while True:
        num_seeds = int(2 ** (11 * rng.random()))
        fanouts = tuple(int(rng.integers(1, 33)) for _ in range(int(rng.integers(1, 4))))
        if _one_launch(num_seeds, fanouts):
            break
    replace = bool(rng.integers(0, 2)) and 1 not in fanouts
    idt = torch.int32 if case % 2 else torch.int64
    _check(dev, indptr, indices, rng.integers(0, n, num_seeds).astype(np.int64), fanouts, replace, idt, case)


def test_seeds_that_are_no_columns_and_sizes_beyond_the_limits(dev):
    n = 1 << 12
    indptr, indices = rmat_csc_np(n, 1 << 16, seed=5)
    seeds = np.array([5, 1 << 20, n, 17, n + 100, 900, 5], dtype=np.int64)
    for idt in (torch.int32, torch.int64):
        _check(dev, indptr, indices, seeds, (3, 3), False, idt, 2)
    assert not _one_launch(2049, (1,)) and not _one_launch(1, (33,)) and not _one_launch(1, (1,) * 9)
    assert not _one_launch(2048, (4,)) and not _one_launch(-1, (1,)) and not _one_launch(683, (2, 3))


@pytest.mark.parametrize("idt", [torch.int32, torch.int64])
@pytest.mark.parametrize("mapped", [False, True])
@pytest.mark.parametrize("replace", [False, True])
def test_edge_data_of_the_samples(dev, idt, mapped, replace):
    n = 1 << 11
    indptr, indices = rmat_csc_np(n, 1 << 15, seed=9)
    rng = np.random.default_rng(3)
    data = to_dev((1.0 - rng.random(indices.size)).astype(np.float32), dev)
    if mapped:  # loaded from an edge list in no order: the data go by an edge-id map
        col = np.repeat(np.arange(n), np.diff(indptr))
        order = rng.permutation(indices.size)
        A = gs.Matrix().load_coo(to_dev(indices[order], dev, idt), to_dev(col[order], dev, idt), data)
        A._graph._CAPI_GetCSC()
    else:
        A = gs.Matrix().load_csc(to_dev(indptr, dev), to_dev(indices, dev, idt), data)
    seeds = to_dev(rng.permutation(n)[:60].astype(np.int64), dev, idt)
    fanouts = [6, 20]
    gs.set_seed(11)
    got = A._graph._CAPI_SampleLayers(seeds, fanouts, replace)
    gs.set_seed(11)
    cols = seeds
    for l, k in enumerate(fanouts):
        sub = A._graph._CAPI_FusedColumnwiseSlicingSampling(cols, k, replace)
        cols, _, _, ptr, idx, _, _ = sub._CAPI_Relabel()
        for a, b in zip(got[4 * l:4 * l + 4], (cols, ptr, idx, sub._CAPI_GetData("default"))):
            assert torch.equal(a, b)


def test_an_id_beyond_32_bits_goes_layer_by_layer(dev):
    indptr = np.array([0, 2, 4, 6], dtype=np.int64)
    indices = np.array([1, 2, 0, (1 << 33) + 5, 0, 1], dtype=np.int64)
    seeds = np.array([0, 1, 2], dtype=np.int64)
    offsets = torch.empty(4, dtype=torch.int64, device=dev)
    out, frontier = (torch.empty(s, dtype=torch.int64, device=dev) for s in (6, 9))
    counts = torch.empty(2, dtype=torch.int64, device=dev)
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    one = lambda t: (ctypes.c_void_p * 1)(t.data_ptr())  # noqa: E731
    d = (to_dev(indptr, dev), to_dev(indices, dev), to_dev(seeds, dev))
    status = capi.lib().gs_minibatch_sample(
        ptr(d[0]), ctypes.c_int64(3), ptr(d[1]), ptr(d[2]), 8, ctypes.c_int64(3), 1,
        (ctypes.c_int64 * 1)(2), 0, (ctypes.c_uint64 * 1)(1), None, None, one(offsets), one(out),
        one(frontier), None, ptr(counts), None, None,
        ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert status == 0
    assert counts.tolist() == [6, -2]
