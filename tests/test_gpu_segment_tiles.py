"""Segment sums and normalisation by 4096-edge tiles against the oracle: segments around the
lengths a lane, sixteen lanes and a wave add up, on both sides of tile borders, with and
without an edge map, with runs of empty segments between."""
import ctypes

import numpy as np
import pytest
import torch

from graph_sampling_amd import capi
from util import to_dev

pytestmark = pytest.mark.gpu

# an addend passes through at most 43 roundings on its way into a sum (its square, 16 additions of
# a lane, 2 + 6 across the wave, 16 + 1 pieces in a row, the division): 43 * 2**-24
RTOL = 2.6e-6

LENGTHS = {
    "lane": [0, 1, 3, 16],
    "group": [17, 18, 63, 128],
    "wave": [129, 200, 1000],
    "border": [4079, 16, 4097, 17, 4095, 1, 15, 8192, 0, 5],
    "hub": [70_001, 2, 300_000, 16, 40],
    "gaps": [0] * 700 + [20] * 60 + [0] * 300 + [5000, 16, 16],
    "mixed": [0, 1, 2, 5, 9, 16, 17, 40, 129, 500, 3000],
    "sparse": [0, 0, 0, 1, 2, 0],
    "low": [0, 2, 7, 30],
}


def _segments(kind, total):
    rng = np.random.default_rng(len(kind))
    base = np.array(LENGTHS[kind])
    lens, n = [], 0
    while n < total:
        part = base if kind in ("border", "hub", "gaps") else rng.permutation(np.repeat(base, 40))
        lens.append(part)
        n += int(part.sum())
    lens = np.concatenate(lens)
    if kind == "gaps" and total == 150_000:  # far more segments than edges
        lens = np.concatenate([lens, np.zeros(400_000, dtype=lens.dtype), [1, 2, 30]])
    return np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)


@pytest.mark.parametrize("emap", [False, True])
@pytest.mark.parametrize("kind", sorted(LENGTHS))
@pytest.mark.parametrize("total", [1, 4096, 150_000, 2_300_000])
def test_sum_and_normalise(dev, kind, total, emap):
    _check(dev, kind, total, emap)


@pytest.mark.parametrize("kind,total", [("sparse", 8_500_000),           # marks, the middle width
                                        ("low", 8_380_000),              # widest and middle on both
                                        ("low", 8_400_000),              # sides of 2048 tiles
                                        ("mixed", 25_160_000),           # middle and narrow on both
                                        ("mixed", 25_200_000)])          # sides of 6144
def test_widths_of_a_tiles_workgroup(dev, kind, total):
    _check(dev, kind, total, False)


@pytest.mark.parametrize("lens", [[3, 17, 5_000_000, 40, 300_000],            # added up tile by tile
                                  [3, 17, 130_000_000, 5_300_000, 40, 300_000]])  # totals made first
def test_segments_of_thousands_of_tiles(dev, lens):
    ptr = torch.tensor(np.concatenate([[0], np.cumsum(lens)]), device=dev)
    data = torch.rand(int(ptr[-1]), device=dev) + 0.25
    parts = torch.split(data.double(), lens)
    # the pieces of the longest by the lanes of a wave, so many in a row, where RTOL counts 17
    rtol = RTOL + max(lens) / 4096 / 64 * 2.0 ** -24
    out = torch.empty(len(lens), device=dev)
    capi.segment_sum(ptr, None, None, data, 1, out)
    total = torch.stack([p.sum() for p in parts])
    torch.testing.assert_close(out.double(), total, rtol=rtol, atol=0)
    out = torch.empty_like(data)
    capi.segment_normalize(ptr, None, data, out)
    for p, t, got in zip(parts, total, torch.split(out, lens)):
        torch.testing.assert_close(got.double(), p / t, rtol=rtol, atol=0)


# both sides of the 2**25 edges from which data and results are streamed; offsets that begin
# at an edge whose place is no multiple of four; more segments than edges (marks)
@pytest.mark.parametrize("kind", ["mixed", "border", "sparse"])
@pytest.mark.parametrize("nnz,front", [((1 << 25) - 1, 0), (1 << 25, 0), ((1 << 25) + 4099, 3)])
def test_streamed_edges(dev, kind, nnz, front):
    some = torch.from_numpy(np.diff(_segments(kind, 1_500_000))).to(dev)
    lens = some.repeat(nnz // int(some.sum()) + 1)
    ends = torch.cumsum(lens, 0).clamp_(max=nnz)
    ptr = torch.cat([ends.new_zeros(1), ends])
    data = torch.rand(front + nnz, device=dev) + 0.25
    owner = torch.repeat_interleave(torch.diff(ptr), output_size=nnz)
    w = data[front:].double()
    for power in (1, 2):
        want = torch.zeros(lens.numel(), dtype=torch.float64, device=dev).index_add_(0, owner, w ** power)
        out = torch.full((lens.numel(),), -1.0, device=dev)
        capi.segment_sum(ptr + front, None, None, data, power, out)
        torch.testing.assert_close(out.double(), want, rtol=RTOL, atol=0)
        if power == 1:
            out = torch.full_like(data, -1.0)
            capi.segment_normalize(ptr + front, None, data, out)
            torch.testing.assert_close(out[front:].double(), w / want[owner], rtol=RTOL, atol=0)
            assert (out[:front] == -1).all()


# 4 bytes an edge and 12 a segment: 2**28 in all, from which on a sum's data are streamed, and an edge less; beyond them
# the last segments are empty
@pytest.mark.parametrize("less", [0, 1])
@pytest.mark.parametrize("nseg", [1000, 5_000_000, (1 << 25) // 3])
def test_streamed_sums(dev, nseg, less):
    nnz = (1 << 26) - 3 * nseg - less
    ptr = (torch.arange(nseg + 1, device=dev) * nnz // (nseg - 7)).clamp_(max=nnz)
    data = torch.rand(nnz, device=dev) + 0.25
    owner = torch.repeat_interleave(torch.diff(ptr), output_size=nnz)
    for power in (1, 2):
        want = torch.zeros(nseg, dtype=torch.float64, device=dev).index_add_(0, owner, data.double() ** power)
        out = torch.full((nseg,), -1.0, device=dev)
        capi.segment_sum(ptr, None, None, data, power, out)
        torch.testing.assert_close(out.double(), want, rtol=RTOL, atol=0)


def _check(dev, kind, total, emap, rtol=RTOL):
    indptr = _segments(kind, total)
    nnz, nseg = int(indptr[-1]), indptr.size - 1
    rng = np.random.default_rng(nnz)
    data = (rng.random(nnz) + 0.25).astype(np.float32)
    order = rng.permutation(nnz) if emap else np.arange(nnz)
    w = data[order].astype(np.float64)
    lens = np.diff(indptr)
    owner = np.repeat(np.arange(nseg), lens)
    want = np.bincount(owner, weights=w * w, minlength=nseg)
    em = to_dev(order, dev) if emap else None
    out = torch.full((nseg,), -1.0, device=dev)
    capi.segment_sum(to_dev(indptr, dev), em, None, to_dev(data, dev), 2, out)
    got = out.cpu().numpy()
    np.testing.assert_allclose(got, want, rtol=rtol)
    short = np.flatnonzero((lens <= 16) & (lens > 0))[:3000]
    for s in short:  # in edge order: the bits of a sequential sum
        acc = np.float32(0)
        for e in order[indptr[s]:indptr[s + 1]]:
            acc = np.float32(acc + data[e] * data[e])
        assert got[s] == acc
    out = torch.full((nnz,), -1.0, device=dev)
    capi.segment_normalize(to_dev(indptr, dev), em, to_dev(data, dev), out)
    total_of = np.bincount(owner, weights=w, minlength=nseg)
    want = np.empty(nnz)
    want[order] = w / total_of[owner]
    np.testing.assert_allclose(out.cpu().numpy(), want, rtol=rtol)


@pytest.mark.parametrize("emap", [False, True])
@pytest.mark.parametrize("kind,total", [("lane", 200), ("mixed", 150_000), ("border", 2_300_000),
                                        ("hub", 150_000), ("gaps", 150_000)])  # (gaps: by marks)
@pytest.mark.parametrize("front", [1, 4096, 10_003])
@pytest.mark.parametrize("count", ["edges", "array"])
def test_first_offset_not_zero(dev, count, front, kind, total, emap):
    """A range of a larger matrix's columns: the offsets start at `front`, the data (and the edge
    map) go on behind the last one or end there, and the caller's count is the range's own or the
    array's.  Edges outside are neither summed nor divided."""
    indptr = _segments(kind, total)
    edges, nseg = int(indptr[-1]), indptr.size - 1
    behind = 0 if count == "edges" else 5000
    held = front + edges + behind
    rng = np.random.default_rng(edges)
    data = (rng.random(held) + 0.25).astype(np.float32)
    order = rng.permutation(held) if emap else np.arange(held)
    w = data[order[front:front + edges]].astype(np.float64)
    owner = np.repeat(np.arange(nseg), np.diff(indptr))
    ptr, d = to_dev(indptr + front, dev), to_dev(data, dev)
    em = to_dev(order, dev) if emap else None
    nnz = edges if count == "edges" else held
    L, st = capi.lib(), capi._stream(dev)
    ws = capi.workspace(L.gs_segment_workspace_bytes(capi._i64(nseg), capi._i64(nnz)), dev)

    out = torch.full((nseg,), -1.0, device=dev)
    capi._check(L.gs_segment_sum(capi._ptr(ptr), capi._ptr(em), capi._ptr(None), 8, capi._ptr(d),
                                 capi._i64(nseg), capi._i64(nnz), capi._i64(2), capi._ptr(out),
                                 capi._ptr(ws), ctypes.c_size_t(ws.numel()), st), "sum")
    np.testing.assert_allclose(out.cpu().numpy(), np.bincount(owner, weights=w * w, minlength=nseg),
                               rtol=RTOL)
    out = torch.full((held,), -1.0, device=dev)
    capi._check(L.gs_segment_normalize(capi._ptr(ptr), capi._ptr(em), capi._ptr(d), capi._i64(nseg),
                                       capi._i64(nnz), capi._ptr(out), capi._ptr(ws),
                                       ctypes.c_size_t(ws.numel()), st), "normalise")
    want = np.full(held, -1.0)
    want[order[front:front + edges]] = w / np.bincount(owner, weights=w, minlength=nseg)[owner]
    np.testing.assert_allclose(out.cpu().numpy(), want, rtol=RTOL)


def test_all_empty_behind_a_first_offset(dev):
    ptr = torch.full((6,), 4096, dtype=torch.int64, device=dev)
    data = torch.rand(9000, device=dev)
    out = torch.full((5,), -1.0, device=dev)
    capi.segment_sum(ptr, None, None, data, 1, out)
    assert torch.equal(out, torch.zeros(5, device=dev))
    out = torch.full((9000,), -1.0, device=dev)
    capi.segment_normalize(ptr, None, data, out)
    assert torch.equal(out, torch.full((9000,), -1.0, device=dev))


@pytest.mark.parametrize("nseg", [1, 64, 4095, 4096, 4097])
@pytest.mark.parametrize("lens", [[0, 1], [0, 0, 0, 2, 1], [1], [0, 0, 0, 17]])
def test_few_edges_of_few_segments(dev, nseg, lens):
    """Fewer edges than twice the segments, on both sides of the number of segments up to which offsets are walked
    and none are marked: bits of sequential sums, zeros of empty segments, and quotients of one rounding."""
    lens = np.resize(lens, nseg)
    lens[-1] = 3
    indptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    nnz = int(indptr[-1])
    data = (np.random.default_rng(nseg).random(nnz) + 0.25).astype(np.float32)
    out = torch.full((nseg,), -1.0, device=dev)
    capi.segment_sum(to_dev(indptr, dev), None, None, to_dev(data, dev), 1, out)
    want = np.bincount(np.repeat(np.arange(nseg), lens), weights=data.astype(np.float64), minlength=nseg)
    got = out.cpu().numpy()
    np.testing.assert_allclose(got, want, rtol=RTOL)
    assert (got[lens == 0] == 0).all()
    out = torch.full((nnz,), -1.0, device=dev)
    capi.segment_normalize(to_dev(indptr, dev), None, to_dev(data, dev), out)
    np.testing.assert_allclose(out.cpu().numpy(), data / np.repeat(want, lens), rtol=RTOL)
