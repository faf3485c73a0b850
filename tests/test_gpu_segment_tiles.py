"""Segment sums and normalisation by 4096-edge tiles against the oracle: segments around the
lengths a lane, sixteen lanes and a wave add up, on both sides of tile borders, with and
without an edge map, with runs of empty segments between."""
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
    np.testing.assert_allclose(got, want, rtol=RTOL)
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
    np.testing.assert_allclose(out.cpu().numpy(), want, rtol=RTOL)
