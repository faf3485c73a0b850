"""u_dot_v and its siblings by (edge, head) pairs: tile borders, row widths, operand targets."""
import numpy as np
import pytest
import torch

from graph_sampling_amd import capi
from tests.util import to_dev

pytestmark = pytest.mark.gpu
TILE, SMALL = 256, 64  # edges of a tile; of a tile where there are fewer than 2048 large ones
# an fp32 sum of R products in any order is within R + 1 roundings of the exact one
EPS = 2.0 ** -24


def _check(dev, E, heads, R, targets, idt, csc, maps, shift):
    rng = np.random.default_rng(E + 31 * heads + R)
    n = 300
    row = rng.integers(0, n, E)
    col = np.sort(rng.integers(0, n, E) // 7 * 7)  # six of seven columns are empty
    e_ids = rng.permutation(E) if maps else None
    eid = e_ids if maps else np.arange(E)
    sel = {0: row, 1: eid, 2: col}
    lhs, rhs = (rng.standard_normal((E if t == 1 else n, heads, R)).astype(np.float32) for t in targets)

    def off(a):  # `shift` floats behind a 16-byte border
        d = torch.empty(a.size + shift, dtype=torch.float32, device=dev)[shift:]
        d.copy_(to_dev(a, dev).view(-1))
        return d.view(a.shape)

    out = torch.full((E, heads, 1), 7.0, device=dev)
    args = (off(lhs), off(rhs), out, *targets, heads * R, heads * R, heads, R)
    ids = to_dev(eid, dev) if maps else None
    if csc:
        indptr = np.concatenate([[0], np.cumsum(np.bincount(col, minlength=n))])
        capi.sddmm_csc("dot", to_dev(indptr, dev), to_dev(row, dev, idt), ids, None, *args)
    else:
        capi.sddmm_coo("dot", to_dev(row, dev, idt), to_dev(col, dev, idt), ids, *args)
    got = out.cpu().numpy()[eid, :, 0]
    x, y = (a[sel[t]].astype(np.float64) for a, t in zip((lhs, rhs), targets))
    exact, size = (x * y).sum(-1), np.abs(x * y).sum(-1)
    assert np.all(np.abs(got - exact) <= (R + 1) * EPS * size)


@pytest.mark.parametrize("heads,R", [(1, 2), (1, 3), (1, 8), (1, 50), (1, 64), (1, 130), (2, 25),
                                     (3, 5), (8, 8), (4, 16), (300, 2), (5, 12)])
@pytest.mark.parametrize("csc", [False, True])
def test_widths_and_heads(dev, heads, R, csc):
    for E in (1, SMALL - 1, SMALL + 1, 3 * SMALL, 1000):
        _check(dev, E, heads, R, (0, 2), torch.int32 if E % 2 else torch.int64, csc, E == 1000, 0)


@pytest.mark.parametrize("shift", [1, 2])  # reads of 4 and of 8 bytes
@pytest.mark.parametrize("targets", [(0, 2), (2, 0), (1, 2), (0, 1)])
def test_unaligned_rows_and_targets(dev, shift, targets):
    _check(dev, 777, 2, 16, targets, torch.int64, False, True, shift)
    _check(dev, 777, 1, 16, targets, torch.int32, True, False, shift)


@pytest.mark.parametrize("E", [2048 * TILE - 1, 2048 * TILE + 1])
def test_large_tiles(dev, E):
    _check(dev, E, 1, 16, (0, 2), torch.int32, False, False, 0)
    _check(dev, E, 3, 4, (0, 2), torch.int64, True, True, 0)
