"""Edge lists: the node count of a loaded COO, the sort's large tiles, offsets over gaps of ids."""
import numpy as np
import pytest
import torch

import graph_sampling_amd as gs
from graph_sampling_amd import capi
from util import to_dev

pytestmark = pytest.mark.gpu
ID_DTYPES = [torch.int32, torch.int64]


@pytest.mark.parametrize("idt", ID_DTYPES)
@pytest.mark.parametrize("E", [1, 4095, 4096, 4097, 70000])
@pytest.mark.parametrize("how", ["complete", "second_larger", "first_larger", "huge", "negative"])
def test_node_count_of_an_edge_list(dev, E, how, idt):
    rng = np.random.default_rng(E)
    row, col = rng.integers(0, max(1, E // 3), E), rng.integers(0, max(1, E // 3), E)
    if how == "complete":          # the first end holds every id: the second is not counted
        row = np.arange(E) % (E // 3 + 1)
    elif how == "second_larger":   # gaps in both, the second end with more ids
        row, col = (row // 7) * 7, (col // 2) * 2
    elif how == "first_larger":
        row, col = (row // 2) * 2, (col // 7) * 7
    elif how == "huge":            # an id far beyond the number of edges: counted another way
        col[E // 2] = (1 << 31) - 1
    else:
        row[E // 2] = -1
    g = gs.Graph(False)
    g._CAPI_LoadCOO(to_dev(row, dev, idt), to_dev(col, dev, idt))
    assert g._CAPI_GetNumRows() == max(np.unique(row).size, np.unique(col).size)


SLICE = 39936 * 32  # ids of one LDS bitmap


@pytest.mark.parametrize("idt", ID_DTYPES)
@pytest.mark.parametrize("largest", [40, SLICE - 1, SLICE, 2 * SLICE, 5 * SLICE + 7, 8 * SLICE - 1,
                                     8 * SLICE])
@pytest.mark.parametrize("how", ["complete", "second_larger", "first_larger"])
def test_node_count_of_a_long_list(dev, largest, how, idt):
    """Lists counted by bits in LDS, the largest id on both sides of a slice's and of the last
    slice's end (beyond it: by bytes), in the first end or in the second only."""
    E = (1 << 22) + 3
    gen = torch.Generator(device=dev)
    gen.manual_seed(largest % 1_000_003)
    row, col = (torch.randint(0, largest + 1, (E,), generator=gen, device=dev) for _ in range(2))
    if how == "complete" and largest < E:
        row = torch.arange(E, device=dev) % (largest + 1)
    elif how == "second_larger":
        row = row // 3
        col[E - 1] = largest
    else:
        col = col // 3
        row[E // 2] = largest
    g = gs.Graph(False)
    g._CAPI_LoadCOO(row.to(idt), col.to(idt))
    assert g._CAPI_GetNumRows() == max(torch.unique(row).numel(), torch.unique(col).numel())


@pytest.mark.parametrize("idt", ID_DTYPES)
@pytest.mark.parametrize("stray", [-1, (1 << 31) - 1])
def test_node_count_of_a_long_list_with_a_stray_id(dev, stray, idt):
    E = 1 << 22
    row, col = torch.arange(E, device=dev) % 1000, torch.arange(E, device=dev) % 77
    col[E - 2] = stray
    g = gs.Graph(False)
    g._CAPI_LoadCOO(row.to(idt), col.to(idt))
    assert g._CAPI_GetNumRows() == 1000


@pytest.mark.parametrize("idt", ID_DTYPES)
@pytest.mark.parametrize("extra", [0, 1, 8191])
@pytest.mark.parametrize("num_keys", [200, 60_000, 3_000_000])
def test_sort_with_large_tiles(dev, num_keys, extra, idt):
    E = (1 << 22) + extra
    gen = torch.Generator(device=dev)
    gen.manual_seed(num_keys + extra)
    key = (torch.rand(E, generator=gen, device=dev) ** 3 * num_keys).to(idt)
    value = torch.randint(0, 1 << 31, (E,), generator=gen, device=dev).to(idt)
    if idt == torch.int64 and extra == 1:
        value[E // 2] = 1 << 40    # one value beyond 32 bits
    ip, val, perm = capi.coo2csc(key, value, num_keys, False)
    want = torch.sort(key, stable=True)
    assert torch.equal(perm, want.indices) and torch.equal(val, value[want.indices])
    ends = torch.cumsum(torch.bincount(key.long(), minlength=num_keys), 0)
    assert int(ip[0]) == 0 and torch.equal(ip[1:], ends)


@pytest.mark.parametrize("idt", ID_DTYPES)
@pytest.mark.parametrize("E", [64 * 4096, 64 * 4096 + 1, 70 * 4096 - 1, (1 << 22) - 1, (1 << 22) + 8193])
@pytest.mark.parametrize("num_keys,skew", [(257, 1), (65536, 3), (65537, 3), (1 << 22, 12), (1 << 24, 1)])
def test_sort_with_the_values_in_its_words(dev, num_keys, skew, E, idt):
    """From 65 tiles on a sort of two or three digits carries the values in its 64-bit words, beside
    a digit of the key or two and the edge's position: the largest value that fits beside two, and one
    more."""
    gen = torch.Generator(device=dev)
    gen.manual_seed(num_keys + E)
    key = (torch.rand(E, generator=gen, device=dev, dtype=torch.float64) ** skew * num_keys).to(idt)
    bits = min(32, 48 - (E - 1).bit_length(), 31 if idt == torch.int32 else 32)
    value = torch.randint(0, 1 << 20, (E,), generator=gen, device=dev).to(idt)
    want = torch.sort(key, stable=True)
    ends = torch.cumsum(torch.bincount(key.long(), minlength=num_keys), 0)
    for extra in ([0, 1] if bits < 31 else [0]):
        value[E // 3] = (1 << bits) - 1 + extra
        ip, val, perm = capi.coo2csc(key, value, num_keys, False)
        assert torch.equal(perm, want.indices) and torch.equal(val, value[want.indices])
        assert int(ip[0]) == 0 and torch.equal(ip[1:], ends)


@pytest.mark.parametrize("idt", ID_DTYPES)
@pytest.mark.parametrize("E,num_keys", [(64 * 4096 + 1, 257), (64 * 4096 + 1, 64 * 4096 + 1), (64 * 4096 + 1, 64 * 4096 + 2),
                                        (1_000_003, 65_536), ((1 << 22) + 5, 65_537), (1 << 24, 1 << 24)])
@pytest.mark.parametrize("keys", ["first", "last", "ends", "one low digit", "few"])
def test_offsets_from_the_last_pass(dev, keys, E, num_keys, idt):
    """Two digits and three, as many columns as edges and one more, and as many as three digits hold; keys
    that leave long runs of columns without edges in front, in between and behind, which single tiles write."""
    gen = torch.Generator(device=dev)
    gen.manual_seed(E)
    choice = {"first": [0], "last": [num_keys - 1], "ends": [0, num_keys - 1],
              "one low digit": list(range(5, num_keys, 256)), "few": [1, 3, 255, 256, num_keys // 2 + 1]}[keys]
    choice = torch.tensor([k for k in choice if k < num_keys], device=dev)
    key = choice[torch.randint(0, choice.numel(), (E,), generator=gen, device=dev)].to(idt)
    ip, val, perm = capi.coo2csc(key, key, num_keys, False)
    assert torch.equal(val, torch.sort(key).values) and torch.equal(key[perm], val)
    ends = torch.cumsum(torch.bincount(key.long(), minlength=num_keys), 0)
    assert int(ip[0]) == 0 and torch.equal(ip[1:], ends)


@pytest.mark.parametrize("idt", ID_DTYPES)
@pytest.mark.parametrize("E,num_keys", [(64 * 4096 + 4, 65_536), (64 * 4096 + 4, 65_537),
                                        (1_300_000, 325_000), (1_300_000, 325_001), (1_299_999, 324_999),
                                        ((1 << 22) + 5, (1 << 22) + 5), ((1 << 22) + 5, (1 << 22) + 6)])
@pytest.mark.parametrize("keys", ["first", "last", "ends", "one low digit", "few"])
def test_offsets_on_both_sides_of_the_last_pass_s_lines(dev, keys, E, num_keys, idt):
    """Up to as many columns as edges the last pass writes the offsets; in small tiles a quarter as many, and of three
    digits only from 1.3 M edges on."""
    test_offsets_from_the_last_pass(dev, keys, E, num_keys, idt)


@pytest.mark.parametrize("idt", ID_DTYPES)
@pytest.mark.parametrize("E,num_keys", [(300_007, 65_536), (1_300_003, 300_000), ((1 << 22) + 5, 1 << 22), ((1 << 22) + 5, 3_000_001),
                                        ((1 << 24) - 7, (1 << 24) - 7)])
def test_offsets_of_one_tile_with_gaps_of_every_length(dev, E, num_keys, idt):
    """Nearly all edges share two lower halves, so one tile finds the columns of all others: gaps on both sides of the
    lengths that a lane stores, a wave, and a launch behind the sort piece by piece, and those behind the last edges."""
    gen = torch.Generator(device=dev)
    gen.manual_seed(E)
    heavy = torch.arange(0, num_keys, 1 << 16, device=dev)
    heavy = torch.cat([heavy, heavy + 60_000])
    chain = torch.cumsum(torch.tensor([1, 4, 5, 6, 63, 64, 65, 127, 128, 129, 130, 2047, 2048, 2049, 4096, 4097, 30_000], device=dev), 0)
    rare = torch.cat([chain, chain + ((num_keys >> 16) - 1 << 16), torch.randint(0, num_keys, (3000,), generator=gen, device=dev)])
    rare = rare[(rare >= 0) & (rare & 0xFFFF < 60_000)]
    heavy = heavy[heavy < num_keys]
    key = torch.cat([rare, heavy[torch.randint(0, heavy.numel(), (E - rare.numel(),), generator=gen, device=dev)]])
    key = key[torch.randperm(E, generator=gen, device=dev)].to(idt)
    ip, val, perm = capi.coo2csc(key, key, num_keys, False)
    assert torch.equal(val, torch.sort(key).values) and torch.equal(key[perm], val)
    ends = torch.cumsum(torch.bincount(key.long(), minlength=num_keys), 0)
    assert int(ip[0]) == 0 and torch.equal(ip[1:], ends)


@pytest.mark.parametrize("idt", ID_DTYPES)
@pytest.mark.parametrize("less", [0, 1])
@pytest.mark.parametrize("num_keys", [60_000, 3_000_000])
def test_sort_with_long_results(dev, num_keys, less, idt):
    """Results of 128 MB and of an edge less, by two digits and by three: the last pass writes the longer ones past
    the caches, and fetches values again where one does not fit its bits."""
    edge = 8 + 4 + (4 if idt == torch.int32 else 8)  # position, key and value
    E = -(-(1 << 27) // edge) - less
    gen = torch.Generator(device=dev)
    gen.manual_seed(num_keys)
    key = (torch.rand(E, generator=gen, device=dev, dtype=torch.float64) ** 3 * num_keys).to(idt)
    value = torch.randint(0, num_keys, (E,), generator=gen, device=dev).to(idt)
    want = torch.sort(key, stable=True).indices
    ends = torch.cumsum(torch.bincount(key.long(), minlength=num_keys), 0)
    # (two digits leave 32 bits for a value of 23-bit positions, three leave 25, or 24 beside 24-bit positions)
    for wide in [0, (1 << 31) - 1] + ([1 << 40] if idt == torch.int64 else []):
        value[E // 3] = wide
        ip, val, perm = capi.coo2csc(key, value, num_keys, False)
        assert torch.equal(perm, want) and torch.equal(val, value[want])
        assert int(ip[0]) == 0 and torch.equal(ip[1:], ends)


@pytest.mark.parametrize("idt", ID_DTYPES)
@pytest.mark.parametrize("num_keys", [60_000, 65_537])
def test_sort_of_values_unlike_the_keys(dev, num_keys, idt):
    """Values below a bound that the caller knows, with two digits of the key (which leave them all 32
    bits) and three: in the words as long as the bound fits there, else beside them; the same
    result when the bound is not kept, up to beyond 32 bits."""
    E = 3_000_000  # (22 bits of a position: 34 and 26 are left)
    gen = torch.Generator(device=dev)
    gen.manual_seed(num_keys)
    key = torch.randint(0, num_keys, (E,), generator=gen, device=dev).to(idt)
    want = torch.sort(key, stable=True).indices
    for top in ([1 << 26, (1 << 26) + 1, (1 << 31) - 1] + ([1 << 32, (1 << 32) + 1, 1 << 40] if idt == torch.int64 else [])):
        value = torch.randint(0, top, (E,), generator=gen, device=dev, dtype=torch.int64)
        value[E // 2] = top - 1
        value = value.to(idt)
        for bound in (top, 0, num_keys):
            _, val, perm = capi.coo2csc(key, value, num_keys, False, num_values=bound)
            assert torch.equal(perm, want) and torch.equal(val, value[want])


@pytest.mark.parametrize("idt", ID_DTYPES)
@pytest.mark.parametrize("keys", [[0], [9999], [0, 17, 18, 9000], [5000, 5016, 5032, 7200, 9998]])
def test_offsets_over_gaps(dev, keys, idt):
    """Sorted keys, more edges than columns, gaps on both sides of the lengths one lane, a wave
    and a workgroup fill, at the front, in between and at the end."""
    num_keys, E = 10_000, 12_289
    rng = np.random.default_rng(len(keys))
    key = np.sort(rng.choice(np.array(keys), E))
    ip, _, _ = capi.coo2csc(to_dev(key, dev, idt), to_dev(key, dev, idt), num_keys, True)
    want = np.concatenate([[0], np.cumsum(np.bincount(key, minlength=num_keys))])
    assert np.array_equal(ip.cpu().numpy(), want)


@pytest.mark.parametrize("idt", ID_DTYPES)
@pytest.mark.parametrize("E", [999, 1000, 31_999, 32_000, 32_001, 64_000, 64_001, 500_000])
def test_offsets_by_edges_per_column(dev, E, idt):
    """Both sides of the lines between the two ways from sorted keys to offsets."""
    num_keys = 1000
    key = np.sort((np.random.default_rng(E).random(E) ** 3 * num_keys).astype(np.int64))
    ip, _, _ = capi.coo2csc(to_dev(key, dev, idt), to_dev(key, dev, idt), num_keys, True)
    want = np.concatenate([[0], np.cumsum(np.bincount(key, minlength=num_keys))])
    assert np.array_equal(ip.cpu().numpy(), want)
