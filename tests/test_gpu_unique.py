"""GPU parity: unique / relabel through the C ABI vs the CPU oracle and closed forms."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from graph_sampling_amd import capi
from tests.util import to_dev

pytestmark = pytest.mark.gpu


def _closed_form_unique(x):
    u, first = np.unique(x, return_index=True)
    return u[np.argsort(first, kind="stable")]


def _run(mapping, queries, dev, idt):
    dm = [to_dev(m, dev, idt) for m in mapping]
    # a query that IS a mapping tensor must alias it (the slot-gather path)
    dq = []
    for q in queries:
        hit = [i for i, m in enumerate(mapping) if m is q]
        dq.append(dm[hit[0]] if hit else to_dev(q, dev, idt))
    frontier, num, outs = capi.unique_relabel(dm, dq)
    n = int(num.item())
    return frontier[:n].cpu().numpy().astype(np.int64), [o.cpu().numpy().astype(np.int64) for o in outs]


@pytest.mark.parametrize("idt", [torch.int64, torch.int32])
@pytest.mark.parametrize("n", [0, 1, 5, 2048, 2049, 100000])
def test_unique_first_occurrence(dev, idt, n):
    rng = np.random.default_rng(n)
    x = rng.integers(0, max(1, n // 3) + 5, size=n).astype(np.int64) * 7919 % 100003
    frontier, _ = _run([x], [], dev, idt)
    assert np.array_equal(frontier, _closed_form_unique(x))
    assert np.array_equal(frontier, O.unique(x))


@pytest.mark.parametrize("idt", [torch.int64, torch.int32])
def test_relabel_seeds_first(dev, idt):
    rng = np.random.default_rng(0)
    seeds = rng.permutation(50000)[:1024].astype(np.int64)
    rows = rng.integers(0, 50000, size=15000).astype(np.int64)
    other = rng.integers(0, 60000, size=777).astype(np.int64)  # holds ids absent from the mapping
    frontier, outs = _run([seeds, rows], [rows, other, seeds], dev, idt)
    want_frontier, want = O.relabel([seeds, rows], [rows, other, seeds])
    assert np.array_equal(frontier, want_frontier)
    for g, w in zip(outs, want):
        assert np.array_equal(g, w)
    assert np.array_equal(frontier[:1024], seeds)          # seeds occupy the head of the frontier
    assert np.array_equal(frontier[outs[0]], rows)         # frontier[relabelled] == original
    assert (outs[1] == -1).any() and np.array_equal(outs[2], np.arange(1024))


def test_relabel_reference_vector(dev):
    # reference tests/test_relabel.cc:7-26: slicing cols 1..3 of the 20x5 graph with relabel
    rows = np.arange(5, 20, dtype=np.int64)
    frontier, outs = _run([rows], [rows], dev, torch.int64)
    assert np.array_equal(frontier, rows)
    assert np.array_equal(outs[0], np.arange(15))


def test_unique_large_consecutive_and_clustered(dev):
    # consecutive ids (the case that clusters under an identity hash) plus heavy duplication
    x = np.concatenate([np.arange(300000), np.arange(300000)[::-1], np.full(1000, 42)]).astype(np.int64)
    frontier, outs = _run([x], [x], dev, torch.int64)
    assert np.array_equal(frontier, np.arange(300000))
    assert np.array_equal(frontier[outs[0]], x)


def test_four_mapping_spans(dev):
    rng = np.random.default_rng(4)
    spans = [rng.integers(0, 5000, size=s).astype(np.int64) for s in (10, 0, 3000, 2049)]
    frontier, outs = _run(spans, [spans[3], spans[0]], dev, torch.int64)
    want_frontier, want = O.relabel(spans, [spans[3], spans[0]])
    assert np.array_equal(frontier, want_frontier)
    for g, w in zip(outs, want):
        assert np.array_equal(g, w)


@pytest.mark.parametrize("idt", [torch.int64, torch.int32])
@pytest.mark.parametrize("n", [512 * 2048 - 1, 512 * 2048, 512 * 2048 + 1, 3_000_000])
def test_relabel_million_items(dev, idt, n):
    """Around 2^20 items (512 compaction tiles: several look-back bursts) and 3 M, with an aliased
    and a plain query, heavy and light repetition."""
    rng = np.random.default_rng(n)
    seeds = rng.permutation(5_000_000)[:1000].astype(np.int64)
    rows = np.concatenate([rng.integers(0, 2000, size=n // 2),            # hubs: heavy repetition
                           rng.integers(0, 5_000_000, size=n - 1000 - n // 2)]).astype(np.int64)
    rng.shuffle(rows)
    probe = rng.integers(0, 5_000_100, size=5000).astype(np.int64)        # some absent ids
    frontier, (rel_rows, rel_probe) = _run([seeds, rows], [rows, probe], dev, idt)
    want_frontier, (want_rows, want_probe) = O.relabel([seeds, rows], [rows, probe])
    assert np.array_equal(frontier, want_frontier)
    assert np.array_equal(rel_rows, want_rows)
    assert np.array_equal(rel_probe, want_probe)
    assert (want_probe == -1).any()


@pytest.mark.parametrize("idt", [torch.int64, torch.int32])
def test_relabel_every_item_the_same_key(dev, idt):
    """All tiles fight for one slot; one first occurrence in tile 0, every other tile has none."""
    x = np.full(300_000, 12345, dtype=np.int64)
    y = np.arange(300_000, dtype=np.int64) % 3
    frontier, (rx, ry) = _run([x, y], [x, y], dev, idt)
    assert np.array_equal(frontier, np.array([12345, 0, 1, 2]))
    assert (rx == 0).all() and np.array_equal(ry, y + 1)


def _batches(rng, B, n_nodes, max_seeds, max_ids, empty_every=0):
    seeds, ids, sp, ip = [], [], [0], [0]
    for b in range(B):
        ns = 0 if empty_every and b % empty_every == 1 else int(rng.integers(1, max_seeds + 1))
        ni = 0 if empty_every and b % empty_every == 2 else int(rng.integers(0, max_ids + 1))
        seeds.append(rng.permutation(n_nodes)[:ns])
        ids.append(rng.integers(0, n_nodes, size=ni))
        sp.append(sp[-1] + ns)
        ip.append(ip[-1] + ni)
    cat = lambda xs: np.concatenate(xs).astype(np.int64) if xs else np.empty(0, np.int64)  # noqa: E731
    return cat(seeds), np.array(sp, dtype=np.int64), cat(ids), np.array(ip, dtype=np.int64)


@pytest.mark.parametrize("idt", [torch.int64, torch.int32])
@pytest.mark.parametrize("B,max_seeds,max_ids,empty_every", [(1, 50, 400, 0), (7, 30, 300, 3),
                                                               (64, 256, 4000, 0), (300, 8, 40, 5),
                                                               # both sides of the 511 batches whose
                                                               # offsets a workgroup keeps in LDS
                                                               (511, 6, 30, 7), (512, 6, 30, 7),
                                                               (1500, 4, 12, 4)])
def test_batch_csr_relabel_matches_oracle(dev, idt, B, max_seeds, max_ids, empty_every):
    """Every batch is relabelled on its own: the same id in two batches gets two ranks."""
    rng = np.random.default_rng(B)
    seeds, sp, ids, ip = _batches(rng, B, 3000, max_seeds, max_ids, empty_every)
    unique, unique_ptr, out_ids, num = capi.batch_csr_relabel(to_dev(seeds, dev, idt), to_dev(sp, dev),
                                                              to_dev(ids, dev, idt), to_dev(ip, dev))
    w_unique, w_ptr, w_out = O.batch_csr_relabel(seeds, sp, ids, ip)
    U = int(num.item())
    assert U == w_unique.size
    assert np.array_equal(unique_ptr.cpu().numpy(), w_ptr)
    assert np.array_equal(unique[:U].cpu().numpy().astype(np.int64), w_unique)
    assert np.array_equal(out_ids.cpu().numpy().astype(np.int64), w_out)
    # closed form per batch, independent of the oracle's hash table
    for b in range(B):
        x = np.concatenate([seeds[sp[b]:sp[b + 1]], ids[ip[b]:ip[b + 1]]])
        f = _closed_form_unique(x)
        assert np.array_equal(w_unique[w_ptr[b]:w_ptr[b + 1]], f)
        assert np.array_equal(f[w_out[ip[b]:ip[b + 1]]], ids[ip[b]:ip[b + 1]])


def _check_batch_relabel(dev, idt, seeds, sp, ids, ip, narrow, path):
    unique, unique_ptr, out_ids, num = capi.batch_csr_relabel(
        to_dev(seeds, dev, idt), to_dev(sp, dev), to_dev(ids, dev, idt), to_dev(ip, dev),
        narrow=narrow, path=path)
    w_unique, w_ptr, w_out = O.batch_csr_relabel(seeds, sp, ids, ip)
    U = int(num.item())
    assert U == w_unique.size
    assert np.array_equal(unique_ptr.cpu().numpy(), w_ptr)
    assert np.array_equal(unique[:U].cpu().numpy().astype(np.int64), w_unique)
    assert np.array_equal(out_ids.cpu().numpy().astype(np.int64), w_out)


@pytest.mark.parametrize("idt,narrow", [(torch.int32, False), (torch.int64, True)])
@pytest.mark.parametrize("B,max_seeds,max_ids,empty_every", [(1, 50, 400, 0), (7, 30, 300, 3),
                                                               (64, 256, 4000, 0), (300, 8, 40, 5),
                                                               (511, 6, 30, 7), (3, 3000, 50000, 0)])
def test_batch_csr_relabel_through_bins_small(dev, idt, narrow, B, max_seeds, max_ids, empty_every):
    """The binned relabel (hash classes + LDS tables) forced on inputs far below the size it is
    chosen for: same frontiers, offsets and ranks as the oracle, empty batches included."""
    rng = np.random.default_rng(B + 1)
    seeds, sp, ids, ip = _batches(rng, B, 3000, max_seeds, max_ids, empty_every)
    _check_batch_relabel(dev, idt, seeds, sp, ids, ip, narrow, "bins")


@pytest.mark.parametrize("idt,narrow", [(torch.int32, False), (torch.int64, True)])
@pytest.mark.parametrize("shape", ["even", "one_large", "hubs", "single", "all_same"])
def test_batch_csr_relabel_through_bins_at_size(dev, idt, narrow, shape):
    """Half a million items and more, which the library takes through bins by itself: batches of equal
    size, one batch that holds nearly everything (thousands of classes) beside tiny and empty ones, ids that
    repeat tens of thousands of times, one batch only, one id only; the last batches empty."""
    rng = np.random.default_rng(len(shape))
    n_nodes = 1 << 21
    if shape == "even":
        sizes = [(1000, 60000)] * 16
    elif shape == "one_large":
        sizes = [(5, 40), (0, 0), (2000, 1_500_000), (1, 0), (0, 7), (300, 9000), (0, 0)]
    elif shape == "hubs":
        sizes = [(500, 200000)] * 4
    elif shape == "single":
        sizes = [(4096, 900000)]
    else:
        sizes = [(1, 300000), (1, 300000)]
    seeds, ids, sp, ip = [], [], [0], [0]
    for ns, ni in sizes:
        seeds.append(rng.permutation(n_nodes)[:ns])
        if shape == "hubs":     # a few ids hold most of the positions
            x = (rng.random(ni) ** 8 * n_nodes).astype(np.int64)
        elif shape == "all_same":
            x = np.full(ni, 77, dtype=np.int64)
        else:
            x = rng.integers(0, n_nodes, size=ni)
        ids.append(x)
        sp.append(sp[-1] + ns)
        ip.append(ip[-1] + ni)
    seeds = np.concatenate(seeds).astype(np.int64)
    ids = np.concatenate(ids).astype(np.int64)
    assert seeds.size + ids.size >= 1 << 19
    _check_batch_relabel(dev, idt, seeds, np.array(sp, dtype=np.int64), ids,
                         np.array(ip, dtype=np.int64), narrow, None)


@pytest.mark.parametrize("idt,narrow", [(torch.int32, False), (torch.int64, True)])
@pytest.mark.parametrize("B,items", [(3, (1 << 17) - 1), (3, 1 << 17), (3, (1 << 17) + 1),
                                     (1, 1 << 20), (1, (1 << 20) + 1)])
def test_batch_csr_relabel_at_the_lines_of_its_forms(dev, idt, narrow, B, items):
    """Hash regions below 2^17 items, bins from there on; by runs up to 2^20 items a batch on average,
    counted and scattered beyond."""
    rng = np.random.default_rng(items)
    ends = np.concatenate([[0], np.sort(rng.integers(0, items + 1, B - 1)), [items]])
    sizes = np.diff(ends)
    sp = np.concatenate([[0], np.cumsum(sizes // 5)]).astype(np.int64)
    ip = np.concatenate([[0], np.cumsum(sizes - sizes // 5)]).astype(np.int64)
    seeds = rng.integers(0, 1 << 18, sp[-1]).astype(np.int64)
    ids = (rng.random(ip[-1]) ** 2 * (1 << 18)).astype(np.int64)
    assert seeds.size + ids.size == items
    _check_batch_relabel(dev, idt, seeds, sp, ids, ip, narrow, None)


@pytest.mark.parametrize("idt,narrow", [(torch.int32, False), (torch.int64, True)])
@pytest.mark.parametrize("items,spread", [([1, 63, 64, 65], 1 << 20), ([8191, 8192, 8193, 0, 1], 1 << 20),
                                          ([2048, 2049, 4097, 0, 0, 16385], 40),
                                          ([64 * 8192, 64 * 8192 + 1], 1 << 20),
                                          ([70_000, 100_000], 300)])
def test_batch_csr_relabel_runs_around_their_tiles(dev, idt, narrow, items, spread):
    """A tile is 8192 items of a batch, a class about 2048, a piece of a run 64 records; a workgroup
    looks at 64 tiles' runs at a time and keeps 128 pieces: batches on both sides of each (half of
    the ids drawn from `spread`, so that a class's runs may be a few long ones)."""
    rng = np.random.default_rng(len(items) + spread)
    seeds, ids, sp, ip = [], [], [0], [0]
    for m in items:
        ns = m // 3
        seeds.append(rng.permutation(1 << 20)[:ns])
        ids.append(np.where(rng.random(m - ns) < 0.5, rng.integers(0, spread, m - ns),
                            rng.integers(0, 1 << 20, m - ns)))
        sp.append(sp[-1] + ns)
        ip.append(ip[-1] + m - ns)
    _check_batch_relabel(dev, idt, np.concatenate(seeds).astype(np.int64), np.array(sp, dtype=np.int64),
                         np.concatenate(ids).astype(np.int64), np.array(ip, dtype=np.int64), narrow,
                         "bins")


def test_batch_csr_relabel_one_batch_beyond_the_counters(dev):
    """Batches small on average and one with more classes than a tile's LDS counters; around it
    batches on both sides of one class."""
    rng = np.random.default_rng(9)
    sizes = [(3, 2045), (0, 2049), (10, 9_000_000), (1, 0)] + [(2, 90)] * 12
    sp = np.concatenate([[0], np.cumsum([a for a, _ in sizes])]).astype(np.int64)
    ip = np.concatenate([[0], np.cumsum([n for _, n in sizes])]).astype(np.int64)
    seeds = rng.integers(0, 1 << 22, sp[-1]).astype(np.int64)
    ids = rng.integers(0, 1 << 22, ip[-1]).astype(np.int64)
    _check_batch_relabel(dev, torch.int32, seeds, sp, ids, ip, False, None)


def test_batch_csr_relabel_bins_report_what_they_cannot_take(dev):
    """An id beyond 32 bits among 64-bit ids promised to be narrow: -2, as on the hash regions.  A
    class with more distinct ids than its LDS table holds: -4 from the C ABI, and the host
    layer's operator repeats the call on hash regions by itself."""
    import graph_sampling_amd as gs
    gs.load_library()
    rng = np.random.default_rng(5)
    seeds = rng.permutation(1 << 20)[:100].astype(np.int64)
    ids = rng.integers(0, 1 << 20, size=(1 << 19) + 5).astype(np.int64)
    ids[1234] = (1 << 35) + 3
    sp, ip = np.array([0, 100], dtype=np.int64), np.array([0, ids.size], dtype=np.int64)
    num = capi.batch_csr_relabel(to_dev(seeds, dev), to_dev(sp, dev), to_dev(ids, dev),
                                 to_dev(ip, dev), narrow=True)[3]
    assert int(num.item()) == -2
    # one batch of 20 M distinct ids: 4096 classes of ~4900 distinct ids each, tables of 4096 slots
    n = 20_000_000
    ids = torch.randperm(n, device=dev, dtype=torch.int64).to(torch.int32)
    seeds = ids[:10].clone()
    t_sp = torch.tensor([0, 10], device=dev)
    t_ip = torch.tensor([0, n], device=dev)
    num = capi.batch_csr_relabel(seeds, t_sp, ids, t_ip)[3]
    assert int(num.item()) == -4
    uni, uni_ptr, rel, _ = torch.ops.gs_ops.BatchCSRRelabel(seeds, t_sp, ids, t_ip)
    # closed form: the seeds are the first ten ids, every other id is new, in order
    assert uni_ptr.cpu().tolist() == [0, n]
    assert torch.equal(uni, ids)
    assert torch.equal(rel, torch.arange(n, device=dev, dtype=torch.int32))


# a few tiles of the compaction, with keys all distinct, in long runs, and in between
@pytest.mark.parametrize("idt", [torch.int64, torch.int32])
@pytest.mark.parametrize("n", [8191, 8192, 8193, 16383, 16384, 16385])
@pytest.mark.parametrize("spread", ["distinct", "few", "mixed"])
def test_relabel_few_tiles_by_key_spread(dev, idt, n, spread):
    rng = np.random.default_rng(n)
    if spread == "distinct":
        rows = (rng.permutation(1 << 20)[:n - 100].astype(np.int64) * 7 + 3)
    elif spread == "few":           # long runs of the same key
        rows = rng.integers(0, 17, size=n - 100).astype(np.int64) * 65537
    else:
        rows = rng.integers(0, n // 2, size=n - 100).astype(np.int64)
    seeds = rows[rng.permutation(rows.size)[:100]]
    other = rng.integers(0, 1 << 21, size=999).astype(np.int64)
    frontier, outs = _run([seeds, rows], [rows, other], dev, idt)
    want_frontier, want = O.relabel([seeds, rows], [rows, other])
    assert np.array_equal(frontier, want_frontier)
    for g, w in zip(outs, want):
        assert np.array_equal(g, w)


def test_64_bit_ids_on_one_word_slots(dev):
    """GS_NARROW_IDS: 64-bit ids that fit 32 bits give the same frontier and ranks as the
    two-array table, lookups of ids beyond 32 bits come back absent, and a mapping id beyond
    32 bits is reported (-2) rather than truncated."""
    rng = np.random.default_rng(12)
    a = rng.integers(0, 5000, 30000).astype(np.int64) + 4_000_000_000     # still below 2^32
    b = rng.integers(0, 5000, 20000).astype(np.int64) + 4_000_000_000
    q = np.concatenate([b[:1000], np.array([1 << 40, (1 << 32) + 5], dtype=np.int64)])
    for narrow in (False, True):
        frontier, num, outs = capi.unique_relabel([to_dev(a, dev), to_dev(b, dev)],
                                                  [to_dev(b, dev), to_dev(q, dev)], narrow=narrow)
        w_frontier, w_outs = O.relabel([a, b], [b, q])
        U = int(num.item())
        assert U == w_frontier.size
        assert np.array_equal(frontier[:U].cpu().numpy(), w_frontier)
        assert np.array_equal(outs[0].cpu().numpy(), w_outs[0])
        assert np.array_equal(outs[1].cpu().numpy(), w_outs[1])
        assert outs[1][-1].item() == -1 and outs[1][-2].item() == -1
    big = a.copy()
    big[777] = (1 << 36) + 1
    _, num, _ = capi.unique_relabel([to_dev(big, dev)], [], narrow=True)
    assert int(num.item()) == -2
    # the same with lookups queued behind the pass that gave up: void outputs, but the call ends
    t_big = to_dev(big, dev)
    _, num, _ = capi.unique_relabel([t_big], [t_big, to_dev(q, dev)], narrow=True)
    assert int(num.item()) == -2
    frontier, num, _ = capi.unique_relabel([to_dev(big, dev)], [], narrow=False)
    assert np.array_equal(frontier[:int(num.item())].cpu().numpy(), O.relabel([big], [])[0])


@pytest.mark.parametrize("idt,narrow", [(torch.int32, False), (torch.int64, False),
                                        (torch.int64, True)])
@pytest.mark.parametrize("S,cap,held", [(1, 0, 0), (1, 255, 255), (100, 157, 156), (33, 70000, 69999)])
@pytest.mark.parametrize("spread", ["one", "few", "new"])
def test_relabel_behind_a_sampler_by_repeats(dev, idt, narrow, S, cap, held, spread):
    """Ids that repeat inside a workgroup meet in LDS when there are at least half as many items
    as ids; on both sides of that line the frontier and the ranks are the oracle's, the table
    is empty again and the next call finds it so.  (held: the true length, on the device)"""
    rng = np.random.default_rng(cap + len(spread))
    hi = {"one": 1, "few": 40, "new": 1 << 20}[spread]
    seeds, rows = rng.permutation(1 << 20)[:S], rng.integers(0, hi, cap)
    sub_indptr = np.full(S + 1, held, dtype=np.int64)
    table = capi.RelabelTable(S + cap, idt, dev, narrow=narrow)
    want, w_out = O.relabel([seeds, rows[:held]], [rows[:held]])
    for num_ids in (2 * (S + cap), 2 * (S + cap) + 1, 0):
        frontier, num, out = capi.relabel_sampled(to_dev(seeds, dev, idt), to_dev(sub_indptr, dev),
                                                  to_dev(rows, dev, idt), table, num_ids=num_ids)
        assert int(num) == want.size
        assert np.array_equal(frontier[:want.size].cpu().numpy().astype(np.int64), want)
        assert np.array_equal(out[:held].cpu().numpy().astype(np.int64), w_out[0])


@pytest.mark.parametrize("idt", [torch.int64, torch.int32])
@pytest.mark.parametrize("n", [1, 63, 1024, 1025, 2048, 2049, 4096, 4097, 8192, 8193])
def test_short_lists_by_one_workgroup_and_past_them(dev, idt, n):
    """Around the numbers of items a thread of the one-workgroup relabel takes, and its limit: all
    items distinct, hubs, all the same; four spans, two queries with ids that are not there."""
    rng = np.random.default_rng(n)
    for ids in (rng.permutation(4 * n)[:n], rng.integers(0, max(2, n // 20), n), np.full(n, 77)):
        ids = ids.astype(np.int64)
        cuts = np.sort(rng.integers(0, n + 1, 3))
        spans = np.split(ids, cuts)
        queries = [spans[3], rng.integers(0, 5 * n, 3000).astype(np.int64)]
        want_frontier, want = O.relabel(spans, queries)
        frontier, num, outs = capi.unique_relabel([to_dev(s, dev, idt) for s in spans],
                                                  [to_dev(q, dev, idt) for q in queries],
                                                  narrow=idt == torch.int64)
        assert int(num.item()) == want_frontier.size
        assert np.array_equal(frontier[:want_frontier.size].cpu().numpy().astype(np.int64), want_frontier)
        for got, w in zip(outs, want):
            assert np.array_equal(got.cpu().numpy().astype(np.int64), w)


@pytest.mark.parametrize("idt", [torch.int64, torch.int32])
@pytest.mark.parametrize("queries", [1, 4095, 4096, 4097, 10240, 10241, 24577])
def test_look_ups_of_one_workgroup_and_past_them(dev, idt, queries):
    """Four look-ups of a thread at a time, up to 10240 by the one-workgroup relabel, from two spans
    that meet anywhere."""
    rng = np.random.default_rng(queries)
    for n in (5, 8192):
        ids = rng.integers(0, 3 * n, n).astype(np.int64)
        spans = np.split(rng.integers(0, 4 * n, queries).astype(np.int64), [queries // 3])
        want_frontier, want = O.relabel([ids], spans)
        frontier, num, outs = capi.unique_relabel([to_dev(ids, dev, idt)], [to_dev(q, dev, idt) for q in spans],
                                                  narrow=idt == torch.int64)
        assert int(num.item()) == want_frontier.size
        for got, w in zip(outs, want):
            assert np.array_equal(got.cpu().numpy().astype(np.int64), w)


def test_short_list_with_an_id_beyond_32_bits(dev):
    ids = torch.tensor([3, 1, 3, (1 << 40) + 1], dtype=torch.int64, device=dev)
    assert int(capi.unique_relabel([ids], [ids], narrow=True)[1].item()) == -2
    # as a query it is an id that is not there, whatever its lower half says
    frontier, num, (out,) = capi.unique_relabel([ids[:3].contiguous()], [ids], narrow=True)
    assert int(num.item()) == 2 and out.tolist() == [0, 1, 0, -1]
    assert capi.unique_relabel([ids], [ids])[2][0].tolist() == [0, 1, 0, 2]


@pytest.mark.parametrize("idt", [torch.int64, torch.int32])
@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("S,n,queries", [(1, 1, 1), (300, 5000, 700), (4000, 4192, 10_240), (4000, 4193, 20), (4000, 4192, 10_241),
                                         (5000, 86_000, 86_000)])
def test_queries_that_hold_places(dev, idt, wide, S, n, queries):
    """The rank of mapping[span][place], by one workgroup and past it, as by a gather in front of a relabel by
    ids; repeated ids, places in the second span, and -1 for a place outside its span."""
    rng = np.random.default_rng(S + n + queries)
    seeds, ids = rng.integers(0, 3 * S, S), rng.integers(0, 2 * n, n)
    if wide and idt == torch.int64:
        seeds[S // 2] += 1 << 40
    at, second = rng.integers(0, S, queries), rng.integers(0, n, 5)
    off = at.copy()
    off[:: 7] = np.where(off[:: 7] % 2, -1 - off[:: 7], S + off[:: 7])
    m = [to_dev(seeds, dev, idt), to_dev(ids, dev, idt)]
    frontier, num, outs = capi.unique_relabel(m, [to_dev(off, dev, idt), m[1], to_dev(second, dev, idt), to_dev(seeds[at[:9]], dev, idt)],
                                              places=[0, -1, 1, -1], narrow=idt == torch.int64 and not wide)
    w_frontier, w_outs = O.relabel([seeds, ids], [seeds[at], ids, ids[second], seeds[at[:9]]])
    w_outs[0] = np.where(off == at, w_outs[0], -1)
    U = int(num.item())
    assert np.array_equal(frontier[:U].cpu().numpy().astype(np.int64), w_frontier)
    for got, want in zip(outs, w_outs):
        assert np.array_equal(got.cpu().numpy().astype(np.int64), want)
