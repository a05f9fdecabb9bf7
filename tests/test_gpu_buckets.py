"""The bucketed pass of a last hop (csrc/buckets.h) where it can go wrong: hops that end with a tile of units and
behind it, tiles of the frontier alone, more tiles than a block reads at once, pieces longer than what it reads at
once, a single bucket; in both of its forms, against the CPU oracle."""
import numpy as np
import pytest
import torch

from helpers import LAST_HOP_MODES, load_pkg, powerlaw_graph, set_last_hop_mode

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def pkg():
    return load_pkg()


@pytest.mark.parametrize("mode", LAST_HOP_MODES[1:4])
@pytest.mark.parametrize("id_dtype", [np.int32, np.int64])
@pytest.mark.parametrize("nodes,seeds,k,replace", [
    (3000, 512, 15, False),        # 512 seeds and 7680 positions: exactly a tile
    (3000, 513, 15, True),         # the next unit begins another one
    (20_000, 9000, 1, False),      # a tile of frontier ids alone
    (20_000, 16, 64, True),        # a small hop of the widest fanout
    (90, 90, 40, True),            # 90 ids, so that a bucket's piece is far beyond 32 units
    (512 * 7, 3000, 20, False),    # ids up to a multiple of the buckets
    (400_000, 140_000, 15, False), # 274 tiles: a second round of them in the direct form, which reads 256 at once
    (600_000, 215_000, 15, False), # 420 tiles: in the hashed one as well, which reads 384
])
def test_bucketed_pass_at_its_edges(pkg, oracle, mode, id_dtype, nodes, seeds, k, replace):
    rng = np.random.default_rng(seeds + k)
    indptr, indices = powerlaw_graph(rng, nodes, 12, min(300, nodes), id_dtype=id_dtype)
    if nodes == 512 * 7:
        indices[::2] = indices[::2] // 512 * 512  # half of the edges lead to ids of one bucket
    ip = pkg.create_chunktensor(torch.from_numpy(indptr), 1, 1 << 40)
    ix = pkg.create_chunktensor(torch.from_numpy(indices), 1, 1 << 40)
    start = rng.permutation(nodes)[:seeds].astype(id_dtype)
    fanouts = [k, 0]  # hop order: nothing, then k (the pass serves the last of at least two hops)
    want_f, _, want = oracle.sample_blocks(start, indptr, indices, fanouts, replace, 9, 0)
    try:
        set_last_hop_mode(pkg, mode)
        pkg.set_rng_state(9, 0)
        f, _, blocks = pkg.ChunkTensorSampler(fanouts, ip, ix, replace=replace).sample_blocks(None, torch.from_numpy(start))
        assert np.array_equal(f.cpu().numpy(), want_f)
        for g, w in zip(blocks, want):
            assert np.array_equal(g.src_local.cpu().numpy(), w[0]) and np.array_equal(g.dst_local.cpu().numpy(), w[1])
    finally:
        set_last_hop_mode(pkg, LAST_HOP_MODES[0])


@pytest.mark.parametrize("mode", LAST_HOP_MODES[1:4])
@pytest.mark.parametrize("replace", [False, True])
@pytest.mark.parametrize("hubs,share", [(1, 0.03), (1, 0.5), (12, 0.7), (1, 1.0)])
def test_bucketed_pass_with_hubs(pkg, oracle, mode, replace, hubs, share):
    # ids that come up again and again in a tile, in rows of their own and of others, among the seeds (the even ones of them)
    # and not: the sort hands on the first of each
    rng = np.random.default_rng(hubs * 100 + int(share * 10))
    n = 50_000
    indptr, indices = powerlaw_graph(rng, n, 25, 400, id_dtype=np.int32)
    hub = rng.permutation(n)[:hubs].astype(np.int32)
    at = rng.random(indices.size) < share
    indices[at] = rng.choice(hub, size=int(at.sum()))
    start = rng.permutation(np.setdiff1d(np.arange(n, dtype=np.int32), hub[1::2]))[:4000].astype(np.int32)
    start[-len(hub[::2]):] = hub[::2]
    start = start[np.sort(np.unique(start, return_index=True)[1])]
    ip = pkg.create_chunktensor(torch.from_numpy(indptr), 1, 1 << 40)
    ix = pkg.create_chunktensor(torch.from_numpy(indices), 1, 1 << 40)
    for fanouts in ([15, 0], [12, 4]):
        want_f, _, want = oracle.sample_blocks(start, indptr, indices, fanouts, replace, 3, 0)
        try:
            set_last_hop_mode(pkg, mode)
            pkg.set_rng_state(3, 0)
            f, _, blocks = pkg.ChunkTensorSampler(fanouts, ip, ix, replace=replace).sample_blocks(None, torch.from_numpy(start))
            assert np.array_equal(f.cpu().numpy(), want_f)
            for g, w in zip(blocks, want):
                assert np.array_equal(g.src_local.cpu().numpy(), w[0]) and np.array_equal(g.dst_local.cpu().numpy(), w[1])
        finally:
            set_last_hop_mode(pkg, LAST_HOP_MODES[0])


@pytest.mark.parametrize("nodes,degree,seeds", [
    (262_144, 30, 700),  # 0.69 M picks at most, and rows that fill their positions: the pass
    (262_144, 29, 700),  # the table
    (262_143, 30, 700),  # the table
    (262_144, 12, 930),  # 0.92 M picks at most: the pass
])
def test_last_hop_by_size(pkg, oracle, nodes, degree, seeds):
    rng = np.random.default_rng(nodes + degree)
    indptr = np.arange(nodes + 1, dtype=np.int64) * degree
    indices = rng.integers(0, nodes, size=nodes * degree).astype(np.int32)
    start = rng.permutation(nodes)[:seeds].astype(np.int32)
    ip = pkg.create_chunktensor(torch.from_numpy(indptr), 1, 1 << 40)
    ix = pkg.create_chunktensor(torch.from_numpy(indices), 1, 1 << 40)
    want_f, _, want = oracle.sample_blocks(start, indptr, indices, [15, 10, 5], False, 4, 0)
    pkg.set_rng_state(4, 0)
    f, _, blocks = pkg.ChunkTensorSampler([15, 10, 5], ip, ix).sample_blocks(None, torch.from_numpy(start))
    assert np.array_equal(f.cpu().numpy(), want_f)
    for g, w in zip(blocks, want):
        assert np.array_equal(g.src_local.cpu().numpy(), w[0]) and np.array_equal(g.dst_local.cpu().numpy(), w[1])


def _dev(x):
    return torch.from_numpy(np.ascontiguousarray(x)).cuda()


def _relabel_both_ways(pkg, oracle, mapping, requiring):
    want_u, want = oracle.unique_relabel(mapping, requiring)
    held = {}  # (a tensor that is given twice is one tensor)
    dev = [[held.setdefault(id(x), _dev(x)) for x in part] for part in (mapping, requiring)]
    for u, outs in (pkg.ops._CAPI_tensor_relabel(*dev), pkg.capi.unique_relabel(*dev)):
        assert np.array_equal(u.cpu().numpy(), want_u)
        for a, b in zip(outs, want):
            assert np.array_equal(a.cpu().numpy(), b)


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
@pytest.mark.parametrize("n", [131_071, 131_072, 131_073, 139_263, 524_288, 524_289, 1_200_000])  # where buckets, a tile of 2048, tiles of 8192 begin
@pytest.mark.parametrize("distinct", [1, 3000, 1 << 30])
def test_relabel_of_long_lists(pkg, oracle, dtype, n, distinct):
    rng = np.random.default_rng(n)
    seeds = rng.integers(0, distinct, size=n // 16).astype(dtype)
    cols = rng.integers(0, distinct, size=n - seeds.size).astype(dtype)
    rows = np.repeat(seeds, 16)[:cols.size]  # runs that begin and end anywhere in a tile
    _relabel_both_ways(pkg, oracle, [seeds, cols], [rows, cols])
    # ids in no order, ids that are not there, no mapped ones, all mapped ones
    others = np.concatenate([rng.permutation(cols)[:20_000], rng.integers(0, 1 << 31, size=9000).astype(dtype), cols[:1]])
    _relabel_both_ways(pkg, oracle, [seeds, cols], [others])
    _relabel_both_ways(pkg, oracle, [cols, seeds], [cols, seeds])


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
@pytest.mark.parametrize("n,m", [(193 * 8192, 192 * 8192), (1 << 22, 1 << 22)])  # 385 tiles, one more than a round; all that there may be
def test_relabel_of_the_longest_lists(pkg, oracle, dtype, n, m):
    rng = np.random.default_rng(n)
    _relabel_both_ways(pkg, oracle, [rng.integers(0, n, size=n).astype(dtype)], [rng.integers(0, 2 * n, size=m).astype(dtype)])


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
@pytest.mark.parametrize("n", [140_000, 600_000])  # of small tiles and of large ones
@pytest.mark.parametrize("hubs,share", [(1, 0.02), (1, 0.2), (7, 0.5), (40, 0.9)])
def test_relabel_of_lists_with_hubs(pkg, oracle, dtype, n, hubs, share):
    # ids that come up again and again, mapped and looked up, in no runs; the last hub is looked up alone, so that it is not there
    rng = np.random.default_rng(n + hubs)
    hub = rng.integers(0, 1 << 30, size=hubs + 1).astype(dtype)
    ids = rng.integers(0, 1 << 30, size=n).astype(dtype)
    at = rng.random(n) < share
    ids[at] = rng.choice(hub[:-1], size=int(at.sum()))
    look = rng.permutation(ids)
    at = rng.random(n) < share
    look[at] = rng.choice(hub, size=int(at.sum()))
    look[n // 2 - 3000:n // 2] = hub[-1]
    _relabel_both_ways(pkg, oracle, [ids], [look, ids])


def test_relabel_of_hubs_that_meet_in_the_filter(pkg, oracle):
    # ids of one bucket (of 256) and of one entry of the filter (the hash's top 13 bits, by the library's hash, restated here):
    # the smallest of them that a tile holds has the entry, the others go on as they are
    ids = np.arange(1 << 25, dtype=np.uint32)
    h = ids.copy()
    h ^= h >> np.uint32(16); h *= np.uint32(0x85EBCA6B)
    h ^= h >> np.uint32(13); h *= np.uint32(0xC2B2AE35)
    h ^= h >> np.uint32(16)
    meet = ids[((h & 255) == 9) & ((h >> 19) == 77)]
    assert meet.size >= 4
    rng = np.random.default_rng(1)
    for n in (200_000, 700_000):
        mapping = rng.choice(meet, size=n)
        mapping[::5] = rng.integers(0, 1 << 30, size=mapping[::5].size)
        _relabel_both_ways(pkg, oracle, [mapping.astype(np.int64)], [rng.permutation(mapping).astype(np.int64)])


def test_relabel_of_long_lists_in_many_segments(pkg, oracle):
    rng = np.random.default_rng(5)
    sizes = [70_000, 1, 0, 8191, 8192, 8193, 60_000]
    parts = [rng.integers(0, 200_000, size=s).astype(np.int64) for s in sizes]
    _relabel_both_ways(pkg, oracle, parts, [parts[3], parts[0][:9000].copy(), parts[2], parts[6], parts[4][::-1].copy(), parts[1]])
    # more ids to look up than are mapped: the table serves them
    _relabel_both_ways(pkg, oracle, parts, [np.tile(parts[0], 3)])
    # a segment that lies where the one before it would go on, were it not for the one in between
    whole, between = _dev(parts[0]), _dev(parts[3])
    mapping = [whole[:20_000], between, whole[20_000 + between.numel():], _dev(parts[6]), _dev(parts[4])]
    host = [m.cpu().numpy() for m in mapping]
    want_u, want = oracle.unique_relabel(host, host)
    u, outs = pkg.ops._CAPI_tensor_relabel(mapping, mapping)
    assert np.array_equal(u.cpu().numpy(), want_u) and all(np.array_equal(a.cpu().numpy(), b) for a, b in zip(outs, want))


def test_relabel_of_long_lists_with_ids_beyond_32_bits(pkg, oracle):
    rng = np.random.default_rng(6)
    cols = rng.integers(0, 500_000, size=150_000).astype(np.int64)
    odd = cols[:30_000].copy()
    odd[::7] += 1 << 32   # not there, though their low halves are
    odd[1::7] = -1
    odd[5000:5100] = (1 << 32) - 1  # a run of them
    _relabel_both_ways(pkg, oracle, [cols], [odd, cols])
    cols[77_777] += 1 << 33  # among the mapped ones: the attempt is void
    _relabel_both_ways(pkg, oracle, [cols], [odd, cols])


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
def test_relabel_of_ids_that_crowd_a_bucket(pkg, oracle, dtype):
    # 40 000 ids of one bucket (of 256, by the library's hash, restated here), twice, are its table of 16 384 in 10 parts; if they
    # are of two of these as well, those go range by range
    ids = np.arange(60_000_000, dtype=np.uint32)
    h = ids.copy()
    h ^= h >> np.uint32(16); h *= np.uint32(0x85EBCA6B)
    h ^= h >> np.uint32(13); h *= np.uint32(0xC2B2AE35)
    h ^= h >> np.uint32(16)
    bucket = ids[(h & 255) == 0]
    part = ids[((h & 255) == 0) & ((h >> 23) % 5 == 0)]
    others = ids[(h & 255) == 1][:100_000]
    for crowd in (bucket[:40_000], part[:40_000]):
        assert crowd.size == 40_000
        mapping = [np.concatenate([crowd, others]).astype(dtype)]
        _relabel_both_ways(pkg, oracle, mapping, [mapping[0], crowd[::-1].astype(dtype)])


def test_draws_that_crowd_a_bucket(pkg, oracle):
    # 20 000 ids of one bucket (of 256) and of one of the 3 parts that its 22 000 units make: more than a table's 16 384 slots
    n = 1 << 24
    h = np.arange(n, dtype=np.uint32)
    h ^= h >> np.uint32(16); h *= np.uint32(0x85EBCA6B)
    h ^= h >> np.uint32(13); h *= np.uint32(0xC2B2AE35)
    h ^= h >> np.uint32(16)
    crowd = np.flatnonzero(((h & 255) == 0) & ((h >> 23) % 3 == 0))[:20_000].astype(np.int32)
    assert crowd.size == 20_000
    seeds = np.arange(2000, dtype=np.int32)
    indptr = np.minimum(np.arange(n + 1, dtype=np.int64), 2000) * 10
    ip = pkg.create_chunktensor(torch.from_numpy(indptr), 1, 1 << 40)
    ix = pkg.create_chunktensor(torch.from_numpy(crowd), 1, 1 << 40)
    want_f, _, want = oracle.sample_blocks(seeds, indptr, crowd, [10, 0], False, 2, 0)
    try:
        set_last_hop_mode(pkg, LAST_HOP_MODES[2])
        pkg.set_rng_state(2, 0)
        f, _, blocks = pkg.ChunkTensorSampler([10, 0], ip, ix).sample_blocks(None, torch.from_numpy(seeds))
        assert np.array_equal(f.cpu().numpy(), want_f)
        assert np.array_equal(blocks[0].src_local.cpu().numpy(), want[0][0])
    finally:
        set_last_hop_mode(pkg, LAST_HOP_MODES[0])
