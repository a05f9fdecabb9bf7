"""GPU parity of the block-wise weighted choice (csrc/choose.h) at the edges of its row classes, against the
CPU oracle: picks are bit-exact whatever the float32 race decides and whatever it leaves to 64-bit keys."""
import numpy as np
import pytest
import torch

from helpers import load_pkg

pytestmark = pytest.mark.gpu

# quads, the counting limit, stretches of a wave, the limits of block turns and queues, more than one go
EDGES = [0, 1, 2, 3, 4, 5, 7, 8, 9, 31, 32, 33, 63, 64, 65, 127, 128, 129, 130, 255, 256, 257, 511, 512, 513, 1023, 1024,
         1025, 2047, 2048, 2049, 4095, 4096, 4097, 5121, 20480, 20481]
SEED, STREAM = 0x5eed5eed77, 3


@pytest.fixture(scope="module")
def pkg():
    return load_pkg()


def _graph(rng, n):
    deg = rng.integers(0, 40, size=n)
    deg[rng.permutation(n)[:2 * len(EDGES)]] = EDGES * 2
    indptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.int64)
    return deg, indptr, rng.integers(0, n, size=int(indptr[-1])).astype(np.int32)


def _weights(kind, rng, oracle, deg, indptr):
    w = (rng.random(int(indptr[-1])) + 0.01).astype(np.float32)
    if kind == "spread":   # hundreds of binades, denormal ones and huge ones among them, and no weight at all
        w = np.exp2(rng.uniform(-148, 126, size=w.size)).astype(np.float32)
        w[rng.random(w.size) < 0.3] = rng.choice(np.array([0, -1, np.nan], dtype=np.float32))
    if kind == "few":      # mostly unusable: they are picked in order of their positions
        w[rng.random(w.size) < 0.9] = 0.0
    if kind == "infinite":
        w[rng.random(w.size) < 0.2] = np.inf
    if kind == "level":    # every weight is its own variate: all of a row's keys are 1 to within a float32
        for row in range(len(deg)):
            for p in range(min(int(deg[row]), 1100)):
                w[indptr[row] + p] = oracle.weighted_key(SEED, STREAM, row, p, 1.0)
    return w


@pytest.mark.parametrize("replace", [False, True])
@pytest.mark.parametrize("kind", ["plain", "spread", "few", "infinite", "level"])
def test_choice_at_the_edges_of_the_row_classes(pkg, oracle, kind, replace):
    rng = np.random.default_rng(5)
    n = 600
    deg, indptr, indices = _graph(rng, n)
    probs = _weights(kind, rng, oracle, deg, indptr)
    cts = [pkg.create_chunktensor(torch.from_numpy(a), 1, 1 << 40) for a in (indptr, indices, probs)]
    for n_seeds, fanouts in [(n, [7]), (n, [33]), (n, [64]), (n, [1]), (1, [5, 3]), (300, [2, 0, 4])]:
        seeds = rng.permutation(n)[:n_seeds].astype(np.int32)
        pkg.set_rng_state(SEED, STREAM)
        f, _, blocks = pkg.ChunkTensorSampler(fanouts, *cts, replace=replace).sample_blocks(None, torch.from_numpy(seeds))
        want_f, _, want = oracle.sample_blocks(seeds, indptr, indices, fanouts, replace, SEED, STREAM, probs=probs)
        assert np.array_equal(f.cpu().numpy(), want_f), (n_seeds, fanouts)
        for g, w in zip(blocks, want):
            assert np.array_equal(g.src_local.cpu().numpy(), w[0]) and np.array_equal(g.dst_local.cpu().numpy(), w[1])


@pytest.mark.parametrize("kind", ["one", "infinite", "equal"])
@pytest.mark.parametrize("n_seeds,fanouts", [(300, [64]), (300, [5, 3]),      # long rows by blocks of 16 waves ...
                                             (12289, [64]), (12289, [5])])    # ... and of four, from the queue
def test_long_rows_that_floats_alone_do_not_settle(pkg, oracle, n_seeds, fanouts, kind):
    rng = np.random.default_rng(n_seeds)
    n = 2000
    deg = rng.integers(0, 20, size=n)
    deg[:12] = [2048, 2049, 2303, 2304, 2305, 5120, 5121, 20480, 20481, 33333, 4096, 40000]
    indptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.int64)
    indices = rng.integers(0, n, size=int(indptr[-1])).astype(np.int32)
    probs = (rng.random(indices.size) + 0.01).astype(np.float32)
    if kind == "one":         # a row's first and last weight
        probs[indptr[:-1][deg > 0]] = 1e-42
        probs[indptr[1:][deg > 0] - 1] = np.inf
    elif kind == "infinite":  # more of them than picks, in the order of their positions
        probs[rng.random(probs.size) < 0.3] = np.inf
    else:                     # keys beyond float32: 64-bit ones of whole rows
        probs[:] = rng.choice(np.array([1e-45, 3e-45, 4e-45], dtype=np.float32), size=probs.size)
    cts = [pkg.create_chunktensor(torch.from_numpy(a), 1, 1 << 40) for a in (indptr, indices, probs)]
    seeds = rng.integers(0, n, size=n_seeds).astype(np.int32)
    seeds[:24] = np.arange(24) % 12
    pkg.set_rng_state(SEED, STREAM)
    f, _, blocks = pkg.ChunkTensorSampler(fanouts, *cts, replace=False).sample_blocks(None, torch.from_numpy(seeds))
    want_f, _, want = oracle.sample_blocks(seeds, indptr, indices, fanouts, False, SEED, STREAM, probs=probs)
    assert np.array_equal(f.cpu().numpy(), want_f)
    for g, w in zip(blocks, want):
        assert np.array_equal(g.src_local.cpu().numpy(), w[0]) and np.array_equal(g.dst_local.cpu().numpy(), w[1])


@pytest.mark.parametrize("replace", [False, True])
@pytest.mark.parametrize("n_seeds,fanouts", [(14000, [5]),           # more long rows than blocks of the queue: from segments ...
                                             (1500, [4, 12]),        # ... and from the queue, 600 blocks beside it ...
                                             (5000, [3, 2, 9])])     # ... and more of them than the GPU holds
def test_frontiers_of_long_rows(pkg, oracle, n_seeds, fanouts, replace):
    rng = np.random.default_rng(n_seeds)
    n = 1600
    deg = rng.integers(2049, 2400, size=n)
    deg[::97] = [3, 0, 40, 5120, 5121, 9217, 13313, 13314, 20480, 21505, 26000, 2048, 7, 5119, 8192, 17, 30000]  # (a wave's held and read-ahead stretches end between these)
    indptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.int64)
    indices = rng.integers(0, n, size=int(indptr[-1])).astype(np.int32)
    probs = (rng.random(indices.size) + 0.01).astype(np.float32)
    cts = [pkg.create_chunktensor(torch.from_numpy(a), 1, 1 << 40) for a in (indptr, indices, probs)]
    seeds = rng.integers(0, n, size=n_seeds).astype(np.int32)
    pkg.set_rng_state(SEED, STREAM)
    f, _, blocks = pkg.ChunkTensorSampler(fanouts, *cts, replace=replace).sample_blocks(None, torch.from_numpy(seeds))
    want_f, _, want = oracle.sample_blocks(seeds, indptr, indices, fanouts, replace, SEED, STREAM, probs=probs)
    assert np.array_equal(f.cpu().numpy(), want_f)
    for g, w in zip(blocks, want):
        assert np.array_equal(g.src_local.cpu().numpy(), w[0]) and np.array_equal(g.dst_local.cpu().numpy(), w[1])


@pytest.mark.parametrize("replace", [False, True])
@pytest.mark.parametrize("n_seeds,fanouts", [(200, [6, 4, 3]),     # shared, shared, queued: long rows of every frontier
                                             (900, [6, 4]),        # shared, then queued
                                             (12289, [3, 2]),      # the first hop's long rows come from its segments
                                             (70000, [2])])        # more segments than blocks
def test_long_rows_reach_the_hop_that_has_them(pkg, oracle, n_seeds, fanouts, replace):
    rng = np.random.default_rng(n_seeds)
    n = 6000
    deg = rng.integers(0, 20, size=n)
    hubs = rng.permutation(n)[:40]
    deg[hubs] = rng.integers(2040, 2600, size=40)
    indptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.int64)
    indices = rng.integers(0, n, size=int(indptr[-1])).astype(np.int32)
    indices[rng.random(indices.size) < 0.02] = hubs[0]
    probs = (rng.random(indices.size) + 0.01).astype(np.float32)
    cts = [pkg.create_chunktensor(torch.from_numpy(a), 1, 1 << 40) for a in (indptr, indices, probs)]
    seeds = rng.integers(0, n, size=n_seeds).astype(np.int32)
    seeds[:40] = hubs
    for _ in range(2):  # (the second call works on what the first one left in the buffers)
        pkg.set_rng_state(SEED, STREAM)
        f, _, blocks = pkg.ChunkTensorSampler(fanouts, *cts, replace=replace).sample_blocks(None, torch.from_numpy(seeds))
    want_f, _, want = oracle.sample_blocks(seeds, indptr, indices, fanouts, replace, SEED, STREAM, probs=probs)
    assert np.array_equal(f.cpu().numpy(), want_f)
    for g, w in zip(blocks, want):
        assert np.array_equal(g.src_local.cpu().numpy(), w[0]) and np.array_equal(g.dst_local.cpu().numpy(), w[1])


@pytest.mark.parametrize("n_seeds", [40, 12289])   # a wave for each row; rows shared by a block
@pytest.mark.parametrize("k", [1, 63, 64])         # (with 64 picks the first lane places the seed too)
@pytest.mark.parametrize("at", [0, -1])
def test_an_id_outside_the_graph_in_any_lane_is_refused(pkg, n_seeds, k, at):
    n = 500
    indptr = np.arange(n + 1, dtype=np.int64) * k
    indices = np.random.default_rng(k).integers(0, n, size=n * k).astype(np.int64)
    cts = [pkg.create_chunktensor(torch.from_numpy(a), 1, 1 << 40) for a in (indptr, np.ones(n * k, dtype=np.float32))]
    seeds = torch.arange(n_seeds) % n
    for bad_id in (None, n, -1, 2 ** 35):
        if bad_id is not None:
            indices[indptr[10 + 1] - 1 if at else indptr[10]] = bad_id   # of node 10, whose row is copied whole
        ix = pkg.create_chunktensor(torch.from_numpy(indices), 1, 1 << 40)
        sampler = pkg.ChunkTensorSampler([k], cts[0], ix, cts[1])
        if bad_id is None:
            sampler.sample_blocks(None, seeds)
            continue
        with pytest.raises(RuntimeError, match="neighbour id"):
            sampler.sample_blocks(None, seeds)
