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
    (400_000, 140_000, 15, False), # 274 tiles: a second round of them
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
