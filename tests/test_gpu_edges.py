"""The last hop's edge list written by the launch that gathers the feature rows (or by its own, where there is
no such launch): every kind of gather behind it, against the CPU oracle."""
import numpy as np
import pytest
import torch

from helpers import load_pkg, powerlaw_graph

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def pkg():
    return load_pkg()


@pytest.mark.parametrize("replace", [False, True])
@pytest.mark.parametrize("n_seeds,fanouts,dim,dtype,hbm", [
    (3000, [7, 4], 100, torch.float32, 1.0),      # one launch
    (3000, [7, 4], 100, torch.float32, 0.5),      # ... over both tiers
    (3000, [7, 4], 301, torch.bfloat16, 1.0),     # rows that 16 bytes do not divide: a list of its own
    (300, [5, 4], 140_000, torch.float32, 1.0),   # rows beyond the flat gather
    (9000, [20, 9, 3], 8, torch.float32, 1.0),    # a worst case beyond the blocks that write the list
    (3000, [0, 4], 100, torch.float32, 1.0),      # a last hop without edges
    (2000, [9], 100, torch.float32, 1.0),         # one hop: nothing is left to the gather
])
def test_edge_list_in_the_gathers_launch(pkg, oracle, n_seeds, fanouts, dim, dtype, hbm, replace):
    rng = np.random.default_rng(11)
    n = 400 if dim > 1000 else 20_000
    indptr, indices = powerlaw_graph(rng, n, 12, 300)
    ip = pkg.create_chunktensor(torch.from_numpy(indptr), 1, 1 << 40)
    ix = pkg.create_chunktensor(torch.from_numpy(indices), 1, 1 << 40)
    x = torch.from_numpy(rng.standard_normal((n, dim)).astype(np.float32)).to(dtype)
    feats = pkg.create_chunktensor(x, 1, int(n * hbm) * dim * x.element_size())
    seeds = rng.integers(0, n, size=n_seeds).astype(indices.dtype)
    sampler = pkg.ChunkTensorSampler(fanouts, ip, ix, replace=replace)
    want_f, _, want = oracle.sample_blocks(seeds, indptr, indices, fanouts, replace, 31, 4)
    for _ in range(2):
        pkg.set_rng_state(31, 4)
        f, _, blocks, rows = sampler.sample_blocks_and_index(None, torch.from_numpy(seeds), feats)
        assert np.array_equal(f.cpu().numpy(), want_f)
        for g, w in zip(blocks, want):
            assert np.array_equal(g.src_local.cpu().numpy(), w[0]) and np.array_equal(g.dst_local.cpu().numpy(), w[1])
        assert torch.equal(rows.cpu(), x[torch.from_numpy(want_f.astype(np.int64))])


@pytest.mark.parametrize("n_seeds,fanouts,dim,cap", [
    (3000, [7, 4], 0, 0),        # no features: a list of its own, by a block for every tile
    (3000, [7, 4], 0, 3),        # ... by blocks that loop
    (3000, [7, 4], 301, 0),      # in front of a gather of odd-width rows
    (3000, [7, 4], 301, 1),
    (40_000, [40, 49], 0, 0),    # more tiles than a launch has blocks
])
def test_edge_list_in_a_launch_of_its_own(pkg, oracle, n_seeds, fanouts, dim, cap):
    rng = np.random.default_rng(12)
    n = 20_000
    indptr, indices = powerlaw_graph(rng, n, 12, 300)
    ip = pkg.create_chunktensor(torch.from_numpy(indptr), 1, 1 << 40)
    ix = pkg.create_chunktensor(torch.from_numpy(indices), 1, 1 << 40)
    seeds = rng.integers(0, n, size=n_seeds).astype(indices.dtype)
    sampler = pkg.ChunkTensorSampler(fanouts, ip, ix)
    want_f, _, want = oracle.sample_blocks(seeds, indptr, indices, fanouts, False, 31, 4)
    capi = pkg.capi
    capi.check(capi.lib.dgs_debug_set(capi.DEBUG_SAMPLER_GRID_CAP, cap))
    try:
        pkg.set_rng_state(31, 4)
        if dim:
            x = torch.from_numpy(rng.standard_normal((n, dim)).astype(np.float32)).to(torch.bfloat16)
            f, _, blocks, rows = sampler.sample_blocks_and_index(None, torch.from_numpy(seeds), pkg.create_chunktensor(x, 1, 1 << 40))
            assert torch.equal(rows.cpu(), x[torch.from_numpy(want_f.astype(np.int64))])
        else:
            f, _, blocks = sampler.sample_blocks(None, torch.from_numpy(seeds))
        assert np.array_equal(f.cpu().numpy(), want_f)
        for g, w in zip(blocks, want):
            assert np.array_equal(g.src_local.cpu().numpy(), w[0]) and np.array_equal(g.dst_local.cpu().numpy(), w[1])
    finally:
        capi.check(capi.lib.dgs_debug_set(capi.DEBUG_SAMPLER_GRID_CAP, 0))
