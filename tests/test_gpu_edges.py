"""The last hop's edge list written by the launch that gathers the feature rows (or by its own, where there is
no such launch): every kind of gather behind it, against the CPU oracle."""
import ctypes

import numpy as np
import pytest
import torch

from helpers import LAST_HOP_MODES, load_pkg, powerlaw_graph, set_last_hop_mode

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


@pytest.mark.parametrize("last_hop", [LAST_HOP_MODES[0], LAST_HOP_MODES[1], LAST_HOP_MODES[4]])
@pytest.mark.parametrize("n_seeds,fanouts,replace", [
    (33_000, [33, 1], False),    # a fill that loops, a compact launch that does not (hop 0's list, through the table)
    (33_000, [33, 1], True),
    (4096, [15, 10, 5], False),  # both loop (a later hop's list)
    (9000, [64, 3, 4], True),    # ... and the hop may outgrow the bucketed pass
    (300_000, [4, 1], True),     # ... with tiles of 4096 positions
])
def test_edge_list_in_the_compact_launch(pkg, oracle, last_hop, n_seeds, fanouts, replace):
    rng = np.random.default_rng(n_seeds)
    n = 300_000
    indptr, indices = powerlaw_graph(rng, n, 12, 300, id_dtype=np.int32)
    ip = pkg.create_chunktensor(torch.from_numpy(indptr), 1, 1 << 40)
    ix = pkg.create_chunktensor(torch.from_numpy(indices), 1, 1 << 40)
    seeds = rng.integers(0, n, size=n_seeds).astype(indices.dtype)
    want_f, _, want = oracle.sample_blocks(seeds, indptr, indices, fanouts, replace, 8, 1)
    try:
        set_last_hop_mode(pkg, last_hop)
        for _ in range(2):  # (the second one finds the node table used)
            pkg.set_rng_state(8, 1)
            f, _, blocks = pkg.ChunkTensorSampler(fanouts, ip, ix, replace=replace).sample_blocks(None, torch.from_numpy(seeds))
            assert np.array_equal(f.cpu().numpy(), want_f)
            for g, w in zip(blocks, want):
                assert np.array_equal(g.src_local.cpu().numpy(), w[0]) and np.array_equal(g.dst_local.cpu().numpy(), w[1])
    finally:
        set_last_hop_mode(pkg, LAST_HOP_MODES[0])


@pytest.fixture(scope="module")
def batch(pkg, oracle):
    """What a caller of the C ABI holds, and what dgs_sample_blocks_leave_edges has to come to."""
    capi = pkg.capi
    rng = np.random.default_rng(13)
    n, fan = 5000, [4, 7]  # in the order of the hops
    indptr, indices = powerlaw_graph(rng, n, 12, 300, id_dtype=np.int32)
    probs = (rng.random(indices.size) + 0.01).astype(np.float32)
    seeds = rng.integers(0, n, size=700).astype(np.int32)
    x = torch.from_numpy(rng.standard_normal((n, 20)).astype(np.float32)).cuda()
    dev = [torch.from_numpy(a).cuda() for a in (seeds, indptr, indices, probs)]
    want = {w: oracle.sample_blocks(seeds, indptr, indices, fan[::-1], False, 5, 2, probs=probs if w else None) for w in (False, True)}

    def leave(weighted):
        lib, k = capi.lib, (capi.c_i64 * 2)(*fan)
        smax, emax = (capi.c_i64 * 3)(), (capi.c_i64 * 2)()
        capi.check(lib.dgs_sample_blocks_plan(len(seeds), k, 2, smax, emax))
        ws_of = lib.dgs_sample_blocks_weighted_workspace_bytes if weighted else lib.dgs_sample_blocks_workspace_bytes
        nb = ws_of(len(seeds), k, 2, 4)
        b = {"frontier": torch.full((smax[2],), -1, dtype=torch.int32, device="cuda"),
             "src": [torch.full((e,), -1, dtype=torch.int32, device="cuda") for e in emax],
             "dst": [torch.full((e,), -1, dtype=torch.int32, device="cuda") for e in emax],
             "sizes": torch.zeros(7, dtype=torch.int64, device="cuda"), "ws": torch.empty(nb, dtype=torch.uint8, device="cuda"),
             "left": capi.EdgeJob(), "max": smax[2], "want": want[weighted]}
        outs = (capi.BlockOut * 2)(*[capi.BlockOut(s.data_ptr(), d.data_ptr()) for s, d in zip(b["src"], b["dst"])])
        pv = capi.tensor_view(dev[3])
        capi.check(lib.dgs_sample_blocks_leave_edges(
            dev[0].data_ptr(), 4, len(seeds), capi.tensor_view(dev[1]), capi.tensor_view(dev[2]), ctypes.byref(pv) if weighted else None,
            k, 2, 0, 5, 2, None, 0, b["frontier"].data_ptr(), outs, b["sizes"].data_ptr(), None, ctypes.byref(b["left"]),
            b["ws"].data_ptr(), nb, capi.stream_ptr()))
        return b

    def check(b):
        f, _, blocks = b["want"]
        assert np.array_equal(b["frontier"][:f.size].cpu().numpy(), f)
        for h, w in enumerate(reversed(blocks)):
            assert np.array_equal(b["src"][h][:w[0].size].cpu().numpy(), w[0]) and np.array_equal(b["dst"][h][:w[1].size].cpu().numpy(), w[1])
            assert (b["src"][h][w[0].size:] == -1).all()
    return capi, x, leave, check


@pytest.mark.parametrize("weighted", [False, True])
def test_edges_left_and_written(batch, weighted):
    capi, _, leave, check = batch
    b = leave(weighted)
    assert (b["src"][1] == -1).all()  # the last list is left; the first one is there
    capi.check(capi.lib.dgs_write_edges(ctypes.byref(b["left"]), capi.stream_ptr()))
    check(b)


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("index_bytes,n_max,blocks_per_cu,elems,tier", [
    (4, None, 0, 20, 0),   # in the gather's launch
    (4, None, 4, 20, 0),   # ... which leaves wave slots to others
    (8, None, 0, 20, 0),   # indices of another width than the ids
    (4, 0, 0, 20, 0),      # no rows to gather
    (4, None, 0, 20, 1),   # one tier
    (4, None, 0, 1, 0)])   # chunks of 1 or 2 bytes: a list of its own
def test_edges_left_to_a_gather(batch, weighted, index_bytes, n_max, blocks_per_cu, elems, tier):
    capi, x, leave, check = batch
    b = leave(weighted)
    f = torch.from_numpy(b["want"][0].astype(np.int64))
    rows = x if elems == 20 else x[:, 0].to(torch.uint8).contiguous()
    index = b["frontier"] if index_bytes == 4 else torch.cat([f, f.new_zeros(b["max"] - f.numel())]).cuda()
    out = torch.zeros((b["max"], elems), dtype=rows.dtype, device="cuda")
    bad = torch.zeros(1, dtype=torch.int64, device="cuda")
    capi.check(capi.lib.dgs_gather_rows_dyn_edges(capi.tensor_view(rows), elems, index.data_ptr(), index_bytes,
                                                  b["max"] if n_max is None else n_max, b["sizes"][2:].data_ptr(), 1000, out.data_ptr(), tier,
                                                  blocks_per_cu, bad.data_ptr(), ctypes.byref(b["left"]), capi.stream_ptr()))
    check(b)
    assert bad.item() == 0
    want = rows[f.cuda()].view(-1, elems) if n_max is None else out[:0]
    assert torch.equal(out[:want.shape[0]], want) and (out[want.shape[0]:] == 0).all()


def test_edge_jobs_that_are_empty_or_refused(batch):
    capi, x, leave, check = batch
    lib, st = capi.lib, capi.stream_ptr()
    n = torch.tensor([3], dtype=torch.int64, device="cuda")
    index = torch.tensor([4, 0, 2], dtype=torch.int32, device="cuda")
    out = torch.zeros((3, 20), device="cuda")
    args = (capi.tensor_view(x), 20, index.data_ptr(), 4, 3, n.data_ptr(), 3, out.data_ptr())
    empty = capi.EdgeJob()
    capi.check(lib.dgs_gather_rows_dyn_edges(*args, 0, 0, None, ctypes.byref(empty), st))
    assert torch.equal(out, x[index.long()])
    capi.check(lib.dgs_write_edges(ctypes.byref(empty), st))
    b = leave(False)
    left = ctypes.byref(b["left"])
    assert lib.dgs_write_edges(None, st) == capi.DGS_ERR_INVALID
    assert lib.dgs_gather_rows_dyn_edges(*args, 0, 0, None, None, st) == capi.DGS_ERR_INVALID
    assert lib.dgs_gather_rows_dyn_edges(*args, 0, -1, None, left, st) == capi.DGS_ERR_INVALID
    assert lib.dgs_gather_rows_dyn_edges(*args, 7, 0, None, left, st) == capi.DGS_ERR_INVALID
    assert lib.dgs_gather_rows_dyn_edges(*args[:5], None, *args[6:], 0, 0, None, left, st) == capi.DGS_ERR_INVALID
    capi.check(lib.dgs_write_edges(left, st))  # (what was refused has used nothing up)
    check(b)
