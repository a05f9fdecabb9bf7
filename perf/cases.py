"""What a program that samples neighbourhoods with this package asks of it, as measurable cases.

Every case runs one pass through the package's public entry points on inputs that such a program
holds beforehand (a CSC graph and a feature matrix in ChunkTensors, a sampler, seed ids).  Kinds:

  step     ChunkTensorSampler.sample_blocks_and_index: one batch, sampled, relabelled and gathered
  loader   SeedLoader: a short epoch of batches, several of them on the GPU at a time
  per_hop  one sampling operator and one relabel operator per hop, then _CAPI_index: the loop of a
           program written against the operators (and of any sampler with a fanout above 64)
  gather   ChunkTensor._CAPI_index alone: features for a list of node ids

Graphs: "powerlaw" (Pareto in-degrees, sources uniform) and "rmat" (hubs are sources of a large
share of the edges, many rows are empty).  Results are node ids, ranks and copied feature rows,
so they are compared exactly.
"""
import importlib
import math

import numpy as np
import torch

_DTYPES = {"float32": torch.float32, "bfloat16": torch.bfloat16, "float16": torch.float16}
_EVERYTHING = 1 << 62       # a capacity that keeps a whole store in HBM
_DEGREE_ONE = 0.05          # share of the power-law rows that have a single neighbour
_RMAT = (0.57, 0.19, 0.19, 0.05)

_BASE = dict(kind="step", graph="powerlaw", nodes=2_449_029, edges=123_718_280, max_deg=17_000, id_bits=64, dim=100,
             dtype="float32", hbm=1.0, batch=1024, fanouts="15,10,5", replace=False, weighted=False, batches=1, rows=0)


def _case(name, **changes):
    return dict(_BASE, name=name, **changes)


def listed():
    big = dict(nodes=111_059_956, edges=1_615_685_872, max_deg=30_000, id_bits=32, dim=128, dtype="bfloat16")
    return [
        # a service that answers for a handful of nodes at a time: nothing but latency
        _case("query", nodes=100_000, edges=2_000_000, max_deg=5_000, batch=16, fanouts="10,5"),
        # the smallest training configuration: a two-layer model on a 10 k-node graph
        _case("small_step", nodes=10_000, edges=200_000, max_deg=1_000, dim=128, fanouts="10,5"),
        # the headline training configuration, one batch at a time (a loop without prefetching)
        _case("train_step"),
        # the same batches through the loader that a training loop iterates
        _case("train_loader", kind="loader", batches=8),
        # the same batch through the operators, hop by hop (a harness that is used as it is)
        _case("per_hop_step", kind="per_hop"),
        # importance sampling: a float32 weight per edge, without and with replacement
        _case("weighted_step", weighted=True),
        _case("weighted_replace_step", weighted=True, replace=True, id_bits=32, batch=512),
        # a graph of 10^8 nodes with bf16 features, all in HBM; larger batches from a training subset
        _case("large_graph_step", **big, batch=4096),
        # draws with replacement on a graph whose hubs come up again and again, two wide hops
        _case("rmat_replace_step", graph="rmat", nodes=1 << 26, edges=1 << 30, id_bits=32, dim=64, batch=16384,
              fanouts="50,50", replace=True),
        # features that exceed the HBM share given to them: 40 % of the rows there, the rest in host memory
        _case("two_tier_step", nodes=8_000_000, edges=120_000_000, id_bits=32, dim=256, hbm=0.4),
        # evaluation with (nearly) whole neighbourhoods: fanouts that only the per-hop operators take
        _case("wide_fanout_step", kind="per_hop", id_bits=32, fanouts="100,50", batch=512),
        # features for a list of nodes (layer-wise inference), half precision, a width that is no
        # multiple of anything
        _case("gather_odd", kind="gather", id_bits=32, dim=301, dtype="bfloat16", rows=500_000),
    ]


def draw(rng):
    """A case of the same kinds, over the ranges between the listed ones."""
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    while True:
        kind = rng.choice(["step", "step", "step", "loader", "per_hop", "gather"])
        c = dict(_BASE, kind=kind)
        c["nodes"] = log_int(10_000, 20_000_000)
        c["edges"] = c["nodes"] * rng.randint(5, 50) + rng.randint(0, 999)
        c["max_deg"] = rng.choice([1_000, 5_000, 17_000])
        c["id_bits"] = rng.choice([32, 64])
        c["dim"] = log_int(16, 512)
        c["dtype"] = rng.choice(["float32", "float32", "bfloat16", "float16"])
        if kind == "gather":
            c["rows"] = log_int(500, 2_000_000)
        else:
            c["batch"] = log_int(32, 8192)
            hops = rng.randint(1, 3)
            widest = 256 if kind == "per_hop" and rng.random() < 0.5 else 25
            c["fanouts"] = ",".join(str(log_int(3, widest)) for _ in range(hops))
            c["replace"] = rng.random() < 0.3
            c["weighted"] = rng.random() < 0.3 and widest <= 64
            if kind == "loader":
                c["batches"] = rng.randint(4, 8)
        if rng.random() < 0.15:
            c["hbm"] = round(rng.uniform(0.3, 0.9), 2)
        rows = _rows_gathered(c) * c["batches"]
        row_bytes = c["dim"] * _DTYPES[c["dtype"]].itemsize
        edges = sum(_hops(c)[1]) * c["batches"] if kind != "gather" else 0
        # no dearer than the largest listed cases, and a state that is quick to make
        if (c["nodes"] * row_bytes <= 4e9 and c["edges"] <= 400_000_000 and edges <= 4_000_000 and
                rows * row_bytes <= 3e9 and rows * row_bytes * (1.0 - c["hbm"]) <= 3e8):
            return c


# ---- expected sizes (for work() and draw()): closed forms, nothing is run ---------------------

def _fanouts(case):
    """In the order the hops run (the reverse of the sampler's argument)."""
    return [int(f) for f in reversed(case["fanouts"].split(","))]


def _degrees(case):
    """The power-law degrees at evenly spaced quantiles, and the scale that gives the mean degree."""
    q = (np.arange(1 << 14) + 0.5) / (1 << 14)
    raw = (1.0 - q) ** (-1.0 / 1.25)
    want = (case["edges"] / case["nodes"] - _DEGREE_ONE) / (1.0 - _DEGREE_ONE)
    lo, hi = 0.0, 1e5
    for _ in range(60):
        mid = 0.5 * (lo + hi)
        lo, hi = (mid, hi) if np.clip(np.floor(raw * mid), 2, case["max_deg"]).mean() < want else (lo, mid)
    return np.clip(np.floor(raw * lo), 2, case["max_deg"]), lo


def _distinct(deg, k):
    """Expected number of different edges among k draws with replacement from a row."""
    return deg * (1.0 - (1.0 - 1.0 / np.maximum(deg, 1.0 + 1e-9)) ** k)


def _hops(case):
    """Expected (seeds of every hop and the last frontier, edges of every hop, weights read)."""
    seeds, edges, weights = [], [], 0.0
    if case["graph"] == "rmat":  # nodes in classes by the number of ones in their id: all of a class are alike
        bits = case["nodes"].bit_length() - 1
        a, b, c, d = _RMAT
        ones = np.arange(bits + 1)
        size = np.array([math.comb(bits, j) for j in ones], dtype=np.float64)
        mean = case["edges"] * (b + d) ** ones * (a + c) ** (bits - ones)
        has_edges = -np.expm1(-mean)
        deg = mean / has_edges  # of the rows that have any
        front = size * (1.0 - np.exp(-case["batch"] / case["nodes"]))
        for k in _fanouts(case):
            seeds.append(front.sum())
            edges.append((front * has_edges * k).sum())
            picks = front * has_edges * _distinct(deg, k)
            one = (ones * d / (b + d) + (bits - ones) * c / (a + c)) / bits  # share of ones among a pick's bits
            for j, m in zip(ones, picks):
                p = one[j] ** ones * (1.0 - one[j]) ** (bits - ones)
                front = front + (size - front) * (1.0 - np.exp(-m * p))
        return seeds + [front.sum()], edges, weights
    n = case["nodes"]
    deg, _ = _degrees(case)

    def mean(of_row):  # over the rows: the ones of a single neighbour among them
        return of_row(deg).mean() * (1 - _DEGREE_ONE) + float(of_row(np.ones(1))[0]) * _DEGREE_ONE

    def unseen(fanouts):  # of every row's edges, the share that no draw so far has picked
        return lambda d: np.prod([(1.0 - 1.0 / d) ** k if case["replace"] else 1.0 - np.minimum(k / d, 1.0) for k in fanouts], axis=0)

    front = n * -math.expm1(-case["batch"] / n)
    ages = [front]  # the frontier by the hop that found its nodes: the rows of older ones are drawn from again
    fanouts = _fanouts(case)
    for h, k in enumerate(fanouts):
        s = case["batch"] if h == 0 else front
        seeds.append(s)
        edges.append(s * (k if case["replace"] else mean(lambda d: np.minimum(d, k))))
        if case["weighted"]:
            weights += s * mean(lambda d: d if case["replace"] else np.where(d > k, d, 0.0))
        fresh = sum(rows * mean(lambda d: d * (unseen(fanouts[a:h])(d) - unseen(fanouts[a:h + 1])(d)))
                    for a, rows in enumerate(ages))
        found = (n - front) * -math.expm1(-fresh / n)
        ages.append(found)
        front += found
    return seeds + [front], edges, weights


def _rows_gathered(case):
    return case["rows"] if case["kind"] == "gather" else _hops(case)[0][-1]


def work(case):
    """Bytes of one pass: every input element that the result depends on read once, every output
    element written once.  There is no arithmetic to speak of: no contraction anywhere."""
    w = case["id_bits"] // 8
    rows = _rows_gathered(case)
    row_bytes = case["dim"] * _DTYPES[case["dtype"]].itemsize
    total = rows * (2 * row_bytes + w)
    if case["kind"] != "gather":
        seeds, edges, weights = _hops(case)
        # seed ids and their pair of offsets; picked ids; local source and destination of every edge
        total += sum(seeds[:-1]) * (w + 16) + sum(edges) * 3 * w + 4 * weights
    return {"bytes": float(total * case["batches"]), "flops": 0.0}


def tolerance(case):
    """Ids, ranks and copied rows: whole numbers and bytes."""
    return "exact"


# ---- inputs -----------------------------------------------------------------------------------

def _powerlaw_csc(case, gen):
    n = case["nodes"]
    _, scale = _degrees(case)
    raw = (1.0 - torch.rand(n, generator=gen, device="cuda", dtype=torch.float64)).pow_(-1.0 / 1.25)
    deg = raw.mul_(scale).floor_().clamp_(2, case["max_deg"]).long()
    deg[torch.rand(n, generator=gen, device="cuda") < _DEGREE_ONE] = 1
    indptr = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    torch.cumsum(deg, 0, out=indptr[1:])
    return indptr


def _rmat_indptr(case, gen):
    n, e = case["nodes"], case["edges"]
    bits = n.bit_length() - 1
    a, b, c, d = _RMAT
    ids = torch.arange(n, device="cuda", dtype=torch.int32)
    ones = torch.zeros(n, device="cuda", dtype=torch.float32)
    for bit in range(bits):
        ones += (ids >> bit) & 1
    deg = torch.poisson(torch.exp(ones * math.log(b + d) + (bits - ones) * math.log(a + c) + math.log(e)), generator=gen).long()
    indptr = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    torch.cumsum(deg, 0, out=indptr[1:])
    return indptr


def _fill_rmat_sources(out, indptr, gen):
    """Every bit of an edge's source given the same bit of its destination (the edge's row)."""
    a, b, c, d = _RMAT
    bits = (indptr.numel() - 1).bit_length() - 1
    deg = indptr[1:] - indptr[:-1]
    step = 1 << 26
    for lo in range(0, out.numel(), step):
        hi = min(out.numel(), lo + step)
        first = int(torch.searchsorted(indptr, lo, right=True)) - 1
        last = int(torch.searchsorted(indptr, hi - 1, right=True)) - 1
        count = deg[first:last + 1].clone()
        count[0] -= lo - int(indptr[first])
        count[-1] -= int(indptr[last + 1]) - hi
        row = torch.repeat_interleave(torch.arange(first, last + 1, device="cuda", dtype=torch.int32), count, output_size=hi - lo)
        src = torch.zeros(hi - lo, dtype=torch.int32, device="cuda")
        for bit in range(0, bits, 2):  # two bits from the halves of one random word
            word = torch.randint(-1 << 31, 1 << 31, (hi - lo,), generator=gen, device="cuda", dtype=torch.int32)
            for b2, value in ((bit, word & 0xffff), (bit + 1, (word >> 16) & 0xffff)):
                if b2 < bits:
                    bar = torch.where(((row >> b2) & 1) == 1, int(65536 * d / (b + d)), int(65536 * c / (a + c)))
                    src |= (value < bar).int() << b2
        out[lo:hi] = src


def _features(dgs, case, gen):
    n, dim = case["nodes"], case["dim"]
    dtype = _DTYPES[case["dtype"]]
    feats = dgs.ChunkTensor([n, dim], dtype, int(n * case["hbm"]) * dim * dtype.itemsize if case["hbm"] < 1.0 else _EVERYTHING)
    dev, host = feats._CAPI_get_sub_device_tensor(), feats._CAPI_get_host_tensor()
    chunk = 1 << 28
    for a in range(0, dev.numel(), chunk):
        dev[a:a + chunk].normal_(generator=gen)
    stage = torch.empty(min(chunk, host.numel()), device="cuda", dtype=dtype)
    for a in range(0, host.numel(), chunk):
        part = stage[:min(chunk, host.numel() - a)].normal_(generator=gen)
        host[a:a + part.numel()].copy_(part)
    return feats


def prepare(case, seed):
    dgs = importlib.import_module("dist-gpu-sampling_amd")
    gen = torch.Generator(device="cuda").manual_seed(seed)
    ids = torch.int64 if case["id_bits"] == 64 else torch.int32
    state = {"dgs": dgs, "case": case, "seed": seed, "feats": _features(dgs, case, gen)}
    if case["kind"] == "gather":
        state["ids"] = torch.randint(0, case["nodes"], (case["rows"],), generator=gen, device="cuda", dtype=ids)
        return state
    rmat = case["graph"] == "rmat"
    indptr = _rmat_indptr(case, gen) if rmat else _powerlaw_csc(case, gen)
    edges = int(indptr[-1])
    ct_indptr = dgs.ChunkTensor([case["nodes"] + 1], torch.int64, _EVERYTHING)
    ct_indptr._CAPI_get_sub_device_tensor().copy_(indptr)
    ct_indices = dgs.ChunkTensor([edges], ids, _EVERYTHING)
    indices = ct_indices._CAPI_get_sub_device_tensor()
    if rmat:
        _fill_rmat_sources(indices, indptr, gen)
    else:
        for a in range(0, edges, 1 << 28):
            part = indices[a:a + (1 << 28)]
            part.random_(0, case["nodes"], generator=gen)
    ct_weights = None
    if case["weighted"]:
        ct_weights = dgs.ChunkTensor([edges], torch.float32, _EVERYTHING)
        ct_weights._CAPI_get_sub_device_tensor().uniform_(0.01, 1.01, generator=gen)
    fanouts = [int(f) for f in case["fanouts"].split(",")]
    state["sampler"] = dgs.ChunkTensorSampler(fanouts, ct_indptr, ct_indices, ct_weights, replace=case["replace"],
                                              fused=case["kind"] != "per_hop")
    seeds = torch.randint(0, case["nodes"], (case["batch"] * case["batches"],), generator=gen, device="cuda", dtype=ids)
    if case["kind"] == "loader":  # the loader is given node ids in host memory, as a training set is held
        state["loader"] = dgs.SeedLoader(None, seeds.cpu(), state["sampler"], batch_size=case["batch"],
                                         chunk_features=state["feats"])
    state["seeds"] = seeds
    frontiers, edges, _ = _hops(case)
    state["rows"] = _window_rows(frontiers[-1]), [_window_rows(m) for m in reversed(edges)]
    torch.cuda.synchronize()
    return state


# ---- one pass ---------------------------------------------------------------------------------

def _window_rows(expected):
    return max(1, int(0.7 * expected))


def _windows(t, rows):
    """Two windows of one length over the first dimension of a result whose length depends on what
    was drawn: a view of its first and of its last `rows` rows that together cover all of it, of the
    same shape for every input of a case.  `rows` is 0.7 of the expected length."""
    n = t.shape[0]
    if not rows <= n <= 2 * rows:
        raise RuntimeError(f"a result of {n} rows where about {rows / 0.7:.0f} were expected")
    if t.dim() == 1:
        return t.as_strided((2, rows), (n - rows, 1))
    width = t.shape[1]
    return t.as_strided((2, rows, width), ((n - rows) * width, width, 1))


def _outputs(batch, rows):
    frontier_rows, edge_rows = rows
    input_nodes, _, blocks, x = batch
    out = [_windows(input_nodes, frontier_rows), _windows(x, frontier_rows)]
    for b, m in zip(blocks, edge_rows):  # the inner frontiers are prefixes of input_nodes
        out += (_windows(b.src_local, m), _windows(b.dst_local, m))
    return out


def run(state):
    kind, feats = state["case"]["kind"], state["feats"]
    if kind == "gather":
        return feats._CAPI_index(state["ids"])
    state["dgs"].set_rng_state(state["seed"], 0)  # a pass can be repeated: it draws from the same streams
    if kind == "loader":
        return [_outputs(batch, state["rows"]) for batch in state["loader"]]
    return _outputs(state["sampler"].sample_blocks_and_index(None, state["seeds"], feats), state["rows"])
