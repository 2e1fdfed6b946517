"""The triangle-counting calls whose speed is measured.

Every case is one call (or one burst of calls) through the package's public
entry points, on graphs drawn from the generators' two families -- uniform
pairs G(n, m) and R-MAT (.57, .19, .19, .05) with shuffled ids -- in the sizes
of the repository's benchmark workloads and of the requests its server takes:

  * counting one graph resident in HBM, from a thousand vertices to R-MAT
    scale 22, with sorted and unsorted lists, with and without per-vertex
    counts, under the library's default knobs and under the autotuner's table;
  * counting and orienting graphs held in host memory;
  * many graphs per call (batch) and a burst of requests (server);
  * one rank's shard: CeTriC on given inputs, DiTriC on inputs built from the
    whole resident graph;
  * caller-given sorted lists (intersection).

Outputs are whole numbers: totals, per-vertex counts, ids.
"""
import math

import numpy as np
import torch

import katric_amd as K
from katric_amd import batch as KB
from katric_amd import serve as KV
from katric_amd import shard as KS
from katric_amd import tune as KT

A, B, C = 0.57, 0.19, 0.19  # R-MAT quadrants (upper left, upper right, lower left)

# wedges up to which exact() enumerates them
EXACT_WEDGES = 3_000_000_000


def listed():
    return [
        # the smallest request a server or an interactive caller sends: launch and round-trip latency
        {"name": "count_tiny", "op": "count", "model": "rmat", "n": 1531, "pairs": 12_301, "sorted": True,
         "per_vertex": True, "tuned": False},
        # uniform graph of 2^16 vertices, 2^20 pairs: short lists, few triangles
        {"name": "count_gnm_64k", "op": "count", "model": "gnm", "n": 1 << 16, "pairs": 1 << 20, "sorted": True,
         "per_vertex": True, "tuned": True},
        # an ordinary skewed graph with a ragged vertex count, under the default knobs
        {"name": "count_rmat_300k", "op": "count", "model": "rmat", "n": 300_007, "pairs": 4_000_037, "sorted": True,
         "per_vertex": True, "tuned": False},
        # adjacency lists in arbitrary order, as a loader without a sort delivers them
        {"name": "count_unsorted", "op": "count", "model": "rmat", "n": 1 << 19, "pairs": 1 << 23, "sorted": False,
         "per_vertex": True, "tuned": False},
        # the headline workload: R-MAT scale 22, edge factor 16, under the tuned knobs
        {"name": "count_rmat_22", "op": "count", "model": "rmat", "n": 1 << 22, "pairs": 1 << 26, "sorted": True,
         "per_vertex": True, "tuned": True},
        # Context.count on numpy arrays: upload, count, download of the per-vertex counts
        {"name": "count_host", "op": "count_host", "model": "rmat", "n": 65_521, "pairs": 1 << 20, "sorted": True},
        # the oriented CSR of a host graph, for a caller that goes on with its own algorithm
        {"name": "orient_host", "op": "orient", "model": "gnm", "n": 150_001, "pairs": 1_600_007, "edges": 1_500_007,
         "sorted": True},
        # 768 mixed graphs of 64 to 65536 vertices per call, resident in HBM, under the tuned knobs
        {"name": "batch_mixed", "op": "batch", "graphs": 768, "n_min": 64, "n_max": 65_536, "deg_min": 4.0,
         "deg_max": 64.0, "tuned": True},
        # a burst of 48 requests from page-locked memory through the server, with their per-vertex counts
        {"name": "serve_burst", "op": "serve", "graphs": 48, "n_min": 1 << 10, "n_max": 1 << 15, "deg_min": 4.0,
         "deg_max": 32.0},
        # one of 16 ranks of a scale-20 graph: CeTriC local and contracted phase on inputs in HBM
        {"name": "shard_cetric", "op": "shard", "model": "rmat", "n": 1 << 20, "pairs": 1 << 24, "ranks": 16,
         "rank": 1},
        # one of 6 ranks, DiTriC, its inputs built on the device from the whole graph (odd range bounds)
        {"name": "shard_graph_ditric", "op": "shard_graph", "model": "rmat", "n": 500_009, "pairs": 8_000_009,
         "ranks": 6, "rank": 2, "ditric": True},
        # caller-given sorted lists of ragged lengths, counts and common ids
        {"name": "intersect_lists", "op": "intersect", "lists": 300, "len_min": 16, "len_max": 60_000},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["count", "count", "count", "count", "count_host", "orient", "batch", "serve", "shard",
                     "shard_graph", "intersect"])
    if op == "count":
        n = _log_uniform(rng, 700, 1 << 21)
        return {"op": op, "model": rng.choice(["rmat", "rmat", "gnm"]), "n": n,
                "pairs": int(n * rng.uniform(3.0, 16.0)), "sorted": rng.random() < 0.75,
                "per_vertex": rng.random() < 0.75, "tuned": rng.random() < 0.4}
    if op in ("count_host", "orient"):
        n = _log_uniform(rng, 2_000, 300_000)
        case = {"op": op, "model": rng.choice(["rmat", "gnm"]), "n": n, "pairs": int(n * rng.uniform(3.0, 16.0)),
                "sorted": rng.random() < 0.8}
        if op == "orient":
            case.update(model="gnm", edges=int(case["pairs"] * 0.9))
        return case
    if op == "batch":
        return {"op": op, "graphs": _log_uniform(rng, 16, 700), "n_min": 64, "n_max": _log_uniform(rng, 2_000, 65_536),
                "deg_min": 4.0, "deg_max": rng.uniform(8.0, 64.0), "tuned": rng.random() < 0.5}
    if op == "serve":
        return {"op": op, "graphs": _log_uniform(rng, 4, 64), "n_min": 1 << 10,
                "n_max": _log_uniform(rng, 1 << 11, 1 << 16), "deg_min": 4.0, "deg_max": 32.0}
    if op in ("shard", "shard_graph"):
        ranks = rng.randint(2, 16)
        n = _log_uniform(rng, 20_000, 1 << 20)
        case = {"op": op, "model": rng.choice(["rmat", "rmat", "gnm"]), "n": n,
                "pairs": int(n * rng.uniform(4.0, 16.0)), "ranks": ranks, "rank": rng.randrange(ranks)}
        if op == "shard_graph":
            case["ditric"] = rng.random() < 0.5
        return case
    return {"op": "intersect", "lists": _log_uniform(rng, 1, 600), "len_min": 2,
            "len_max": _log_uniform(rng, 200, 60_000)}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _rmat_ids(scale, count, gen):
    """Endpoints of `count` R-MAT samples; `scale` is a number or one entry per sample."""
    u = torch.zeros(count, dtype=torch.int64, device="cuda")
    v = torch.zeros(count, dtype=torch.int64, device="cuda")
    levels = int(scale if isinstance(scale, int) else scale.max())
    for level in range(levels):
        r = torch.rand(count, device="cuda", generator=gen)
        bu = (r >= A + B).long()
        bv = (((r >= A) & (r < A + B)) | (r >= A + B + C)).long()
        if isinstance(scale, int):
            u = 2 * u + bu
            v = 2 * v + bv
        else:
            on = level < scale
            u = torch.where(on, 2 * u + bu, u)
            v = torch.where(on, 2 * v + bv, v)
    return u, v


def _csr(n, u, v, edges=None, gen=None):
    """Symmetric CSR (int64 offsets, int32 heads, ascending lists) without loops and duplicates; with
    `edges`, a random choice of that many of its edges."""
    lo, hi = torch.minimum(u, v), torch.maximum(u, v)
    key = (lo * n + hi)[lo != hi].unique()
    if edges is not None:
        key = key[torch.randperm(key.numel(), device="cuda", generator=gen)[:edges]]
    lo, hi = key // n, key % n
    key = torch.cat([key, hi * n + lo]).sort().values
    tails, heads = key // n, (key % n).to(torch.int32)
    off = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    off[1:] = torch.bincount(tails, minlength=n).cumsum(0)
    return off, heads


def _graph(case, seed):
    """The case's CSR on the device."""
    n, pairs, gen = case["n"], case["pairs"], _generator(seed)
    if case["model"] == "gnm":
        u = torch.randint(n, (pairs,), device="cuda", generator=gen)
        v = torch.randint(n, (pairs,), device="cuda", generator=gen)
    else:
        scale = max(1, math.ceil(math.log2(n)))
        u, v = _rmat_ids(scale, pairs, gen)
        perm = torch.randperm(1 << scale, device="cuda", generator=gen)
        u, v = perm[u] % n, perm[v] % n
    off, heads = _csr(n, u, v, case.get("edges"), gen)
    if not case.get("sorted", True):
        # shuffle every list: order by (tail, random key)
        tails = torch.repeat_interleave(torch.arange(n, device="cuda"), off.diff())
        key = tails * (1 << 31) + torch.randint(1 << 31, (heads.numel(),), device="cuda", generator=gen)
        heads = heads[key.argsort()].contiguous()
    return off, heads


def _batch(case, seed):
    """Disjoint union of the case's graphs: host vertex bases, device offsets and heads (global ids)."""
    graphs = case["graphs"]
    rng = np.random.default_rng(graphs)  # the sizes belong to the case, the edges to the seed
    n = np.exp(rng.uniform(math.log(case["n_min"]), math.log(case["n_max"]), graphs)).astype(np.int64)
    n = np.maximum(n, 2)
    pairs = (n * rng.uniform(case["deg_min"], case["deg_max"], graphs) / 2).astype(np.int64)
    rmat = rng.random(graphs) < 0.5
    base = np.zeros(graphs + 1, np.int64)
    base[1:] = np.cumsum(n)
    gen = _generator(seed)
    count = int(pairs.sum())
    which = torch.repeat_interleave(torch.arange(graphs), torch.from_numpy(pairs)).cuda()
    ng, vb = torch.from_numpy(n).cuda()[which], torch.from_numpy(base[:-1]).cuda()[which]
    scale = torch.from_numpy(np.ceil(np.log2(n)).astype(np.int64)).cuda()[which]
    u, v = _rmat_ids(scale, count, gen)
    # R-MAT ids shuffled inside their graph by a multiplication with a prime above every size
    u, v = u * 1_000_003 % ng, v * 1_000_003 % ng
    flat = ~torch.from_numpy(rmat).cuda()[which]
    uu = (torch.rand(count, device="cuda", generator=gen).double() * ng).long() % ng
    uv = (torch.rand(count, device="cuda", generator=gen).double() * ng).long() % ng
    u, v = torch.where(flat, uu, u) + vb, torch.where(flat, uv, v) + vb
    off, heads = _csr(int(base[-1]), u, v)
    return base.astype(np.uint64), off, heads


def _host(off, heads):
    return off.cpu().numpy().astype(np.uint64), heads.cpu().numpy().astype(np.uint32)


def _host_graph(case, seed):
    off, heads = _host(*_graph(case, seed))
    return K.Graph(case["n"], off, heads)


def _request_graphs(case, seed):
    base, off, heads = _batch(case, seed)
    off, heads = _host(off, heads)
    return [KB.Batch(base, off, heads).graph(g) for g in range(case["graphs"])]


def _lists(case, seed):
    """Pairs of strictly increasing id lists of ragged lengths, part of each shorter list common to both;
    lengths belong to the case, ids to the seed."""
    sizes, rng = np.random.default_rng(case["lists"]), np.random.default_rng(seed)
    pairs = []
    for _ in range(case["lists"]):
        la, lb = np.exp(sizes.uniform(math.log(case["len_min"]), math.log(case["len_max"]), 2)).astype(np.int64)
        common = int(min(la, lb) * sizes.uniform(0.0, 0.9))
        ids = rng.choice(3 * (la + lb), la + lb - common, replace=False).astype(np.uint32)
        pairs.append((np.sort(ids[:la]), np.sort(np.concatenate([ids[:common], ids[la:]]))))
    return pairs


class _Buffer:
    """A torch tensor as the device buffer (`.ptr`) that the package's calls take."""

    def __init__(self, tensor):
        self.tensor = tensor
        self.ptr = tensor.data_ptr()


def prepare(case, seed):
    op = case["op"]
    state = {"case": case, "ctx": K.Context(0)}
    ctx = state["ctx"]
    if op == "count":
        off, heads = _graph(case, seed)
        state.update(n=case["n"], off=off, heads=heads)
        state["pv"] = torch.zeros(case["n"], dtype=torch.int64, device="cuda") if case["per_vertex"] else None
        if case["tuned"]:
            KT.apply(ctx, KT.graph_key(case["n"], off.cpu().numpy()), KT.load_table(KT.PACKAGE_TABLE))
    elif op in ("count_host", "orient"):
        state["graph"] = _host_graph(case, seed)
    elif op == "batch":
        base, off, heads = _batch(case, seed)
        host_off = off.cpu().numpy().astype(np.uint64)
        # the offsets and heads live on the device only; the host keeps the bases and offsets
        state["batch"] = KB.DeviceBatch(KB.Batch(base, host_off, np.zeros(0, np.uint32)), _Buffer(off), _Buffer(heads))
        state["pv"] = _Buffer(torch.zeros(int(base[-1]), dtype=torch.int64, device="cuda"))
        if case["tuned"]:
            KT.apply(ctx, KT.batch_key(case["graphs"], host_off), KT.load_table(KT.PACKAGE_TABLE))
    elif op == "serve":
        state["graphs"], state["owners"] = zip(*[KV.pinned_graph(g) for g in _request_graphs(case, seed)])
        state["pv"] = np.zeros(sum(g.n for g in state["graphs"]), np.uint64)
        state["pv_of"] = np.split(state["pv"], np.cumsum([g.n for g in state["graphs"]])[:-1])
        state["server"] = KV.Server(ctx)
    elif op == "shard":
        shard = KS.make_shard(_host_graph(case, seed), case["ranks"], case["rank"], KS.CETRIC)
        state["shard"] = KS.upload_shard(ctx, shard)
        # owned and ghost vertices: at most all of them
        state["pv"] = _Buffer(torch.zeros(case["n"], dtype=torch.int64, device="cuda"))
    elif op == "shard_graph":
        off, heads = _graph(case, seed)
        state["graph"] = K.DeviceGraph(case["n"], heads.numel(), _Buffer(off), _Buffer(heads))
        state["pv"] = _Buffer(torch.zeros(case["n"], dtype=torch.int64, device="cuda"))
    else:
        state["pairs"] = _lists(case, seed)
    torch.cuda.synchronize()
    return state


def run(state):
    case, ctx = state["case"], state["ctx"]
    op = case["op"]
    if op == "count":
        total = ctx.count_device(state["n"], state["off"], state["heads"], per_vertex_out=state["pv"])
        return (total, state["pv"]) if case["per_vertex"] else total
    if op == "count_host":
        return ctx.count(state["graph"])
    if op == "orient":
        oriented = ctx.orient(state["graph"])
        return oriented.offsets, oriented.heads
    if op == "batch":
        return KB.count_batch(ctx, state["batch"], per_vertex_out=state["pv"]), state["pv"].tensor
    if op == "serve":
        server = state["server"]
        tickets = [server.submit(g, pv) for g, pv in zip(state["graphs"], state["pv_of"])]
        results = [server.wait(t) for t in tickets]
        return (np.array([r.total for r in results], np.uint64), np.array([r.status for r in results], np.int64),
                state["pv"])
    if op == "shard":
        local, type3 = KS.count_shard_device(ctx, state["shard"], per_vertex_out=state["pv"])
        return local, type3, state["pv"].tensor
    if op == "shard_graph":
        local, type3, _ = KS.count_shard_graph(ctx, state["graph"], case["ranks"], case["rank"],
                                               KS.DITRIC if case["ditric"] else KS.CETRIC,
                                               per_vertex_out=state["pv"])
        return local, type3, state["pv"].tensor
    counts, matches = ctx.intersect(state["pairs"])
    return counts, np.concatenate(matches)


def work(case):
    """Input read once, output written once; integer work only."""
    op = case["op"]
    if op in ("count", "count_host", "orient", "shard_graph"):
        n, pairs = case["n"], case.get("edges", case["pairs"])
        nbytes = 8 * (n + 1) + 8 * pairs  # offsets, two slots per pair
        if op == "orient":
            nbytes += 8 * (n + 1) + 4 * pairs
        elif op != "count" or case["per_vertex"]:
            nbytes += 8 * n
    elif op in ("batch", "serve"):
        span = math.log(case["n_max"] / case["n_min"])
        n = case["graphs"] * (case["n_max"] - case["n_min"]) / span  # mean of a log-uniform size
        pairs = n * (case["deg_min"] + case["deg_max"]) / 4
        nbytes = 8 * n + 8 * pairs + 8 * n + 8 * case["graphs"]
    elif op == "shard":
        # the rank's slots and about as many received ids, its vertices and ghosts
        n, pairs = case["n"], case["pairs"]
        nbytes = 2 * 8 * pairs / case["ranks"] + 8 * n / case["ranks"] + 16 * min(n, 2 * pairs / case["ranks"])
    else:
        span = math.log((case["len_max"] + 1) / case["len_min"])
        mean = (case["len_max"] + 1 - case["len_min"]) / max(span, 1e-9)
        pairs = case["lists"] * mean
        nbytes = 2 * 4 * pairs + 4 * pairs / 4 + 8 * case["lists"]
    return {"bytes": float(nbytes), "flops": 0.0}


# ---------------------------------------------------------------------------
# the same numbers from plain torch, by enumerating wedges
# ---------------------------------------------------------------------------
def _oriented(n, off, heads):
    deg = off.diff()
    tails = torch.repeat_interleave(torch.arange(n, device="cuda"), deg)
    heads = heads.long()
    keep = (deg[tails] < deg[heads]) | ((deg[tails] == deg[heads]) & (tails < heads))
    key = (tails[keep] * n + heads[keep]).sort().values
    tails, heads = key // n, key % n
    ooff = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    ooff[1:] = torch.bincount(tails, minlength=n).cumsum(0)
    return key, tails, heads, ooff


def _per_vertex(n, off, heads):
    """Triangles of every vertex, or None when there are too many wedges."""
    key, tails, heads, ooff = _oriented(n, off, heads)
    pv = torch.zeros(n, dtype=torch.int64, device="cuda")
    if key.numel() == 0:
        return pv
    wedges = ooff.diff()[heads]
    ends = wedges.cumsum(0)
    if int(ends[-1]) > EXACT_WEDGES:
        return None
    one = torch.ones(1, dtype=torch.int64, device="cuda")
    done, first, step = 0, 0, 1 << 27
    while first < key.numel():
        last = max(int(torch.searchsorted(ends, done + step, right=True)), first + 1)
        w = wedges[first:last]
        edge = torch.repeat_interleave(torch.arange(first, last, device="cuda"), w)
        rank = torch.arange(edge.numel(), device="cuda") - (ends[first:last] - w - done).repeat_interleave(w)
        third = heads[ooff[heads[edge]] + rank]
        probe = tails[edge] * n + third
        at = torch.searchsorted(key, probe).clamp_(max=key.numel() - 1)
        hit = key[at] == probe
        for ids in (tails[edge[hit]], heads[edge[hit]], third[hit]):
            pv.index_add_(0, ids, one.expand(ids.numel()))
        done, first = int(ends[last - 1]), last
    return pv


def exact(case, seed):
    op = case["op"]
    if op in ("count", "count_host"):
        off, heads = _graph(case, seed)
        pv = _per_vertex(case["n"], off, heads)
        if pv is None:
            return None
        total = int(pv.sum()) // 3
        if op == "count_host":
            return total, pv.cpu().numpy().astype(np.uint64)
        return (total, pv) if case["per_vertex"] else total
    if op == "orient":
        off, heads = _graph(case, seed)
        _, _, oheads, ooff = _oriented(case["n"], off, heads)
        return ooff.cpu().numpy().astype(np.uint64), oheads.cpu().numpy().astype(np.uint32)
    if op in ("batch", "serve"):
        base, off, heads = _batch(case, seed)
        pv = _per_vertex(int(base[-1]), off, heads)
        if pv is None:
            return None
        ends = torch.cat([pv.new_zeros(1), pv.cumsum(0)]).cpu().numpy()[base.astype(np.int64)]
        totals = (np.diff(ends) // 3).astype(np.uint64)
        if op == "batch":
            return totals, pv
        return totals, np.zeros(len(totals), np.int64), pv.cpu().numpy().astype(np.uint64)
    if op == "intersect":
        common = [np.intersect1d(a, b, assume_unique=True) for a, b in _lists(case, seed)]
        return np.array([len(c) for c in common], np.uint64), np.concatenate(common)
    return None  # a rank's share of the triangles has no short closed form
