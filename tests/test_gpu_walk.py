"""How the intersection shares out tails, at the sizes where that can go wrong.

Closed forms (cliques, wheels) for the edges of packs, parts, list blocks and
windows; the oracle for a skewed graph whose workgroup tails are partly hubs.
"""
import ctypes as C

import numpy as np
import pytest

import katric_amd as K
from katric_amd import serve as V
from katric_amd import shard as S
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _cliques(sizes):
    """Disjoint cliques: (graph, per-vertex counts)."""
    edges, pv, at = [], [], 0
    for k in sizes:
        iu = np.triu_indices(k, 1)
        edges.append(np.stack(iu, 1) + at)
        pv.append(np.full(k, (k - 1) * (k - 2) // 2, np.uint64))
        at += k
    return K.Graph.from_edges(at, np.concatenate(edges)), np.concatenate(pv)


def _wheel(n):
    """Vertex 0 joined to a cycle of n - 1 > 3 vertices."""
    rim = np.arange(1, n)
    e = np.concatenate([np.stack([np.zeros(n - 1, np.int64), rim], 1),
                        np.stack([rim, np.roll(rim, -1)], 1)])
    pv = np.full(n, 2, np.uint64)
    pv[0] = n - 1
    return K.Graph.from_edges(n, e), pv


@pytest.fixture
def knobs(ctx):
    saved = ctx.params()
    yield ctx.set_params
    ctx.set_params(**saved)


def _check(ctx, g, pv):
    total, got = ctx.count(g)
    np.testing.assert_array_equal(got, pv)
    assert total == int(pv.sum()) // 3


@pytest.mark.parametrize("order", [K.ORDER_DEGREE, K.ORDER_VERTEX])
@pytest.mark.parametrize("min_side", [0, 1])
# one wave's pack: 64 set members and 64 entries; its tables: 512 slots
@pytest.mark.parametrize("sizes", [[2, 3, 4, 5] * 40, [63, 64, 65, 66, 67], [3] * 500 + [33, 64, 65] * 8,
                                   list(range(2, 140))])
def test_packs(ctx, knobs, sizes, min_side, order):
    knobs(min_side=min_side, order=order)
    g, pv = _cliques(sizes)
    _check(ctx, g, pv)


@pytest.mark.parametrize("order", [K.ORDER_DEGREE, K.ORDER_VERTEX])
# a row of one part, two parts, and of many parts (the least and the largest part size)
@pytest.mark.parametrize("n", [5, 17, 65, 513, 514, 1025, 4097, 5000, 300_001])
def test_long_rows(ctx, knobs, n, order):
    knobs(order=order)
    g, pv = _wheel(n)
    _check(ctx, g, pv)


@pytest.mark.parametrize("wave_max_deg", [2, 128, 256])
# cliques beyond 2^22 slots have hub tails (every vertex is one) with list lengths over the blocks of
# eight and the windows of 2048 blocks; 2100 also has tails above the workgroup bin
@pytest.mark.parametrize("k", [1025, 2049, 2052, 2100])
def test_hub_cliques(ctx, knobs, k, wave_max_deg):
    knobs(wave_max_deg=wave_max_deg)
    g, pv = _cliques([k, 5, 64])
    _check(ctx, g, pv)


@pytest.mark.parametrize("per_vertex", [True, False])
@pytest.mark.parametrize("unsorted", [False, True])
def test_hubs_and_others(ctx, knobs, unsorted, per_vertex):
    knobs(wave_max_deg=32)
    g = K.gen_rmat(18, 16, seed=5)  # 262144 vertices: more than there are hubs
    ot, opv, ost = O.run_shmem(g, threads=4)
    if unsorted:
        heads = g.heads.copy()
        for v in range(g.n):
            a, b = int(g.offsets[v]), int(g.offsets[v + 1])
            heads[a:b] = heads[a:b][::-1]
        g = K.Graph(g.n, g.offsets, heads)
    total, pv = ctx.count(g, per_vertex=per_vertex)
    assert total == ot
    if per_vertex:
        np.testing.assert_array_equal(pv, opv)
    st = ctx.stats()
    assert st["wedge_checks"] == ost["wedge_checks"]
    assert st["intersection_size_local"] == ost["intersection_size_local"]


def test_no_hubs_in_a_regular_graph(ctx):
    # a circulant graph of 40000 vertices and degree 32: one degree bin, more
    # vertices than hubs can be.  i ~ i + 1 .. i + 16: triangles at i are pairs
    # (a, b) of distinct offsets in +-1 .. +-16 whose difference is one too
    n, k = 40_000, 16
    i = np.arange(n)
    e = np.concatenate([np.stack([i, (i + d) % n], 1) for d in range(1, k + 1)])
    offs = [d for d in range(-k, k + 1) if d]
    per = sum(1 for a in offs for b in offs if a < b and 0 < b - a <= k)
    _check(ctx, K.Graph.from_edges(n, e), np.full(n, per, np.uint64))


def test_tight_budget_counts_without_the_optional_room():
    # a budget that holds the buffers every count needs, but not part list,
    # hub lists and per-vertex copies beside them
    g = K.gen_rmat(16, 16, seed=3)
    want = O.run_shmem(g, threads=4)
    with K.Context(0) as free:
        free.count(g)
        rich = free.device_bytes()
    with K.Context(0, hbm_budget_bytes=rich - 64 * g.n) as tight:
        total, pv = tight.count(g)
        assert tight.device_bytes() < rich - 64 * g.n + 1
    assert total == want[0]
    np.testing.assert_array_equal(pv, want[1])


@pytest.mark.parametrize("lens", [
    [(0, 5), (5, 0), (0, 0), (1, 1)],                      # empty lists
    [(2047, 10), (1, 2048), (2048, 3000), (2049, 1)],      # a tile's edges
    [(6000, 7), (7, 6000), (64, 64), (63, 65)] * 3,        # lists over several tiles
    [(1, 1)] * 3000 + [(0, 1)] * 5000 + [(3, 2)] * 100,    # more pairs than a tile has ids
])
def test_intersect_tiles(ctx, lens):
    rng = np.random.default_rng(7)
    pairs = [tuple(np.sort(rng.choice(2 * (la + lb) + 1, n, replace=False)).astype(np.uint32) for n in (la, lb))
             for la, lb in lens]
    counts, matches = ctx.intersect(pairs)
    for (a, b), c, m in zip(pairs, counts, matches):
        want = np.intersect1d(a, b)
        assert c == len(want)
        np.testing.assert_array_equal(m, want)


@pytest.mark.parametrize("at", [0, 63, 64, 2047, 2048, 4999])
def test_intersect_order_check_at_tile_edges(ctx, at):
    ids = np.arange(1, 5002, dtype=np.uint32)
    bad = ids.copy()
    bad[at + 1] = bad[at]
    for pair in ((bad, ids), (ids, bad)):
        with pytest.raises(K.KatricError):
            ctx.intersect([pair])
    assert ctx.intersect([(ids, ids[::2])])[0].tolist() == [2501]


@pytest.mark.parametrize("k", [2, 3, 40, 600, 3000])
def test_repeated_edges_in_unsorted_rows(ctx, k):
    # a triangle whose edges all come k times, never twice in a row: only the
    # sort can see it, and with many copies the lists are longer than a simple
    # graph's can be
    rows = [[1, 2] * k, [2, 0] * k, [0, 1] * k]
    off = np.array([0, 2 * k, 4 * k, 6 * k], np.uint64)
    with pytest.raises(K.KatricError):
        ctx.count(K.Graph(3, off, np.concatenate(rows).astype(np.uint32)))
    g, pv = _cliques([5, 9])
    _check(ctx, g, pv)  # the context is none the worse


@pytest.mark.parametrize("n", [1, 2, 4095, 4096, 16383, 16384, 16385, 70_001])
@pytest.mark.parametrize("unsorted", [False, True])
def test_scan_sizes(ctx, n, unsorted):
    # a path of n vertices with a triangle at its end where there is room
    e = np.stack([np.arange(n - 1), np.arange(1, n)], 1)
    tri = n >= 3
    if tri:
        e = np.concatenate([e, [[n - 3, n - 1]]])
    g = K.Graph.from_edges(n, e)
    if unsorted and tri:
        heads = g.heads.copy()
        a, b = int(g.offsets[n - 2]), int(g.offsets[n - 1])
        heads[a:b] = heads[a:b][::-1]
        g = K.Graph(n, g.offsets, heads)
    pv = np.zeros(n, np.uint64)
    if tri:
        pv[n - 3:] = 1
    _check(ctx, g, pv)
    o = ctx.orient(g)
    assert int(o.offsets[-1]) == len(e)


@pytest.mark.parametrize("algo", [S.CETRIC, S.DITRIC])
@pytest.mark.parametrize("longest", [16, 17, 1024, 1025, 4096, 4097])
@pytest.mark.parametrize("lens", [(0, 4096, 0, 0, 1, 4095, 64, 65, 0), (3, 0, 4090, 3, 5000, 9001), (0, 0), (1,)])
def test_shard_lists_and_messages(ctx, algo, longest, lens):
    """Lists at the sort's size classes and messages at the edges of the entry
    tiles: one rank, every ghost above every owned vertex in degree, so an owned
    vertex' list is its ghosts and a message [a, list] closes a triangle for every
    owned u in the list and every ghost of u in it."""
    rng = np.random.default_rng(longest + len(lens))
    nl, n = 40, 30000
    ghosts = np.sort(rng.choice(np.arange(nl, n), 12000, replace=False))
    rows = [np.sort(rng.choice(ghosts, longest if u == 7 else int(rng.integers(0, 60)), replace=False)) for u in range(nl)]
    rows[11] = rows[11][:0]
    msgs = [np.sort(rng.choice(n, k, replace=False)) for k in lens]
    offsets = lambda lists: np.concatenate([[0], np.cumsum([len(x) for x in lists])]).astype(np.uint64)
    ids = lambda lists: np.concatenate(lists).astype(np.uint32)
    sh = S.Shard(algorithm=algo, rank=0, bounds=np.array([0, nl, n], np.uint64), offsets=offsets(rows),
                 heads=ids(rows), ghost_ids=ghosts.astype(np.uint32),
                 ghost_degree=np.full(len(ghosts), 1 << 20, np.uint64),
                 msg_src=rng.choice(ghosts, len(lens), replace=False).astype(np.uint32), msg_offsets=offsets(msgs),
                 msg_heads=ids(msgs))
    want = sum(len(np.intersect1d(rows[u], m)) for m in msgs for u in m[m < nl])
    loc, t3, pv = S.count_shard(ctx, sh)
    assert (loc, t3) == (0, want)
    assert int(pv.sum()) == 3 * want


def test_serve_reads_each_kind_of_memory(ctx):
    """Requests with offsets, heads and counts each in pageable or page-locked
    memory, at the edges of the gather's chunks, mixed in one burst."""
    sizes = [1, 2, 255, 257, 4095, 4096, 4097, 8193]
    cases, owners = [], []
    for i in range(32):
        n = sizes[i % len(sizes)]
        g = K.gen_gnm(n, min(3 * n, n * (n - 1) // 2), seed=i)
        view = V.Graph.__new__(V.Graph)
        pinned, own = V.pinned_graph(g)
        counts = V.PinnedArray(n, np.uint64)
        owners += own + [counts]
        view.n = n
        view.offsets = pinned.offsets if i & 1 else g.offsets
        view.heads = pinned.heads if i & 2 else g.heads
        out = counts.array if i & 4 else np.zeros(n, np.uint64)
        out[:] = 99
        cases.append((view, out, *ctx.count(g)))
    with K.Context(0) as sctx:
        srv = V.Server(sctx)
        tickets = [srv.submit(view, out) for view, out, _, _ in cases]
        results = [srv.wait(t) for t in tickets]
        srv.stop()
    for r, (_, out, total, pv) in zip(results, cases):
        assert (r.status, r.total) == (0, total)
        np.testing.assert_array_equal(out, pv)


@pytest.mark.parametrize("order", [K.ORDER_DEGREE, K.ORDER_VERTEX])
@pytest.mark.parametrize("n", [5, 1023, 1024, 1025, 4095, 4096, 4097])  # one block bins up to 4096 tails
def test_bins_of_one_block(ctx, knobs, n, order):
    knobs(order=order)
    _check(ctx, *_wheel(n))
    g = K.gen_gnm(n, min(8 * n, n * (n - 1) // 2), seed=n)
    _, pv, want = O.run_shmem(g, threads=4)
    _check(ctx, g, pv)
    st = ctx.stats()
    assert st["wedge_checks"] == want["wedge_checks"]
    assert st["intersection_size_local"] == want["intersection_size_local"]


@pytest.mark.parametrize("rank", [0, 1])
def test_shard_hubs(ctx, knobs, rank):
    """CeTriC's local phase above 2^22 slots: hub lists over owned and ghost tails."""
    knobs(wave_max_deg=32)
    g = K.gen_rmat(18, 24, seed=9)
    sh = S.make_shard(g, 2, rank, S.CETRIC)
    assert len(sh.heads) >= 1 << 22
    loc, t3, pv = S.count_shard(ctx, sh)
    oloc, ot3, opv, _ = O.rank_sim(g, 2, rank, S.CETRIC, threads=4)
    assert (loc, t3) == (oloc, ot3)
    full = np.zeros(g.n, np.uint64)
    full[sh.vertex_ids()] = pv
    np.testing.assert_array_equal(full, opv)


def _few_ghost_messages(algo, pad, seed):
    """A shard whose messages hold 1 to 3 known ghosts and 63 to 2000 owned ids, and one message of `pad` unknown
    ids (the length of walks that are split goes with the received entries): (shard, triangles, per-vertex counts)."""
    rng = np.random.default_rng(seed)
    nl, ng = 4096, 200
    n = nl + 2000 + pad
    ghosts = np.sort(rng.choice(np.arange(nl, nl + 1000), ng, replace=False))
    adj = rng.random((nl, ng)) < 0.1
    rows = [ghosts[a] for a in adj]
    src, msgs, pv = [], [], np.zeros(nl + ng, np.uint64)
    for r in (63, 64, 65, 128, 129, 2000):
        for k in (1, 2, 3, 1):
            own = np.sort(rng.choice(nl, r, replace=False))
            sender, *known = rng.choice(ng, k + 1, replace=False)
            known = np.sort(known)
            src.append(sender)
            msgs.append(np.concatenate([own, ghosts[known]]))
            hit = adj[np.ix_(own, known)].astype(np.uint64)
            pv[own] += hit.sum(1)
            pv[nl + known] += hit.sum(0)
            pv[nl + sender] += hit.sum()
    src.append(0)
    msgs.append(np.arange(nl + 2000, n))
    offsets = lambda lists: np.concatenate([[0], np.cumsum([len(x) for x in lists])]).astype(np.uint64)
    ids = lambda lists: np.concatenate(lists).astype(np.uint32)
    sh = S.Shard(algorithm=algo, rank=0, bounds=np.array([0, nl, n], np.uint64), offsets=offsets(rows),
                 heads=ids(rows), ghost_ids=ghosts.astype(np.uint32), ghost_degree=np.full(ng, 1 << 20, np.uint64),
                 msg_src=ghosts[src].astype(np.uint32), msg_offsets=offsets(msgs), msg_heads=ids(msgs))
    return sh, int(pv.sum()) // 3, pv


@pytest.mark.parametrize("order", [K.ORDER_DEGREE, K.ORDER_VERTEX])
@pytest.mark.parametrize("algo", [S.CETRIC, S.DITRIC])
@pytest.mark.parametrize("pad", [0, 900_000, 7_000_000])  # walks split at 16 entries, at 128, not at all
def test_few_ghost_messages(ctx, knobs, order, algo, pad):
    knobs(order=order)
    sh, want, pv = _few_ghost_messages(algo, pad, seed=pad)
    loc, t3, got = S.count_shard(ctx, sh)
    assert (loc, t3) == (0, want)
    np.testing.assert_array_equal(got, pv)


@pytest.mark.parametrize("order", [K.ORDER_DEGREE, K.ORDER_VERTEX])
def test_few_ghost_messages_under_a_tight_budget(order):
    sh, want, pv = _few_ghost_messages(S.CETRIC, 0, seed=1)
    with K.Context(0) as free:
        S.count_shard(free, sh)
        rich = free.device_bytes()
    with K.Context(0, hbm_budget_bytes=rich - 64 * len(pv)) as tight:
        tight.set_params(order=order)
        loc, t3, got = S.count_shard(tight, sh)
        assert tight.device_bytes() <= rich - 64 * len(pv)
    assert (loc, t3) == (0, want)
    np.testing.assert_array_equal(got, pv)


@pytest.mark.parametrize("algo", [S.CETRIC, S.DITRIC])
@pytest.mark.parametrize("n", [1023, 8191, 8193, 100_003])  # the stripes of tails that go to one XCD: 1024
def test_shard_by_vertex(ctx, knobs, n, algo):
    knobs(order=K.ORDER_VERTEX)
    g = K.gen_rmat(17, 12, seed=n, n=n)
    bounds = np.array([0, n // 5, n], np.uint64)
    for rank in (0, 1):
        sh = S.make_shard(g, 2, rank, algo, bounds=bounds)
        loc, t3, pv = S.count_shard(ctx, sh)
        oloc, ot3, opv, _ = O.rank_sim(g, 2, rank, algo, bounds=bounds, threads=4)
        assert (loc, t3) == (oloc, ot3)
        full = np.zeros(g.n, np.uint64)
        full[sh.vertex_ids()] = pv
        np.testing.assert_array_equal(full, opv)


@pytest.mark.parametrize("order", [K.ORDER_DEGREE, K.ORDER_VERTEX])
@pytest.mark.parametrize("n", [150_000, 700_003, 1_700_001])  # 2, 3 and 8 long tails per grab by degree
def test_many_long_tails(ctx, knobs, n, order):
    # a ring where everyone knows the k nearest on both sides: 66 walk entries a tail
    k = 33
    knobs(order=order, min_side=1)
    near = np.concatenate([np.arange(-k, 0), np.arange(1, k + 1)])
    heads = ((np.arange(n)[:, None] + near) % n).astype(np.uint32)
    ends = np.r_[:k, n - k:n]
    heads[ends] = np.sort(heads[ends], 1)
    g = K.Graph(n, np.arange(n + 1, dtype=np.uint64) * (2 * k), heads.reshape(-1))
    per = sum(1 for a in near for b in near if a < b and b - a <= k)
    _check(ctx, g, np.full(n, per, np.uint64))


@pytest.mark.parametrize("algo", [S.CETRIC, S.DITRIC])
def test_messages_beyond_the_cache(ctx, knobs, algo):
    knobs(order=K.ORDER_DEGREE)
    sh, want, pv = _few_ghost_messages(algo, 1 << 26, seed=3)  # taken by vertex from there on
    loc, t3, got = S.count_shard(ctx, sh)
    assert (loc, t3) == (0, want)
    np.testing.assert_array_equal(got, pv)


@pytest.mark.parametrize("wave_max_deg", [2, 64])  # the hubs' lists that k_tc_hub would take: all, none
def test_shard_hub_rule(ctx, knobs, wave_max_deg):
    """Above 2^22 slots, global degrees far above a rank's list lengths."""
    knobs(wave_max_deg=wave_max_deg)
    n = 70_000
    g = K.gen_gnm(n, 9_000_000, seed=4)
    bounds = np.array([0, n // 4, n], np.uint64)
    sh = S.make_shard(g, 2, 0, S.CETRIC, bounds=bounds)
    assert len(sh.heads) >= 1 << 22
    loc, t3, pv = S.count_shard(ctx, sh)
    oloc, ot3, opv, _ = O.rank_sim(g, 2, 0, S.CETRIC, bounds=bounds, threads=4)
    assert (loc, t3) == (oloc, ot3)
    full = np.zeros(n, np.uint64)
    full[sh.vertex_ids()] = pv
    np.testing.assert_array_equal(full, opv)


@pytest.mark.parametrize("lens", [
    [(255, 256), (1, 1), (0, 0), (257, 255), (0, 3)],     # tiles of one id per thread: 256 ids
    [(2047, 9)], [(2048, 9)], [(2049, 9)],                # sums of 2048 ids: one, one, two
    [(0, 700)], [(700, 0)],
    [(1, 1)] * 300 + [(0, 0)] * 400 + [(64, 64)] * 9,     # more pairs than a tile has ids
    [(32768, 32768)], [(32768, 32769)],                   # 2^16 ids in all: the larger tiles from there on
])
@pytest.mark.parametrize("device", [False, True])
def test_intersect_few_ids(ctx, lens, device):
    rng = np.random.default_rng(len(lens))
    pairs = [tuple(np.sort(rng.choice(2 * (la + lb) + 1, n, replace=False)).astype(np.uint32) for n in (la, lb))
             for la, lb in lens]
    want = [np.intersect1d(a, b) for a, b in pairs]
    if not device:
        counts, matches = ctx.intersect(pairs)
    else:
        arrays = []
        for side in (0, 1):
            arrays.append(np.concatenate([[0], np.cumsum([len(p[side]) for p in pairs])]).astype(np.uint64))
            arrays.append(np.concatenate([p[side] for p in pairs]).astype(np.uint32))
        bufs = [ctx.alloc(max(a.nbytes, 8)) for a in arrays]
        for b, a in zip(bufs, arrays):
            if a.size:
                b.upload(a)
        cap = sum(len(w) for w in want)
        out = [ctx.alloc(8 * len(pairs)), ctx.alloc(4 * cap + 8)]
        total = C.c_uint64()
        ctx.check(K._ffi.lib().kt_intersect(ctx.handle, len(pairs), *[b.ptr for b in bufs],
                                            K.KT_DEVICE_INPUT | K.KT_DEVICE_OUTPUT, out[0].ptr, out[1].ptr, cap,
                                            C.byref(total)), "kt_intersect")
        assert total.value == cap
        counts = out[0].download(np.uint64, len(pairs))
        matches = np.split(out[1].download(np.uint32, cap) if cap else np.zeros(0, np.uint32),
                           np.cumsum([len(w) for w in want])[:-1])
    assert counts.tolist() == [len(w) for w in want]
    for m, w in zip(matches, want):
        np.testing.assert_array_equal(m, w)
