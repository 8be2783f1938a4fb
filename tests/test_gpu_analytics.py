"""GPU BFS and PageRank over the gapped layout against the host oracles:
BFS levels bit-exact, PageRank (FP32) within 1e-6 L1 of the FP64 oracle run
for the same number of iterations."""
import numpy as np
import pytest

import lpma_amd as L
import oracle
from gpu_util import say

pytestmark = pytest.mark.gpu


def build(scale, E, seed, deletes=0):
    V = 1 << scale
    keys = L.shuffle(L.gen_rmat(scale, E, seed=seed), seed + 1)
    pma = L.PMA(V)
    pma.insert(keys[: E // 2])
    for i in range(E // 2, E, 5000):
        pma.insert(keys[i:i + 5000])
    ref = oracle.sort_unique(keys)
    if deletes:
        rng = np.random.default_rng(seed)
        d = ref[rng.choice(ref.size, deletes, replace=False)]
        pma.delete(d)
        ref = oracle.apply(ref, (), d)
    return V, pma, ref


@pytest.mark.parametrize("scale,E,deletes", [(10, 6000, 0), (14, 150000, 20000), (16, 400000, 100000)])
def test_bfs_levels_bit_exact(scale, E, deletes):
    say(f"bfs scale={scale}")
    V, pma, ref = build(scale, E, 5, deletes)
    for src in (0, 1, V // 2):
        lv, depth, scanned = pma.bfs(src)
        got = lv.cpu().numpy().view(np.uint32)
        want = oracle.bfs(ref, V, src)
        assert np.array_equal(got, want)
        reached = want != 0xFFFFFFFF
        assert depth == int(want[reached].max()) + 1
        ro, _ = oracle.csr_of(ref, V)
        deg = np.diff(ro.astype(np.int64))
        assert scanned == int(deg[reached].sum())
    pma.close()


@pytest.mark.parametrize("scale,E,deletes", [(10, 6000, 0), (14, 150000, 20000), (16, 400000, 100000),
                                             (18, 2000000, 300000)])
def test_pagerank_fp32_within_1e6_of_fp64(scale, E, deletes):
    say(f"pagerank scale={scale}")
    V, pma, ref = build(scale, E, 7, deletes)
    pr, iters, delta = pma.pagerank(0.85, 1e-6, 50)
    got = pr.cpu().numpy().astype(np.float64)
    want, _ = oracle.pagerank(ref, V, 0.85, iters)
    assert abs(got.sum() - 1.0) < 1e-5
    l1 = np.abs(got - want).sum()
    assert l1 < 1e-6, (l1, iters, delta)
    pma.close()


def test_bfs_frontier_of_empty_rows():
    """Level 1 is 6000 rows of which all but every 97th are empty, so one run
    of the expansion (2048 slots) spans more frontier entries than it stages
    in LDS and the rest are found by the global search."""
    say("bfs empty-row frontier")
    from gpu_util import keys_of
    V = 1 << 14
    hub = np.arange(1, 6001)
    srcs = [np.zeros(hub.size, dtype=np.int64)]
    dsts = [hub]
    for i in range(1, 6001, 97):
        srcs.append(np.full(12, i))
        dsts.append(6001 + (i * 13 + np.arange(12) * 131) % 9000)
    keys = oracle.sort_unique(keys_of(np.concatenate(srcs), np.concatenate(dsts)))
    pma = L.PMA(V)
    pma.insert(keys)
    for src in (0, 97):
        lv, depth, scanned = pma.bfs(src)
        want = oracle.bfs(keys, V, src)
        assert np.array_equal(lv.cpu().numpy().view(np.uint32), want)
        reached = want != 0xFFFFFFFF
        ro, _ = oracle.csr_of(keys, V)
        deg = np.diff(ro.astype(np.int64))
        assert scanned == int(deg[reached].sum())
        assert depth == int(want[reached].max()) + 1
    pma.close()


def bfs_shape(shape):
    """(V, edge sources, edge destinations)"""
    if shape == "lone":  # no edges at all
        return 1, [], []
    if shape == "path":  # many more levels than are queued at a time
        n = 131
        return n, np.arange(n - 1), np.arange(1, n)
    if shape == "star":  # one row over many runs, then many empty ones
        n = 70001
        return n, np.zeros(n - 1, dtype=np.int64), np.arange(1, n)
    if shape == "ones":  # rows of one edge: as many entries as places in a run
        n = 5000
        return 2 * n + 1, np.concatenate([np.zeros(n, dtype=np.int64), np.arange(1, n + 1)]), np.concatenate(
            [np.arange(1, n + 1), np.arange(n + 1, 2 * n + 1)])
    n = 3001  # rows of every length from 0 to 300 and back
    rng = np.random.default_rng(17)
    src = np.repeat(np.arange(n), np.abs(np.arange(n) % 601 - 300))
    return n, src, rng.integers(0, n, src.size)


@pytest.mark.parametrize("shape", ["lone", "path", "star", "ones", "ramp"])
@pytest.mark.parametrize("slots", [16, 128])
def test_bfs_shapes(shape, slots):
    """Searches of one live graph and of its snapshot, the latter with the
    default width and with one workgroup."""
    from gpu_util import keys_of
    V, s, d = bfs_shape(shape)
    say(f"bfs {shape} S={slots}")
    keys = oracle.sort_unique(keys_of(np.asarray(s, dtype=np.int64), np.asarray(d, dtype=np.int64)))
    pma = L.PMA(V, segment_slots=slots)
    if keys.size:
        pma.insert(keys)
    snap = L.Snapshot(pma)
    deg = np.diff(oracle.csr_of(keys, V)[0].astype(np.int64))
    for src in {0, V // 2, V - 1}:
        want = oracle.bfs(keys, V, src)
        reached = want != 0xFFFFFFFF
        for width in (None, 0, 1):
            if width is not None:
                assert L.lib().lpma_snapshot_set_search_width(snap._h, width) == 0
            lv, depth, scanned = pma.bfs(src) if width is None else snap.bfs(src)
            assert np.array_equal(lv.cpu().numpy().view(np.uint32), want)
            assert depth == int(want[reached].max()) + 1
            assert scanned == int(deg[reached].sum())
    snap.close()
    pma.close()


# large levels through lists: from 2^24 slots and 2^22 places; a bitmap of one
# window, of several, of whole ones and with a few vertices over; a vertex
# beyond the listed sizes; dangling vertices and a hub
@pytest.mark.parametrize("V,listed", [(1500, True), (1 << 20, True), ((1 << 20) + 33, True), (3 << 20, True),
                                      (1 << 22, True), ((1 << 22) + 1, False)])
def test_bfs_large_levels(V, listed):
    from gpu_util import keys_of
    say(f"bfs lists V={V}")
    rng = np.random.default_rng(V)
    E = 9500000
    # half of the edges leave a twentieth of the vertices, a quarter lead to few
    src = rng.integers(0, V, E)
    src[::2] %= max(1, V // 20)
    dst = rng.integers(0, V, E)
    dst[::4] = V - 1 - dst[::4] % max(1, V // 50)
    if V > 10000:
        src = np.concatenate([src, np.zeros(50000, dtype=np.int64)])
        dst = np.concatenate([dst, rng.integers(0, V, 50000)])
    keys = oracle.sort_unique(keys_of(src, dst))
    pma = L.PMA(V)
    pma.bulk_load(keys)
    if V > 10000:
        assert pma.view().capacity >= 1 << 24
    deg = np.diff(oracle.csr_of(keys, V)[0].astype(np.int64))
    for src in (0, V - 1):
        want = oracle.bfs(keys, V, src)
        reached = want != 0xFFFFFFFF
        for _ in range(2):
            lv, depth, scanned = pma.bfs(src)
            assert np.array_equal(lv.cpu().numpy().view(np.uint32), want)
            assert depth == int(want[reached].max()) + 1
            assert scanned == int(deg[reached].sum())
    pma.close()


def test_bfs_large_levels_without_lists():
    """A search that cannot have its lists (a word a slot), and one of a given
    width, find the same."""
    from gpu_util import keys_of
    say("bfs without lists")
    rng = np.random.default_rng(3)
    V, E = 200000, 9500000
    keys = oracle.sort_unique(keys_of(rng.integers(0, V, E) % 150000, rng.integers(0, V, E)))
    pma = L.PMA(V)
    pma.bulk_load(keys)
    assert pma.view().capacity >= 1 << 24
    want = oracle.bfs(keys, V, 1)
    snap = L.Snapshot(pma)
    assert L.lib().lpma_snapshot_set_search_width(snap._h, 64) == 0
    pma.bfs(1)  # its other scratch is in the pool now
    L.lib().lpma_pool_trim()
    try:
        L.set_pool_budget(L.pool_reserved_bytes() + (8 << 20))
        got = [pma.bfs(1), snap.bfs(1)]
    finally:
        L.set_pool_budget(0)
    got.append(pma.bfs(1))
    for lv, depth, scanned in got:
        assert np.array_equal(lv.cpu().numpy().view(np.uint32), want)
        assert (depth, scanned) == (got[2][1], got[2][2])
    snap.close()
    pma.close()


def test_pagerank_partial_last_bin():
    """V = 20000: three destination bins of 8192 vertices, the last one
    partial; uniform edges with a tenth of the vertices dangling."""
    say("pagerank V=20000")
    from gpu_util import keys_of
    V = 20000
    rng = np.random.default_rng(11)
    src = rng.integers(0, V, 300000)
    src = src[src % 10 != 3]  # vertices 3, 13, ... have no out-edges
    dst = rng.integers(0, V, src.size)
    keep = src != dst
    keys = oracle.sort_unique(keys_of(src[keep], dst[keep]))
    pma = L.PMA(V)
    pma.insert(keys)
    pr, iters, delta = pma.pagerank(0.85, 1e-6, 50)
    got = pr.cpu().numpy().astype(np.float64)
    want, _ = oracle.pagerank(keys, V, 0.85, iters)
    assert abs(got.sum() - 1.0) < 1e-5
    l1 = np.abs(got - want).sum()
    assert l1 < 1e-6, (l1, iters, delta)
    pma.close()


def test_pagerank_more_bins_than_staged_pass():
    """V = 2^24 + 5: 2049 destination bins, past the staged bin pass's LDS,
    so the unstaged bin pass (no padding) runs."""
    say("pagerank V=2^24+5")
    from gpu_util import keys_of
    V = (1 << 24) + 5
    rng = np.random.default_rng(12)
    src = rng.integers(0, V, 200000)
    dst = np.concatenate([rng.integers(0, 1 << 12, 100000), rng.integers(V - 4096, V, 100000)])
    keep = src != dst
    keys = oracle.sort_unique(keys_of(src[keep], dst[keep]))
    pma = L.PMA(V)
    pma.insert(keys)
    pr, iters, delta = pma.pagerank(0.85, 1e-6, 50)
    got = pr.cpu().numpy().astype(np.float64)
    want, _ = oracle.pagerank(keys, V, 0.85, iters)
    assert abs(got.sum() - 1.0) < 1e-5
    l1 = np.abs(got - want).sum()
    assert l1 < 1e-6, (l1, iters, delta)
    pma.close()


def test_pagerank_atomic_push_above_binned_limit():
    """V = 2^27 + 1: more destination bins than the binned push's LDS cursors
    hold, so PageRank takes the per-edge compensated atomic push."""
    say("pagerank V=2^27+1")
    from gpu_util import keys_of
    V = (1 << 27) + 1
    rng = np.random.default_rng(13)
    src = rng.integers(0, V, 100000)
    dst = np.concatenate([rng.integers(0, 4096, 50000), rng.integers(V - 4096, V, 50000)])
    keep = src != dst
    keys = oracle.sort_unique(keys_of(src[keep], dst[keep]))
    pma = L.PMA(V)
    pma.insert(keys)
    pr, iters, delta = pma.pagerank(0.85, 1e-6, 50)
    got = pr.cpu().numpy().astype(np.float64)
    del pr
    want, _ = oracle.pagerank(keys, V, 0.85, iters)
    assert abs(got.sum() - 1.0) < 1e-5
    l1 = np.abs(got - want).sum()
    assert l1 < 1e-6, (l1, iters, delta)
    pma.close()


@pytest.mark.parametrize("slots", [4, 64, 256])
def test_bfs_and_pagerank_other_segment_sizes(slots):
    """The expansion and the bin passes read live lines through the segment
    counts, whose geometry follows the segment size."""
    say(f"analytics segment_slots={slots}")
    V = 1 << 14
    keys = L.shuffle(L.gen_rmat(14, 150000, seed=21), 22)
    pma = L.PMA(V, segment_slots=slots)
    pma.insert(keys[:100000])
    pma.insert(keys[100000:])
    ref = oracle.sort_unique(keys)
    rng = np.random.default_rng(23)
    d = ref[rng.choice(ref.size, 20000, replace=False)]
    pma.delete(d)
    ref = oracle.apply(ref, (), d)
    for src in (0, 3):
        lv, depth, scanned = pma.bfs(src)
        assert np.array_equal(lv.cpu().numpy().view(np.uint32), oracle.bfs(ref, V, src))
    pr, iters, delta = pma.pagerank(0.85, 1e-6, 50)
    want, _ = oracle.pagerank(ref, V, 0.85, iters)
    l1 = np.abs(pr.cpu().numpy().astype(np.float64) - want).sum()
    assert l1 < 1e-6, (l1, iters, delta)
    pma.close()


@pytest.mark.parametrize("V", [1, 2, 3])
def test_tiny_and_empty_graphs(V):
    """No edges: every vertex dangles, so PageRank is uniform and BFS reaches
    only its root; then one edge 0 -> 1 where there is a vertex 1."""
    say(f"analytics tiny V={V}")
    from gpu_util import keys_of
    pma = L.PMA(V)
    for keys in ([], [(0, 1)] if V > 1 else []):
        if keys:
            pma.insert(keys_of([k[0] for k in keys], [k[1] for k in keys]))
        ref = oracle.sort_unique(keys_of([k[0] for k in keys], [k[1] for k in keys])) if keys else \
            np.empty(0, dtype=np.uint64)
        lv, depth, scanned = pma.bfs(0)
        want = oracle.bfs(ref, V, 0)
        assert np.array_equal(lv.cpu().numpy().view(np.uint32), want)
        assert scanned == len(keys)
        pr, iters, delta = pma.pagerank(0.85, 1e-6, 50)
        got = pr.cpu().numpy().astype(np.float64)
        exp, _ = oracle.pagerank(ref, V, 0.85, iters)
        assert np.abs(got - exp).sum() < 1e-6, (got, exp)
    pma.close()


@pytest.mark.parametrize("V,E", [(128, 2400), (8192, 60000), (8193, 60000), (30000, 2500000), (3000, 1200000)])
def test_pagerank_bins_and_chunks(V, E):
    """One bin and one vertex more, bins of one chunk of edges and of several,
    parts of one and of many steps, padded groups in every run, most edges
    into a few vertices; fixed iteration counts, the last one reported."""
    say(f"pagerank bins V={V} E={E}")
    from gpu_util import keys_of
    rng = np.random.default_rng(V)
    src = rng.integers(0, V, E)
    dst = np.where(rng.random(E) < 0.5, rng.integers(0, V, E), rng.integers(0, min(V, 40), E))
    keys = oracle.sort_unique(keys_of(src, dst))
    pma = L.PMA(V)
    pma.insert(keys)
    for iters in (1, 2, 7):
        pr, it, delta = pma.pagerank(0.85, 0.0, iters)
        assert it == iters
        got = pr.cpu().numpy().astype(np.float64)
        want, _ = oracle.pagerank(keys, V, 0.85, iters)
        assert np.abs(got - want).sum() < 1e-6
    before, _ = oracle.pagerank(keys, V, 0.85, 6)
    assert abs(delta - np.abs(want - before).sum()) < 1e-6
    pma.close()


@pytest.mark.parametrize("V,E", [((1 << 17) + 3, 2000), (1 << 20, 150000), ((1 << 24) + 5, 20000000)])
def test_pagerank_runs_of_edges(V, E):
    """Few edges over many bins and parts, whose runs go without padding, and
    more bins than the staged bin pass takes with enough edges for padding."""
    say(f"pagerank runs V={V} E={E}")
    from gpu_util import keys_of
    rng = np.random.default_rng(V)
    dst = rng.integers(0, V, E)
    dst[::3] = V - 1 - dst[::3] % 5000
    keys = oracle.sort_unique(keys_of(rng.integers(0, V, E), dst))
    pma = L.PMA(V)
    pma.insert(keys)
    pr, iters, delta = pma.pagerank(0.85, 0.0, 3)
    want, _ = oracle.pagerank(keys, V, 0.85, 3)
    assert np.abs(pr.cpu().numpy().astype(np.float64) - want).sum() < 1e-6
    pma.close()


@pytest.mark.parametrize("degree", [1000, 37])
def test_pagerank_small_ranks(degree):
    """Ranks far below 1/V keep FP32's relative precision: with damping 1 a
    path whose vertices also lead to a cycle passes 1/degree of its rank on at
    each step (1/V degree^-k after k of them).  A rank's value is rounded four
    times an iteration and once when it is scaled, to 2^-24 each."""
    say(f"pagerank small ranks degree={degree}")
    from gpu_util import keys_of
    V, steps = 5000, 6
    cycle = np.arange(2000, V)
    src, dst = [cycle], [np.roll(cycle, -1)]
    for k in range(2000):
        to = np.append(cycle[(np.arange(degree - 1) * 7 + k) % cycle.size], (k + 1) % 2000 if k < 1999 else 2000)
        src.append(np.full(degree, k))
        dst.append(to)
    keys = oracle.sort_unique(keys_of(np.concatenate(src), np.concatenate(dst)))
    pma = L.PMA(V)
    pma.insert(keys)
    for it in range(1, steps + 1):
        got = pma.pagerank(1.0, 0.0, it)[0].cpu().numpy().astype(np.float64)
        want, _ = oracle.pagerank(keys, V, 1.0, it)
        there = want > 0
        assert np.array_equal(got > 0, there)
        assert np.max(np.abs(got[there] - want[there]) / want[there]) < (4 * it + 2) * 2.0 ** -24
    pma.close()


# a bitmap of less than a window, of one and a few vertices, and past the last one
@pytest.mark.parametrize("V,listed", [(4100, True), (5000, True), ((1 << 20) + 1, True), ((1 << 22) + 1, False)])
def test_bfs_levels_that_take_lists(V, listed):
    """Graphs of 2^24 slots and up to 2^22 vertices have lists (a word a slot of
    the pool), which a level of 2^22 places goes through."""
    from gpu_util import keys_of
    say(f"bfs levels through lists V={V}")
    rng = np.random.default_rng(V)
    E = 9500000
    keys = oracle.sort_unique(keys_of(rng.integers(0, V, E), rng.integers(0, V, E)))
    while keys.size < 9000000:
        keys = oracle.sort_unique(np.append(keys, keys_of(rng.integers(0, V, E), rng.integers(0, V, E))))[:E]
    keys = np.sort(rng.permutation(keys)[:9000000])
    pma = L.PMA(V)
    pma.bulk_load(keys)
    slots = int(pma.view().capacity)
    assert slots >= 1 << 24
    row_off = pma.copy_view()[1].cpu().numpy().view(np.uint32).astype(np.int64)
    places = np.diff(row_off)
    want = oracle.bfs(keys, V, 0)
    widest = max(int(places[want == k].sum()) for k in range(int(want[want != 0xFFFFFFFF].max()) + 1))
    assert widest >= 1 << 22 or not listed
    L.lib().lpma_pool_trim()
    held = L.pool_reserved_bytes()
    lv, depth, scanned = pma.bfs(0)
    vectors = 4 << (4 * V + 3).bit_length()  # four words a vertex, in the pool's blocks
    assert (L.pool_reserved_bytes() - held - vectors >= 4 * slots) == listed
    assert np.array_equal(lv.cpu().numpy().view(np.uint32), want)
    deg = np.diff(oracle.csr_of(keys, V)[0].astype(np.int64))
    assert depth == int(want[want != 0xFFFFFFFF].max()) + 1 and scanned == int(deg[want != 0xFFFFFFFF].sum())
    pma.close()


# sums in fixed point where no contribution can fall below what it holds whole
# (by V * V, or from the third iteration on by V and the largest out-degree), else
# in FP64: a hub of every vertex at the rule's edges, and one of a tenth
@pytest.mark.parametrize("V,hub", [(403000, 403000), (405000, 405000), (700000, 233000), (700000, 234000), (50, 50)])
def test_pagerank_smallest_contributions(V, hub):
    say(f"pagerank smallest contributions V={V} hub={hub}")
    from gpu_util import keys_of
    rng = np.random.default_rng(V)
    keys = oracle.sort_unique(keys_of(np.concatenate([np.full(hub, 3), np.arange(V), rng.integers(0, V, 2 * V)]),
                                      np.concatenate([np.arange(hub), (np.arange(V) + 1) % V, rng.integers(0, V, 2 * V)])))
    pma = L.PMA(V)
    pma.insert(keys)
    for it in (1, 2, 5):
        got = pma.pagerank(0.85, 0.0, it)[0].cpu().numpy().astype(np.float64)
        want, _ = oracle.pagerank(keys, V, float(np.float32(0.85)), it)
        # four roundings an iteration and one of the final scale
        assert np.max(np.abs(got - want) / want) < (4 * it + 2) * 2.0 ** -24
    pma.close()
