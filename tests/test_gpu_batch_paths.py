"""Batches at the sizes where the update path changes kernels, against the
oracle (edges, CSR offsets) and its layout model (slots, row offsets)."""
import numpy as np
import pytest

import lpma_amd as L
import oracle
from gpu_util import Triple, keys_of, say

pytestmark = pytest.mark.gpu


def rand_keys(rng, V, n):
    return keys_of(rng.integers(0, V, n), rng.integers(0, V, n))


# 2048 blocks of 256 keys: the last size whose locate and compaction sum the
# blocks directly, and the first with groups of blocks and staged separators
@pytest.mark.parametrize("n", [524288, 524289, 700001])
@pytest.mark.parametrize("V,S,spread", [(3000, 32, 1), (200, 2, 1), (1 << 18, 64, 1), (3000, 32, 7)])
def test_large_batch_locate(n, V, S, spread):
    rng = np.random.default_rng(n + V)
    t = Triple(V, segment_slots=S)
    say(f"locate n={n} V={V} S={S} spread={spread}")
    a = np.repeat(rand_keys(rng, V, -(-n // spread)), spread)[:n]  # runs of equal keys
    t.insert(a)
    t.compare()
    b = rand_keys(rng, V, n)
    t.mixed(b[: n // 2], np.concatenate([a[: n // 3], b[n // 2:]])[: n - n // 2])
    t.compare()
    t.close()


def test_locate_tile_wider_than_its_stage():
    """Few keys over many segments: a tile's separators do not fit the LDS."""
    V, n = 1 << 22, 530001
    rng = np.random.default_rng(5)
    say(f"locate wide V={V} n={n}")
    t = Triple(V, segment_slots=2, model=False)
    t.insert(rand_keys(rng, V, n))
    t.compare(layout=False)
    t.close()


def test_locate_tile_over_two_members():
    """A group round whose tiles hold the end of one member and the start of the next."""
    rng = np.random.default_rng(6)
    Vs = (500, 70000, 9)
    say(f"locate group {Vs}")
    ps = [L.PMA(V) for V in Vs]
    g = L.Group(ps)
    refs = [np.empty(0, dtype=np.uint64) for _ in Vs]
    for r in range(2):
        ins = [rand_keys(rng, V, n) for V, n in zip(Vs, (300001, 300077, 33))]
        dels = [ref[:: 3] for ref in refs]
        g.update(ins, dels)
        for i, V in enumerate(Vs):
            refs[i] = oracle.apply(refs[i], ins[i], dels[i])
            ek, ro = ps[i].export()
            assert np.array_equal(L.to_host_u64(ek), refs[i])
            assert np.array_equal(ro.cpu().numpy().view(np.uint32), oracle.row_offsets(refs[i], V))
            assert ps[i].check() == 0
    g.close()
    for p in ps:
        p.close()


# a rebuild merges when the updates are more than half of the live keys; tiles
# of 2048 merged items: sizes at their edges, deletes on a tile's boundary, a
# hub row, segments from 2 to 1024 slots
@pytest.mark.parametrize("S", [2, 32, 1024])
@pytest.mark.parametrize("V,n", [(1, 1), (3, 5), (100, 2048 - 100), (100, 2049 - 100), (700, 4096), (5000, 60000)])
def test_rebuild_by_merging(V, n, S):
    rng = np.random.default_rng(V + n)
    say(f"rebuild merge V={V} n={n} S={S}")
    t = Triple(V, segment_slots=S)
    a = rand_keys(rng, V, n)
    a[: n // 2] &= np.uint64(0xFFFFFFFF)  # half of the edges leave vertex 0
    t.insert(a)  # grows
    t.compare()
    t.delete(t.ref[rng.random(t.ref.size) < 0.9])  # shrinks: most live keys deleted
    t.compare()
    t.mixed(rand_keys(rng, V, 3 * n), t.ref)  # grows while every edge goes
    t.compare()
    t.delete(t.ref)
    t.compare()
    t.close()


# 3 * 2^16 queries: the first size of the staged search; heights below, at and
# above its table, lines shorter and longer than 16 words
@pytest.mark.parametrize("V,E,S", [(1, 1, 2), (5, 12, 2), (50, 300, 1024), (300, 40000, 2), (20000, 300000, 8),
                                   (20000, 300000, 16), (60000, 1000000, 32), (3000, 900000, 256)])
def test_edge_query_many(V, E, S):
    rng = np.random.default_rng(V + S)
    say(f"edge query V={V} E={E} S={S}")
    import torch
    pma = L.PMA(V, segment_slots=S)
    ref = oracle.sort_unique(rand_keys(rng, V, E))
    pma.insert(ref)
    gone = ref[:: 7]
    pma.delete(gone)
    live = oracle.apply(ref, np.empty(0, dtype=np.uint64), gone)
    for n in ((3 << 16) - 1, 3 << 16, (3 << 16) + 5, 700001):
        q = np.concatenate([rng.choice(ref, n // 2), rand_keys(rng, V, n - n // 2 - 6),
                            keys_of([0, V, V - 1, 0, 0xFFFFFFFF, 0], [0xFFFFFFFF, 0, V, V - 1, 0xFFFFFFFF, 0])])
        rng.shuffle(q)
        got = pma.edge_query(L.to_device(q)).cpu().numpy()
        assert got.size == n and np.array_equal(got != 0, np.isin(q, live))
    pma.close()


# up to 2048 keys: one kernel to the windows; sizes around its sort's powers of
# two, duplicates, mixed and merged requests, growth, shrink, empty effects,
# heights below and above the staged separators and the pyramid's chunk levels
@pytest.mark.parametrize("V,S,fill", [(1, 2, 0), (3, 32, 4), (700, 2, 6000), (700, 1024, 6000), (4096, 32, 40000),
                                      (60000, 2, 200000), (300000, 16, 300000)])
def test_small_batches(V, S, fill):
    rng = np.random.default_rng(V + S)
    say(f"small batches V={V} S={S}")
    t = Triple(V, segment_slots=S)
    if fill:
        t.insert(rand_keys(rng, V, fill))
    for n in (1, 2, 63, 64, 65, 500, 1023, 1024, 1025, 2047, 2048, 2049):
        a = rand_keys(rng, V, n)
        a[: n // 4] = a[n - n // 4: n]  # duplicates
        t.insert(a)
        t.insert(a)  # no effect
        t.compare()
        d = rng.choice(t.ref, min(n, t.ref.size)) if t.ref.size else a
        t.delete(d)
        t.compare()
        k = n // 2
        t.mixed(rand_keys(rng, V, n - k), np.concatenate([a[: k // 2], d[: k - k // 2]])[:k])
        t.compare()
    row = keys_of(np.full(2048, V // 2), rng.integers(0, V, 2048))  # one row: wide windows
    for _ in range(3):
        t.insert(row)
        t.compare()
        t.delete(row)
        t.compare()
    t.close()


def test_small_batch_refused_and_merged():
    V = 5000
    rng = np.random.default_rng(8)
    say("small batches: invalid keys, merged requests")
    t = Triple(V)
    t.insert(rand_keys(rng, V, 30000))
    for n in (1, 64, 2048):
        bad = rand_keys(rng, V, n)
        bad[n // 2] = keys_of([V], [0])[0]
        with pytest.raises(L.LpmaError):
            t.pma.insert(bad)
        t.compare()
    for _ in range(4):
        a, b = rand_keys(rng, V, 700), rand_keys(rng, V, 600)
        b[:300] = a[:300]
        t.pma.update_sequence([(a, b), (b, a[:500])])
        t.mixed(a, b)
        t.mixed(b, a[:500])
        # the layout is that of one batch; the edges are those of two
        t.compare(layout=False)
    t.close()


# the sample-split sort: bucket counts double at powers of two, a thread takes
# two keys above 2^18, buckets of equal keys outgrow their workgroup
@pytest.mark.parametrize("n", [2049, 65537, 131073, 262144, 262145, 400003])
@pytest.mark.parametrize("V,equal", [(1 << 14, 0.0), (1 << 14, 0.5), (40, 0.0)])
def test_sample_split_sort(n, V, equal):
    rng = np.random.default_rng(n)
    say(f"sort n={n} V={V} equal={equal}")
    t = Triple(V)
    a = rand_keys(rng, V, n)
    a[rng.random(n) < equal] = keys_of([V // 3], [V // 2])[0]
    t.insert(a)
    t.compare()
    t.mixed(rand_keys(rng, V, n // 2), a[: n - n // 2])
    t.compare()
    t.close()


# the radix sort: its smallest batch, 4 keys a thread up to 2^20 and 8 above
# (whole tiles and one key more), digits of 7 bits (V = 2^20: 41 bits; 40: 13)
# and of 8 (2^14: 29), half of the keys equal
@pytest.mark.parametrize("n", [(1 << 19) + 1, 1 << 20, (1 << 20) + 1, (1 << 20) + (3 << 13), 1500001])
@pytest.mark.parametrize("V,equal", [(1 << 20, 0.0), (1 << 14, 0.5), (40, 0.0)])
def test_radix_sort(n, V, equal):
    rng = np.random.default_rng(n)
    say(f"sort n={n} V={V} equal={equal}")
    t = Triple(V)
    a = rand_keys(rng, V, n)
    a[rng.random(n) < equal] = keys_of([V // 3], [V // 2])[0]
    t.insert(a)
    t.compare()
    t.mixed(rand_keys(rng, V, n // 2), a[: n - n // 2])
    t.compare()
    t.close()


def test_many_sources():
    """More requests than the split kernel stages, and as many as it does."""
    V = 3000
    rng = np.random.default_rng(3)
    for requests in (64, 65, 100):
        say(f"sources {2 * requests}")
        pma = L.PMA(V)
        ref = rand_keys(rng, V, 50000)
        pma.insert(ref)
        ref = oracle.sort_unique(ref)
        batches = [(rand_keys(rng, V, 1500), rand_keys(rng, V, int(rng.integers(0, 1500)))) for _ in range(requests)]
        pma.update_sequence(batches)
        for a, d in batches:
            ref = oracle.apply(ref, a, d)
        ek, ro = pma.export()
        assert np.array_equal(L.to_host_u64(ek), ref)
        assert np.array_equal(ro.cpu().numpy().view(np.uint32), oracle.row_offsets(ref, V))
        assert pma.check() == 0
        pma.close()


# a group's sources travel as arguments of its first kernel up to 4 and up to
# 64, and as a copy beyond; a lone PMA's as arguments of its sort up to 64
@pytest.mark.parametrize("members", [1, 2, 3, 32, 33])
def test_group_sources(members):
    say(f"group sources {2 * members}")
    rng = np.random.default_rng(members)
    Vs = [int(rng.integers(50, 400)) for _ in range(members)]
    pmas = [L.PMA(V) for V in Vs]
    refs = [oracle.sort_unique(rand_keys(rng, V, 2000)) for V in Vs]
    group = L.Group(pmas)
    group.update(refs, None)
    for _ in range(3):
        ins = [rand_keys(rng, V, 150) for V in Vs]
        dels = [rng.choice(r, 100) for r in refs]
        group.update(ins, dels)
        refs = [oracle.apply(r, a, d) for r, a, d in zip(refs, ins, dels)]
    for p, r in zip(pmas, refs):
        assert np.array_equal(L.to_host_u64(p.export()[0]), r)
        assert p.check() == 0
    group.close()
    one = pmas[0]
    for requests in (2, 3, 32, 33):
        batches = [(rand_keys(rng, Vs[0], 30), rng.choice(refs[0], 20)) for _ in range(requests)]
        one.update_sequence(batches)
        for a, d in batches:
            refs[0] = oracle.apply(refs[0], a, d)
    assert np.array_equal(L.to_host_u64(one.export()[0]), refs[0])
    for p in pmas:
        p.close()


# export: fewer segments than a tile has at least (8), one tile a workgroup, and
# tiles of more segments than are scanned at a time (512: over 2^19 segments)
@pytest.mark.parametrize("V,E,slots", [(1, 0, 32), (3, 2, 2), (500, 3000, 128), (40000, 300000, 16),
                                       (1 << 20, 500000, 2), (1 << 20, 2500000, 2)])
def test_export_tiles(V, E, slots):
    rng = np.random.default_rng(V + E)
    say(f"export V={V} E={E} S={slots}")
    ref = oracle.sort_unique(rand_keys(rng, V, E))
    pma = L.PMA(V, segment_slots=slots)
    if E:
        pma.insert(ref)
        pma.delete(ref[::7])
        ref = np.delete(ref, np.arange(0, ref.size, 7))
    ro = oracle.row_offsets(ref, V)
    ek, got = pma.export()
    assert np.array_equal(L.to_host_u64(ek), ref)
    assert np.array_equal(got.cpu().numpy().view(np.uint32), ro)
    assert np.array_equal(pma.row_offsets().cpu().numpy().view(np.uint32), ro)
    # every live key, markers at the rows' ends, in the order of the store
    src = np.concatenate([ref >> np.uint64(32), np.arange(V, dtype=np.uint64)]).astype(np.int64)
    dst = np.concatenate([ref & np.uint64(0xFFFFFFFF), np.full(V, 0xFFFFFFFF, dtype=np.uint64)])
    order = np.argsort(src, kind="stable")
    src, dst = src[order], dst[order].astype(np.int64)
    data = L.to_host_u64(pma.get_data())
    assert np.array_equal(data >> np.uint64(32), src.astype(np.uint64))
    mark = dst == 0xFFFFFFFF
    assert np.array_equal(data[~mark], ref)
    row, col = pma.to_csr()
    assert np.array_equal(col.cpu().numpy().view(np.uint32), np.where(mark, src, dst).astype(np.uint32))
    assert np.array_equal(row.cpu().numpy().view(np.uint32)[1:], (np.flatnonzero(mark) + 1).astype(np.uint32))
    pma.close()


# neighbor offsets: one workgroup takes 1024 rows and alone stores its result;
# rows inside one segment, over a few (a lane sums them) and over many (a wave
# does), empty ones, ids out of range and repeats
@pytest.mark.parametrize("n", [0, 1, 63, 1024, 1025, 5000, (1 << 20) + 1])
@pytest.mark.parametrize("slots", [16, 64])
def test_neighbor_lists(n, slots):
    import torch
    V = 3000
    rng = np.random.default_rng(n + slots)
    say(f"neighbors n={n} S={slots}")
    hub = np.arange(0, V, 2)
    ref = np.concatenate([rand_keys(rng, V, 30000), keys_of(np.full(hub.size, 7), hub),
                          keys_of(np.full(200, V - 1), rng.integers(0, V, 200))])
    ref = oracle.sort_unique(ref[(ref >> np.uint64(32)) % np.uint64(11) != 0])
    pma = L.PMA(V, segment_slots=slots)
    pma.insert(ref)
    gone = rng.choice(ref, 3000, replace=False)  # gaps
    pma.delete(gone)
    ref = oracle.apply(ref, (), gone)
    ro = oracle.row_offsets(ref, V).astype(np.int64)
    srcs = rng.integers(0, V + 2, n)
    srcs[: min(n, 8)] = [7, V - 1, 0, V, 7, 11, -1, 1][: min(n, 8)]
    at = np.where((srcs >= 0) & (srcs < V), srcs, 0)
    ln = np.where((srcs >= 0) & (srcs < V), ro[at + 1] - ro[at], 0)
    want = np.concatenate([[0], np.cumsum(ln)])
    inner = np.arange(want[-1]) - np.repeat(want[:-1], ln)
    vals = (ref & np.uint64(0xFFFFFFFF)).astype(np.int64)[np.repeat(ro[at], ln) + inner]
    snap = L.Snapshot(pma)
    for store in (pma, snap, pma):
        offs, nb = store.neighbors(torch.from_numpy(srcs.astype(np.int32)))
        assert offs.dtype == torch.int32 and nb.dtype == torch.int32
        assert np.array_equal(offs.cpu().numpy(), want)
        assert np.array_equal(nb.cpu().numpy(), vals)
    ln_dev = torch.empty(max(n, 1), dtype=torch.int32, device="cuda")
    s_dev = torch.from_numpy(srcs.astype(np.int32)).cuda()
    assert L.lib().lpma_neighbor_count(pma._h, s_dev.data_ptr(), n, ln_dev.data_ptr(), None) == 0
    torch.cuda.synchronize()
    assert np.array_equal(ln_dev.cpu().numpy()[:n], ln)
    snap.close()
    pma.close()


def test_neighbor_lists_from_threads():
    """Calls at once on one handle, each on a stream of its own."""
    import threading
    import torch
    V = 2000
    rng = np.random.default_rng(5)
    ref = oracle.sort_unique(rand_keys(rng, V, 30000))
    pma = L.PMA(V)
    pma.insert(ref)
    torch.cuda.synchronize()
    ro = oracle.row_offsets(ref, V).astype(np.int64)
    bad = []

    def work(k):
        r = np.random.default_rng(k)
        st = torch.cuda.Stream()
        with torch.cuda.stream(st):
            for _ in range(20):
                srcs = r.integers(0, V, int(r.integers(1, 4000)))
                s = torch.from_numpy(srcs.astype(np.int32)).cuda()
                offs = torch.empty(srcs.size + 1, dtype=torch.int32, device="cuda")
                total = L.ctypes.c_uint64(0)
                rc = L.lib().lpma_neighbor_offsets(pma._h, s.data_ptr(), srcs.size, offs.data_ptr(),
                                                   L.ctypes.byref(total), st.cuda_stream)
                st.synchronize()
                want = np.concatenate([[0], np.cumsum(ro[srcs + 1] - ro[srcs])])
                if rc or total.value != want[-1] or not np.array_equal(offs.cpu().numpy(), want):
                    bad.append(k)

    ts = [threading.Thread(target=work, args=(k,)) for k in range(6)]
    for x in ts:
        x.start()
    for x in ts:
        x.join()
    assert not bad
    pma.close()


# one key repeated: in a bucket of its workgroup's size and past it, and often
# enough for the batch to leave the sample-split sort
@pytest.mark.parametrize("n,copies", [(300001, 4000), (300001, 4600), (300001, 5500), (300001, 12000), (7000, 6500),
                                      (9000, 8990), (131072, 131072), (1 << 19, 1 << 18)])
@pytest.mark.parametrize("form", ["lone", "sequence", "group", "graph"])
def test_repeated_key(n, copies, form):
    rng = np.random.default_rng(n + copies)
    say(f"repeated key n={n} copies={copies} {form}")
    V = 1 << 14
    ps = [L.PMA(V), L.PMA(50)] if form == "group" else [L.PMA(V)]
    p = ps[0]
    p.set_graph(form == "graph")
    group = L.Group(ps) if form == "group" else None
    ref = oracle.sort_unique(rand_keys(rng, V, 400000))
    p.bulk_load(ref)
    key = keys_of([V // 3], [V // 2])[0]
    for r in range(2):
        a = rand_keys(rng, V, n)
        a[rng.choice(n, copies, replace=False)] = key
        ins, dels = (a, ref[:100]) if r == 0 else (ref[100:200], a[: n - 100])
        if form == "sequence":
            parts = [(x, y) for x, y in zip(np.array_split(ins, 7), np.array_split(dels, 7))]
            p.update_sequence(parts)
        else:
            parts = [(ins, dels)]
            if group:
                group.update([ins, rand_keys(rng, 50, 20)], [dels, None])
            else:
                p.update_mixed(ins, dels)
        for x, y in parts:
            ref = oracle.apply(ref, x, y)
        ek, ro = p.export()
        assert np.array_equal(L.to_host_u64(ek), ref)
        assert np.array_equal(ro.cpu().numpy().view(np.uint32), oracle.row_offsets(ref, V))
        assert p.check() == 0
    if group:
        group.close()
    for q in ps:
        q.close()


def test_hub_of_a_wide_graph():
    """A hub's edges in a graph of so many vertices that thousands of them share
    a projection in the sort."""
    rng = np.random.default_rng(8)
    V, n = (1 << 26) + 3, 300000
    say(f"hub V={V} n={n}")
    p = L.PMA(V)
    a = keys_of(np.full(n, V - 2), V - 1 - rng.integers(0, 1 << 22, n))
    p.insert(a)
    ref = oracle.sort_unique(a)
    p.delete(a[::3])
    ref = oracle.apply(ref, (), a[::3])
    assert np.array_equal(L.to_host_u64(p.export()[0]), ref)
    assert p.check() == 0
    p.close()


def test_repeated_key_costs_no_more_than_the_radix_sort():
    """A batch of 4*10^5 keys, half of them one key, against one without
    repeats: sorted by one workgroup it took ten times as long."""
    import time
    import torch
    say("repeated key, time")
    rng = np.random.default_rng(9)
    V, n = 1 << 20, 400000
    p = L.PMA(V)
    p.bulk_load(rand_keys(rng, V, 2000000))
    spread = rand_keys(rng, V, n)
    repeated = np.where(rng.random(n) < 0.5, spread, keys_of([7], [9])[0])
    took = []
    for keys in (spread, repeated):
        keys = L.to_device(keys, p.device)
        times = []
        for _ in range(9):
            torch.cuda.synchronize()
            t = time.perf_counter()
            p.insert(keys)
            p.delete(keys)
            torch.cuda.synchronize()
            times.append(time.perf_counter() - t)
        took.append(sorted(times)[4])
    say(f"{took[0] * 1e6:.0f} us, half repeated {took[1] * 1e6:.0f} us")
    assert took[1] < 3 * took[0]
    p.close()


@pytest.mark.parametrize("copies", [16, 18, 22])
def test_bucket_of_many_keys_of_one_projection(copies):
    """256 neighboring keys, repeated, share a projection (2^20 vertices: 41 bits,
    of which 32 are compared) and a bucket, of 4096 keys and of more than its
    workgroup holds; inserted and deleted at once."""
    rng = np.random.default_rng(copies)
    V, n = 1 << 20, 300000
    say(f"bucket of 256 keys x {copies}")
    p = L.PMA(V)
    ref = np.empty(0, dtype=np.uint64)
    near = keys_of(np.full(256 * copies, 70000), 5 * 256 + np.tile(np.arange(256), copies))
    for _ in range(2):
        ins = np.concatenate([near, rand_keys(rng, V, n)])
        p.insert(rng.permutation(ins))
        ref = oracle.apply(ref, ins)
        assert np.array_equal(L.to_host_u64(p.export()[0]), ref)
        ins, dels = np.concatenate([near[::3], rand_keys(rng, V, n // 2)]), np.concatenate([near, ref[::5][: n // 2]])
        p.update_mixed(rng.permutation(ins), rng.permutation(dels))
        ref = oracle.apply(ref, ins, dels)
        assert np.array_equal(L.to_host_u64(p.export()[0]), ref)
    assert p.check() == 0
    p.close()
