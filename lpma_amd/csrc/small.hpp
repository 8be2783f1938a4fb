// small.hpp -- a lone PMA's small batch in one kernel, up to the elected
// windows (part of update.hip).
//
// A batch of a few thousand keys is a chain of latencies: pack, sort, locate,
// compact, density check and election took eight launches of 3 to 13 us for
// any size below 10^4.  Here the keys are shared out over the chip, a wave a
// key, while other workgroups sum the count pyramid's levels the last batch
// left owing; the last workgroup to arrive compacts the batch, checks the
// density and elects (nothing waits inside the kernel), and stores the outcome
// for the host.  The rebalance kernel follows.  Up to SMALL_MAX_N keys, of
// which the last workgroup holds two a thread.  Bound: latency.  1000 keys on
// 2^20 vertices 19 us (one workgroup sorting and searching alone: 27), 256 on
// 4096 13 (13).  One call with everything around it, on 2^20 vertices and 8
// million edges: 1000 keys 29 us (60 with eight launches, 37 with one
// workgroup), 2000 keys 34 (55 with one).
#pragma once

static constexpr u32 SM_TPB = 1024;
static constexpr u32 SM_ITEMS = SMALL_MAX_N / SM_TPB;
static constexpr u32 SM_PYR_GRID = 1024;     // workgroups of the pyramid's chunk levels

struct SmallLds {
    union {
        u64 sp[SMALL_MAX_N];  // the batch's keys as they came
        struct {
            u32 v0[PYR_CH], v1[PYR_CH / 2];
        };
        u32 top[2 * PYR_TOP_LDS];
    };
    u32 seg[SMALL_MAX_N];     // segments of the compacted updates
    i32 pd[SMALL_MAX_N + 1];  // their prefix
    u32 c0[SMALL_MAX_N];      // their segments' counts
    Density dn;
    u32 wt[SM_ITEMS][SM_TPB / 64];
    u32 cls[NUM_CLASSES];
    u32 flags, mask, last;
    BatchSeg segs[INLINE_SEGS];
};

// Counts one arrival, after the workgroup's stores so far have been written
// (through, by put<true>: a write-back of the L2 for each of 256 workgroups took
// 18 us): true in every thread of the workgroup that arrives last of `of`, which
// then sees the stores of all.  Nothing waits.
__device__ __forceinline__ bool arrive_last(u32 *count, u32 of, SmallLds &S) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0)
        S.last = __hip_atomic_fetch_add(count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == of - 1 ? 1u : 0u;
    __syncthreads();
    if (!S.last) return false;
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    return true;
}

// the density bounds into LDS
__device__ __forceinline__ void small_density(const Group &g, SmallLds &S) {
    static_assert(sizeof(Density) % 8 == 0 && sizeof(Density) / 8 <= SM_TPB, "one word a thread");
    if (threadIdx.x < sizeof(Density) / 8) ((u64 *)&S.dn)[threadIdx.x] = ((const u64 *)&g.tab[0].dn)[threadIdx.x];
}

// Density check and election of the compacted batch (S.seg, S.pd, n_eff): as
// k_density and k_leaders, by one workgroup.  Every run climbs to its own
// window (two gallops in LDS and one pyramid count a level); windows above
// level 0 are claimed, and a run leads if it owns its window's claim and no
// claimed window of a higher level contains it.
__device__ __forceinline__ void small_settle(const Group &g, const BatchBufs &bb, SmallLds &S, u32 n_eff, u32 flags,
                                             EarlyOut *early) {
    const DevState &d = g.one;
    const Density &dn = S.dn;
    const u64 nseg = nseg_of(d);
    const u64 tag = (u64)g.epoch << 32;
    const u32 t = threadIdx.x;
    const i32 delta = S.pd[n_eff];
    if (t == 0) {
        S.flags = flags;
        S.mask = 0;
    }
    if (t < NUM_CLASSES) S.cls[t] = 0;
    __syncthreads();
    u32 lv[SM_ITEMS], u0[SM_ITEMS], u1[SM_ITEMS], fC[SM_ITEMS], fM[SM_ITEMS];
    bool run[SM_ITEMS];
    const i64 mroot = n_eff ? (i64)*count_ptr(d, d.H, 0) + (i64)delta : 0;
    const bool grows = mroot > (i64)(nseg << d.log2S);
    u32 myflags = 0, mymask = 0;
#pragma unroll
    for (u32 r = 0; r < SM_ITEMS; ++r) {
        const u32 j = t + r * SM_TPB;
        run[r] = j < n_eff && (j == 0 || S.seg[j - 1] != S.seg[j]);
        lv[r] = 0;
        u0[r] = j;
        u1[r] = j + 1;
        fC[r] = fM[r] = 0;
        if (!run[r]) continue;
        const u32 s = S.seg[j];
        u32 l = grows ? d.H + 1 : 0;
        for (; l <= d.H; ++l) {
            const u64 w = (u64)s >> l;
            const u64 a = w << l, e = a + (1ull << l);
            const u32 guess = max(1u, u1[r] - u0[r]);
            const u32 C = l == 0 ? S.c0[j] : *count_ptr(d, l, w);
            u0[r] = gallop_back(S.seg, u0[r], (u32)a, guess);
            u1[r] = e < nseg ? gallop_fwd(S.seg, u1[r], n_eff, (u32)e, guess) : n_eff;
            const i64 m = (i64)C + (i64)(S.pd[u1[r]] - S.pd[u0[r]]);
            if (window_fits(dn, l, d.H, (u64)m)) {
                fC[r] = C;
                fM[r] = (u32)m;
                break;
            }
        }
        lv[r] = l;
        if (l >= d.H) {
            myflags |= l == d.H ? FLAG_ROOT : FLAG_RESIZE;
        } else if (l > 0) {
            mymask |= 1u << l;
            atomicMax((unsigned long long *)&d.owner[owner_idx(nseg, l, (u64)s >> l)],
                      (unsigned long long)(tag | (u64)(~j)));
        }
    }
    const u32 f = dpp_or32(myflags), mk = dpp_or32(mymask);
    if (lane_id() == 0) {
        if (f) atomicOr(&S.flags, f);
        if (mk) atomicOr(&S.mask, mk);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the claims, before they are read
    __syncthreads();
    flags = S.flags;
    const u32 mask = S.mask;
    if (!(flags & (FLAG_INVALID_KEY | FLAG_ROOT | FLAG_RESIZE))) {
        Work wk[SM_ITEMS];
        int cls[SM_ITEMS];
        u32 off[SM_ITEMS];
#pragma unroll
        for (u32 r = 0; r < SM_ITEMS; ++r) {
            const u32 j = t + r * SM_TPB;
            cls[r] = -1;
            off[r] = 0;
            if (!run[r]) continue;
            const u32 s = S.seg[j], L = lv[r];
            auto owner = [&](u32 l) {
                return __hip_atomic_load(&d.owner[owner_idx(nseg, l, (u64)s >> l)], __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT);
            };
            bool lead = L == 0 || owner(L) == (tag | (u64)(~j));
            u32 up = lead ? mask & ~((2u << L) - 1u) : 0u;
            while (up) {
                const u32 l2 = (u32)__builtin_ctz(up);
                up &= up - 1;
                if ((owner(l2) >> 32) == (u64)g.epoch) lead = false;
            }
            if (!lead) continue;
            wk[r] = Work{0u, (u32)(((u64)s >> L) << L), L, u0[r], u1[r], fC[r], fM[r]};
            cls[r] = work_class((u64)fC[r] + (u1[r] - u0[r]), L, d.log2S);
            off[r] = atomicAdd(&S.cls[cls[r]], 1u);
        }
#pragma unroll
        for (u32 r = 0; r < SM_ITEMS; ++r)
            if (cls[r] >= 0) bb.work[cls[r]][off[r]] = wk[r];
    }
    __syncthreads();
    if (t == 0) {
        Status st;
        st.flags = flags;
        st.n_eff = n_eff;
        st.delta = delta;
        for (int c = 0; c < NUM_CLASSES; ++c) st.nwork[c] = S.cls[c];
        PmaStat ps;
        ps.flags = flags & (FLAG_ROOT | FLAG_RESIZE);
        ps.u0 = 0;
        ps.u1 = n_eff;
        ps.pd0 = 0;
        ps.pd1 = delta;
        *bb.status = st;
        g.pstat[0] = ps;
        report_early(st, ps, early, g.epoch);
    }
}

// Compacts the batch, update j's (effective, insert) in own[r] of thread t, j = t
// + r * SM_TPB (1 and 1 << 16), with its key, segment and count, into LDS and
// memory.  Returns n_eff.
__device__ __forceinline__ u32 small_compact(const BatchBufs &bb, SmallLds &S, const u32 (&own)[SM_ITEMS],
                                             const u64 (&key)[SM_ITEMS], const u32 (&seg)[SM_ITEMS],
                                             const u32 (&c0)[SM_ITEMS]) {
    const u32 t = threadIdx.x, wv = t >> 6;
    u32 inc[SM_ITEMS];
#pragma unroll
    for (u32 r = 0; r < SM_ITEMS; ++r) {
        inc[r] = dpp_incl_scan32(own[r]);
        if (lane_id() == 63) S.wt[r][wv] = inc[r];
    }
    __syncthreads();
    u32 before = 0;
#pragma unroll
    for (u32 r = 0; r < SM_ITEMS; ++r) {
        u32 pre = before;
        for (u32 w = 0; w < SM_TPB / 64; ++w) {
            const u32 x = S.wt[r][w];
            if (w < wv) pre += x;
            before += x;
        }
        pre += inc[r] - own[r];
        if (own[r]) {
            const u32 j = pre & 0xFFFFu;
            const i32 x = 2 * (i32)(pre >> 16) - (i32)j;
            S.seg[j] = seg[r];
            S.pd[j] = x;
            S.c0[j] = c0[r];
            bb.ckey[j] = key[r];
            bb.cseg[j] = seg[r];
            bb.pd[j] = x;
        }
    }
    const u32 n_eff = before & 0xFFFFu;
    if (t == 0) {
        const i32 x = 2 * (i32)(before >> 16) - (i32)n_eff;
        S.pd[n_eff] = x;
        bb.pd[n_eff] = x;
    }
    return n_eff;
}

// The first `parts` workgroups: the batch, a wave a key.  A workgroup loads all
// the keys and takes SPLIT_KEYS of them: it finds each one's place in the
// batch's order, and whether a later equal one follows, by comparing it with
// all the keys, searches its segment 128 ways at a step, and leaves its outcome
// at its place.  The others: the pyramid (chunks: the chunk levels owed, 0 if
// none; its top levels always).  The last workgroup to arrive compacts, checks
// and elects.  arrive: two counters, zero before and after.
static constexpr u32 SPLIT_KEYS = SM_TPB / 64;

// an outcome: segment, its count (at most 1024), effective, insert
static constexpr u64 SPLIT_EFF = 1ull << 48, SPLIT_INS = 1ull << 49;

__global__ __launch_bounds__(SM_TPB) void k_small(Group g, BatchBufs bb, InlineSegs in, u32 n, u32 parts,
                                                        u32 chunks, u32 *arrive, EarlyOut *early) {
    __shared__ SmallLds S;
    const DevState &d = g.one;
    const u32 t = threadIdx.x, lane = lane_id();
    if (blockIdx.x >= parts) {
        const u32 np = gridDim.x - parts;
        for (u32 c = blockIdx.x - parts; c < chunks; c += np) {
            pyr_chunk<true>(d, c, S.v0, S.v1);
            __syncthreads();
        }
        if (np > 1 && !arrive_last(&arrive[0], np, S)) return;
        pyr_top_levels<true>(d, S.top);
    } else {
        if (t < in.n) S.segs[t] = in.s[t];
        __syncthreads();
        bool bad = false;
#pragma unroll
        for (u32 r = 0; r < SM_ITEMS; ++r) {
            const u32 i = t + r * SM_TPB;
            if (i < n) S.sp[i] = pack_element(S.segs[source_of(S.segs, in.n, i)], i, g.pshift, g.sbits, bad);
        }
        const bool anybad = __syncthreads_or(bad);
        if (blockIdx.x == 0 && t == 0) put<true>(&bb.status->flags, anybad ? FLAG_INVALID_KEY : 0u);
        const u32 i = blockIdx.x * SPLIT_KEYS + (t >> 6);
        if (i < n) {
            const u32 ks = 1 + g.sbits;
            const u64 x = S.sp[i];
            u32 rank = 0;
            bool dup = false;
            for (u32 k = 0; k < n; k += 64) {
                const u32 j = k + lane;
                const u64 y = S.sp[min(j, n - 1)];
                rank += (u32)__popcll(__ballot(j < n && (y < x || (y == x && j < i))));
                dup = dup || (j < n && (y >> ks) == (x >> ks) && (y > x || (y == x && j > i)));
            }
            u64 key = 0, out = 0;
            if (!__any(dup)) {
                const u64 kk = (x & ((1ull << g.pshift) - 1)) >> ks;
                key = ((kk >> d.vbits) << 32) | (kk & ((1ull << d.vbits) - 1));
                const u32 s = wave_locate(d.sep, d.H, key);
                const u64 base = (u64)s << d.log2S;
                const u32 c = d.cnt[s];
                bool there = false;
                for (u32 k = lane; k < 1u << d.log2S; k += 64) there = there || d.keys[base + k] == key;
                const u32 op = (u32)(x & 1);
                out = (u64)s | (u64)c << 32;
                if (op != (__any(there) ? 1u : 0u)) out |= SPLIT_EFF | (op ? SPLIT_INS : 0ull);
            }
            if (lane == 0) {
                put<true>(&bb.ukey[rank], key);
                put<true>(&bb.useg[rank], out);
            }
        }
    }
    if (!arrive_last(&arrive[1], parts + 1, S)) return;
    if (t < 2) __hip_atomic_store(&arrive[t], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    small_density(g, S);
    u64 key[SM_ITEMS];
    u32 own[SM_ITEMS], seg[SM_ITEMS], c0[SM_ITEMS];
#pragma unroll
    for (u32 r = 0; r < SM_ITEMS; ++r) {
        const u32 j = t + r * SM_TPB;
        const u64 out = j < n ? bb.useg[j] : 0ull;
        key[r] = j < n ? bb.ukey[j] : 0ull;
        seg[r] = (u32)out;
        c0[r] = (u32)(out >> 32) & 0xFFFFu;
        own[r] = out & SPLIT_EFF ? 1u | (out & SPLIT_INS ? 1u << 16 : 0u) : 0u;
    }
    const u32 flags = bb.status->flags;
    const u32 n_eff = small_compact(bb, S, own, key, seg, c0);
    __syncthreads();
    small_settle(g, bb, S, n_eff, flags, early);
}

hipError_t small_batch(const Group &g, const BatchBufs &b, const InlineSegs &in, u64 n, u32 chunks, u32 *arrive,
                       EarlyOut *early, hipStream_t st) {
    const u32 np = std::max<u32>(1, std::min<u32>(chunks, SM_PYR_GRID));
    const u32 parts = ((u32)n + SPLIT_KEYS - 1) / SPLIT_KEYS;
    k_small<<<parts + np, SM_TPB, 0, st>>>(g, b, in, (u32)n, parts, chunks, arrive, early);
    return hipGetLastError();
}
