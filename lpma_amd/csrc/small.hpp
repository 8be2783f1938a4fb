// small.hpp -- a lone PMA's small batch in one kernel, up to the elected
// windows (part of update.hip).
//
// A batch of a few thousand keys is a chain of latencies: pack, sort, locate,
// compact, density check and election took eight launches of 3 to 13 us for
// any size below 10^4.  Here one workgroup takes the batch through all of it,
// in LDS, while the others sum the count pyramid's levels the last batch left
// owing; the last of the two to arrive checks the density and elects (nothing
// waits inside the kernel), and stores the outcome for the host.  The rebalance
// kernel follows.  Up to SMALL_MAX_N keys: two a thread.  Bound: latency.  256
// keys on 4096 vertices 15 us (load 1.4, sort 4.1, locate 1.4, presence 1.9,
// store and arrival 1.5, density 3, election and report 1.5); 1000 on 2^20
// 27 us (load 3, sort 6.4, locate 8 to 11 over 2^19 segments).  One call with
// everything around it: 50 -> 26 us and 60 -> 40 us.
#pragma once

static constexpr u32 SM_TPB = 1024;
static constexpr u32 SM_ITEMS = SMALL_MAX_N / SM_TPB;
static constexpr u32 SM_TAB_LOG = 12;        // separators staged in LDS
static constexpr u32 SM_PYR_GRID = 1024;     // workgroups of the pyramid's chunk levels
static_assert(SM_ITEMS == 2, "the sort holds two keys a thread");

struct SmallLds {
    union {
        struct {
            u64 sp[SMALL_MAX_N];  // the sort's buffers; then the sorted keys (sp)
            u64 ex[SMALL_MAX_N];
        };
        struct {
            u32 v0[PYR_CH], v1[PYR_CH / 2];
        };
        u32 top[2 * PYR_TOP_LDS];
    };
    u64 tab[1u << SM_TAB_LOG];  // every 2^(H - SM_TAB_LOG)-th separator
    u32 seg[SMALL_MAX_N];       // segments of the compacted updates
    i32 pd[SMALL_MAX_N + 1];    // their prefix
    u32 c0[SMALL_MAX_N];        // their segments' counts
    Density dn;
    u32 wt[SM_ITEMS][SM_TPB / 64];
    u32 cls[NUM_CLASSES];
    u32 flags, mask, n_eff, last;
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
    const u32 f = dpp_reduce32<false>(myflags), mk = dpp_reduce32<false>(mymask);
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

// Workgroup 0: the batch; the others: the pyramid (chunks: the chunk levels
// owed, 0 if none; its top levels always).  arrive: two counters, zero before
// and after.
__global__ __launch_bounds__(SM_TPB) void k_small(Group g, BatchBufs bb, InlineSegs in, u32 n, u32 chunks, u32 *arrive,
                                                  EarlyOut *early) {
    __shared__ SmallLds S;
    const DevState &d = g.one;
    const u32 t = threadIdx.x, wv = t >> 6;
    u32 n_eff = 0, flags = 0;
    if (blockIdx.x > 0) {
        const u32 np = gridDim.x - 1;
        for (u32 c = blockIdx.x - 1; c < chunks; c += np) {
            pyr_chunk<true>(d, c, S.v0, S.v1);
            __syncthreads();
        }
        if (np > 1 && !arrive_last(&arrive[0], np, S)) return;
        pyr_top_levels<true>(d, S.top);
        if (!arrive_last(&arrive[1], 2, S)) return;
        // the batch arrived first: its compacted updates from memory
        n_eff = bb.status->n_eff;
        flags = bb.status->flags;
        for (u32 j = t; j < n_eff; j += SM_TPB) S.seg[j] = (u32)bb.cseg[j];
        for (u32 j = t; j <= n_eff; j += SM_TPB) S.pd[j] = bb.pd[j];
        for (u32 j = t; j < n_eff; j += SM_TPB) S.c0[j] = d.cnt[S.seg[j]];  // (its own entries)
        small_density(g, S);
        __syncthreads();
    } else {
        // keys and staged separators: one round of loads (the separators are
        // wanted after the sort)
        if (t < in.n) S.segs[t] = in.s[t];
        constexpr u32 TPT = (1u << SM_TAB_LOG) / SM_TPB;
        const u32 tl = min(d.H, SM_TAB_LOG), sh = d.H - tl;
        u64 sepv[TPT];
#pragma unroll
        for (u32 k = 0; k < TPT; ++k) {
            const u32 i = t + k * SM_TPB;
            sepv[k] = d.sep[(u64)(i < (1u << tl) ? i : 0u) << sh];
        }
        __syncthreads();
        bool bad = false;
        u64 p[SM_ITEMS];
#pragma unroll
        for (u32 r = 0; r < SM_ITEMS; ++r) {
            const u32 i = t + r * SM_TPB;
            p[r] = ~0ull;
            if (i < n) p[r] = pack_element(S.segs[source_of(S.segs, in.n, i)], i, g.pshift, g.sbits, bad);
        }
        small_density(g, S);
        const bool anybad = __syncthreads_or(bad);
        flags = anybad ? FLAG_INVALID_KEY : 0u;
        block_bitonic<u64, SM_TPB, SM_ITEMS>(p, n, S.ex, S.sp);
#pragma unroll
        for (u32 r = 0; r < SM_ITEMS; ++r)
            if (t + r * SM_TPB < n) S.sp[t + r * SM_TPB] = p[r];
#pragma unroll
        for (u32 k = 0; k < TPT; ++k) S.tab[t + k * SM_TPB] = sepv[k];
        __syncthreads();
        // dedup (the last of equal keys), locate, presence, as the staged edge
        // queries search: staged separators, probes down to a line, the line
        // read by the row of lanes (one compute unit's gathers bound this: 64
        // clocks a wave and probe)
        const u32 ks = 1 + g.sbits;
        const u32 sw = min(16u, 1u << sh), SS = 1u << d.log2S, kw = min(16u, SS);
        u64 key[SM_ITEMS];
        u32 seg[SM_ITEMS], c0[SM_ITEMS], there[SM_ITEMS];
        bool ok[SM_ITEMS];
#pragma unroll
        for (u32 r = 0; r < SM_ITEMS; ++r) {
            const u32 i = t + r * SM_TPB;
            ok[r] = i < n && !(i + 1 < n && (S.sp[i + 1] >> ks) == (p[r] >> ks));
            const u64 kk = (p[r] & ((1ull << g.pshift) - 1)) >> ks;
            key[r] = ok[r] ? ((kk >> d.vbits) << 32) | (kk & ((1ull << d.vbits) - 1)) : 0ull;
            seg[r] = c0[r] = there[r] = 0;
            if ((t & ~63u) + r * SM_TPB >= n) continue;  // whole waves
            u32 at = 0;
            for (u32 h = (1u << tl) >> 1; h; h >>= 1) at += S.tab[at + h] <= key[r] ? h : 0u;
            at <<= sh;
            for (u32 h = (1u << sh) >> 1; h >= 16; h >>= 1) at += d.sep[at + h] <= key[r] ? h : 0u;
            u64 v[8], w[8];
            if (sh) {
                u32 c = 0;
                row_lines<0>(d.sep, at, sw, v);
                row_lines<8>(d.sep, at, sw, w);
                row_counts<0, true>(v, key[r], c);
                row_counts<8, true>(w, key[r], c);
                at += min(c, sw) - 1;
            }
            seg[r] = at;
            c0[r] = d.cnt[at];
            u64 base = (u64)at << d.log2S;
            for (u32 h = SS >> 1; h >= 16; h >>= 1) base += d.keys[base + h - 1] < key[r] ? h : 0u;
            row_lines<0>(d.keys, base, kw, v);
            row_lines<8>(d.keys, base, kw, w);
            row_counts<0, false>(v, key[r], there[r]);
            row_counts<8, false>(w, key[r], there[r]);
        }
        // compaction: (count, inserts) as the halves of one word
        u32 own[SM_ITEMS], inc[SM_ITEMS];
#pragma unroll
        for (u32 r = 0; r < SM_ITEMS; ++r) {
            const u32 op = (u32)(p[r] & 1);
            own[r] = ok[r] && op != there[r] ? 1u | op << 16 : 0u;
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
                put<true>(&bb.cseg[j], (u64)seg[r]);
                put<true>(&bb.pd[j], x);
            }
        }
        n_eff = before & 0xFFFFu;
        if (t == 0) {
            const i32 x = 2 * (i32)(before >> 16) - (i32)n_eff;
            S.pd[n_eff] = x;
            put<true>(&bb.pd[n_eff], x);
            put<true>(&bb.status->n_eff, n_eff);
            put<true>(&bb.status->flags, flags);
        }
        if (!arrive_last(&arrive[1], 2, S)) return;
    }
    if (t < 2) __hip_atomic_store(&arrive[t], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    small_settle(g, bb, S, n_eff, flags, early);
}

hipError_t small_batch(const Group &g, const BatchBufs &b, const InlineSegs &in, u64 n, u32 chunks, u32 *arrive,
                       EarlyOut *early, hipStream_t st) {
    const u32 np = std::max<u32>(1, std::min<u32>(chunks, SM_PYR_GRID));
    k_small<<<1 + np, SM_TPB, 0, st>>>(g, b, in, (u32)n, chunks, arrive, early);
    return hipGetLastError();
}
