// begin.hpp -- device code that several of the update's kernels share: a
// batch's first work (status, update index, the count pyramid), its elements'
// sort keys, and the searches of the density check.
#pragma once
#include "common.hpp"

namespace pma {

// the pyramid's chunk levels: one workgroup reduces a chunk of 2^PYR_CHL
// segments (levels 1..PYR_CHL); the levels above are summed at the next
// batch's start
static constexpr u32 PYR_CHL = 11;

static constexpr u32 PYR_CH = 1u << PYR_CHL;

// A store other workgroups of the same kernel read (COH): written through to
// where every XCD sees it, so its writer needs no write-back of its L2 before
// it signals them.
template <bool COH, class T>
__device__ __forceinline__ void put(T *p, T v) {
    if (COH) __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else *p = v;
}

// Levels 1..PYR_CHL of one chunk of 2^PYR_CHL segments (all levels of a
// smaller PMA), by nt threads of a workgroup (this one tid of them), through
// LDS (v0: PYR_CH words, v1: half).  Every thread of the workgroup calls it; one
// without a chunk (a place past the last) only meets the others' barriers.
template <bool COH = false>
__device__ inline void pyr_chunk(const DevState &d, u64 chunk, u32 *v0, u32 *v1, u32 tid, u32 nt) {
    const u64 nseg = nseg_of(d);
    const u32 levels = d.H < PYR_CHL ? d.H : PYR_CHL;
    const u32 size = (u32)(nseg < PYR_CH ? nseg : PYR_CH);
    const u64 c0 = chunk * size;
    const u32 n = c0 < nseg ? size : 0;
    for (u32 i = tid; i < n; i += nt) v0[i] = d.cnt[c0 + i];
    __syncthreads();
    u32 *in = v0, *tmp = v1;
    for (u32 l = 1; l <= levels; ++l) {
        u32 nw = n >> l;
        u32 *out = d.pyr + pyr_off(nseg, l) + (c0 >> l);
        for (u32 x = tid; x < nw; x += nt) {
            u32 s = in[2 * x] + in[2 * x + 1];
            tmp[x] = s;
            put<COH>(&out[x], s);
        }
        __syncthreads();
        u32 *sw = in; in = tmp; tmp = sw;
    }
}

template <bool COH = false>
__device__ inline void pyr_chunk(const DevState &d, u64 chunk, u32 *v0, u32 *v1) {
    pyr_chunk<COH>(d, chunk, v0, v1, threadIdx.x, blockDim.x);
}

// Levels above the chunk levels, by one workgroup.  Up to PYR_TOP_LDS
// chunk-level counts (H <= 23) are loaded once into LDS and every level
// above is summed there (no global round trip per level), laid out as in
// the pyramid (each level right after the one below), so the levels are
// written out together at the end.  Taller pyramids go level by level
// through global memory.
static constexpr u32 PYR_TOP_LDS = 4096;

// v: 2 * PYR_TOP_LDS words of LDS
template <bool COH = false>
__device__ inline void pyr_top_levels(const DevState &d, u32 *v) {
    const u64 nseg = nseg_of(d);
    if (d.H <= PYR_CHL) return;
    const u64 nc = nseg >> PYR_CHL;
    if (nc <= PYR_TOP_LDS) {
        const u32 *in = d.pyr + pyr_off(nseg, PYR_CHL);
        for (u32 x = threadIdx.x; x < (u32)nc; x += blockDim.x) v[x] = in[x];
        __syncthreads();
        u32 lo = 0, n = (u32)nc;  // the level below: v[lo, lo + n)
        for (u32 l = PYR_CHL + 1; l <= d.H; ++l) {
            for (u32 x = threadIdx.x; x < n / 2; x += blockDim.x) v[lo + n + x] = v[lo + 2 * x] + v[lo + 2 * x + 1];
            lo += n;
            n /= 2;
            __syncthreads();
        }
        // levels PYR_CHL + 1 .. H: v[nc, 2 nc - 1), contiguous in the pyramid too
        u32 *out = d.pyr + pyr_off(nseg, PYR_CHL + 1);
        for (u32 x = threadIdx.x; x < (u32)nc - 1; x += blockDim.x) put<COH>(&out[x], v[nc + x]);
        return;
    }
    for (u32 l = PYR_CHL + 1; l <= d.H; ++l) {
        u64 nw = nseg >> l;
        const u32 *in = d.pyr + pyr_off(nseg, l - 1);
        u32 *out = d.pyr + pyr_off(nseg, l);
        for (u64 x = threadIdx.x; x < nw; x += blockDim.x) put<COH>(&out[x], in[2 * x] + in[2 * x + 1]);
        if (COH) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
    }
}

// One workgroup's share of a batch's first work for PMA pid: its per-batch
// record and claimed-level masks cleared, its pyramid's top levels summed
// (unless v is null: then a later kernel sums them); the workgroup of
// PMA 0 also clears the status, zero[0, nzero) and, for a lone PMA, resets
// the update index wfirst.  v: the LDS of pyr_top_levels.
__device__ inline void batch_first_work(const Group &g, Status *s, u32 pid, u32 *zero, u32 nzero, u32 *wfirst,
                                        u32 *v) {
    if (pid == 0) {
        for (u32 i = threadIdx.x; i < nzero; i += blockDim.x) zero[i] = 0;
        if (g.npma == 1)
            for (u32 i = threadIdx.x; i <= WFIRST_N; i += blockDim.x) wfirst[i] = 0xFFFFFFFFu;
        if (threadIdx.x == 0) {
            s->flags = 0;
            s->n_eff = 0;
            s->delta = 0;
            for (int c = 0; c < NUM_CLASSES; ++c) s->nwork[c] = 0;
        }
    }
    if (threadIdx.x == 0) {
        PmaStat z;
        z.flags = 0; z.u0 = 0; z.u1 = 0; z.pd0 = 0; z.pd1 = 0;
        g.pstat[pid] = z;
    }
    if (threadIdx.x < LV_REPL) g.lvmask[(u64)pid * LV_REPL + threadIdx.x] = 0;
    if (v) pyr_top_levels(pma_of(g, pid), v);
}

// ------------------------------------------------------- batch elements

// Batch element i comes from the source whose [off, off + n) holds it.
// Sources are few and sorted by off; each thread finds its first source by
// binary search and walks forward from there.
__device__ __forceinline__ u32 source_of(const BatchSeg *__restrict__ segs, u32 nsegs, u64 i) {
    u32 lo = 0, hi = nsegs;
    while (hi - lo > 1) {
        u32 mid = (lo + hi) >> 1;
        if (segs[mid].off <= i) lo = mid; else hi = mid;
    }
    return lo;
}

// element i of the batch, a source's, as its sort key (src or dst >= V: bad)
__device__ __forceinline__ u64 pack_element(const BatchSeg &sg, u64 i, u32 pshift, u32 sbits, bool &bad) {
    u64 k = sg.keys[i - sg.off];
    u32 src = (u32)(k >> 32), dst = (u32)k;
    if (src >= sg.V || dst >= sg.V) { bad = true; src = 0; dst = 0; }
    return ((u64)sg.pid << pshift) | ((((((u64)src) << sg.vbits) | dst) << sbits | sg.seq) << 1) | sg.op;
}

// ------------------------------------------------ searches near a position

// first index >= start with a[idx] >= target, given a[start-1] < target;
// the exponential search starts with strides of `step` (a guess of the
// distance)
template <class T>
__device__ __forceinline__ u32 gallop_fwd(const T *__restrict__ a, u32 start, u32 n, typename std::remove_cv<T>::type target,
                                          u32 step) {
    u32 lo = start;
    if (lo >= n || a[lo] >= target) return lo;
    u32 hi = (n - lo > step) ? lo + step : n;
    while (hi < n && a[hi] < target) {
        lo = hi;
        step <<= 1;
        hi = (n - lo > step) ? lo + step : n;
    }
    // a[lo] < target, hi == n or a[hi] >= target
    u32 l = lo + 1, h = hi;
    while (l < h) {
        u32 m = (l + h) >> 1;
        if (a[m] < target) l = m + 1; else h = m;
    }
    return l;
}

// smallest index <= start whose suffix [idx, start] is >= target, given
// a[start] >= target; strides start at `step` as above
template <class T>
__device__ __forceinline__ u32 gallop_back(const T *__restrict__ a, u32 start, typename std::remove_cv<T>::type target,
                                           u32 step) {
    if (start == 0 || a[start - 1] < target) return start;
    u32 hi = start - 1;  // a[hi] >= target
    u32 lo;
    while (true) {
        lo = hi >= step ? hi - step : 0;
        if (a[lo] < target) break;
        if (lo == 0) return 0;
        hi = lo;
        step <<= 1;
    }
    // a[lo] < target <= a[hi]
    u32 l = lo + 1, h = hi;
    while (l < h) {
        u32 m = (l + h) >> 1;
        if (a[m] < target) l = m + 1; else h = m;
    }
    return l;
}

// ------------------------------------------- lines read by rows of lanes
//
// A lane that searches its own line of 16 words alone asks the memory pipe for
// it at every step.  Here a row of 16 lanes reads the lines of its 16 lanes'
// queries one after the other, a word a lane: one request a line.

// lane J of every row of 16 lanes, in all lanes of the row
template <int J>
__device__ __forceinline__ u32 row_lane(u32 x) {
    return (u32)__builtin_amdgcn_update_dpp(0, (int)x, 0x150 + J, 0xF, 0xF, false);  // row_newbcast
}
template <int J>
__device__ __forceinline__ u64 row_lane(u64 x) {
    return ((u64)row_lane<J>((u32)(x >> 32)) << 32) | row_lane<J>((u32)x);
}

// a[at .. at + w) of the row's queries J0 .. J0 + 7 (w <= 16): every lane loads
// one word of each, KEY_NONE past w
template <int J0>
__device__ __forceinline__ void row_lines(const u64 *a, u64 at, u32 w, u64 (&v)[8]) {
    const u32 gl = lane_id() & 15;
#define LPMA_LINE(K)                                                  \
    {                                                                 \
        const u64 x = row_lane<J0 + K>(at); /* by every lane */       \
        v[K] = gl < w ? a[x + gl] : KEY_NONE;                         \
    }
    LPMA_LINE(0) LPMA_LINE(1) LPMA_LINE(2) LPMA_LINE(3) LPMA_LINE(4) LPMA_LINE(5) LPMA_LINE(6) LPMA_LINE(7)
#undef LPMA_LINE
}

// bit J0 + K of the row's answers: how many of the words are <= (LE) or equal
// to query J0 + K's key
template <int J0, bool LE>
__device__ __forceinline__ void row_counts(const u64 (&v)[8], u64 key, u32 &mine) {
    const u32 gl = lane_id() & 15, sh = lane_id() & 48;
#define LPMA_COUNT(K)                                                                                       \
    {                                                                                                       \
        const u64 k = row_lane<J0 + K>(key);                                                                \
        const u32 c = (u32)__popc((u32)(__ballot(LE ? v[K] <= k : v[K] == k) >> sh) & 0xFFFFu);             \
        if (gl == J0 + K) mine = c;                                                                         \
    }
    LPMA_COUNT(0) LPMA_COUNT(1) LPMA_COUNT(2) LPMA_COUNT(3) LPMA_COUNT(4) LPMA_COUNT(5) LPMA_COUNT(6) LPMA_COUNT(7)
#undef LPMA_COUNT
}

// ------------------------------------------------------- bitonic sort

// lane ^ J's value
template <u32 J>
__device__ __forceinline__ u32 lane_xor(u32 x) {
    if constexpr (J == 1) return (u32)__builtin_amdgcn_update_dpp(0, (int)x, 0xB1, 0xF, 0xF, false);  // quad_perm 1,0,3,2
    if constexpr (J == 2) return (u32)__builtin_amdgcn_update_dpp(0, (int)x, 0x4E, 0xF, 0xF, false);  // quad_perm 2,3,0,1
    if constexpr (J == 4) {  // xor 7 (row_half_mirror), then xor 3 (quad_perm 3,2,1,0)
        const int m = __builtin_amdgcn_update_dpp(0, (int)x, 0x141, 0xF, 0xF, false);
        return (u32)__builtin_amdgcn_update_dpp(0, m, 0x1B, 0xF, 0xF, false);
    }
    if constexpr (J == 8) return (u32)__builtin_amdgcn_update_dpp(0, (int)x, 0x128, 0xF, 0xF, false);  // row_ror:8
    if constexpr (J == 16) {  // odd rows of the one against even rows of the other
        const auto r = __builtin_amdgcn_permlane16_swap(x, x, false, false);
        return lane_id() & 16 ? r[0] : r[1];
    }
    const auto r = __builtin_amdgcn_permlane32_swap(x, x, false, false);
    return lane_id() & 32 ? r[0] : r[1];
}
template <u32 J>
__device__ __forceinline__ u64 lane_xor(u64 x) {
    return ((u64)lane_xor<J>((u32)(x >> 32)) << 32) | lane_xor<J>((u32)x);
}

// steps J, J / 2, ..., 1 of a bitonic merge of runs of K / 2
template <class T, u32 NT, u32 ITEMS, u32 K, u32 J>
__device__ __forceinline__ void bitonic_merge(T (&a)[ITEMS], u32 M, T *&b0, T *&b1) {
    const u32 t = threadIdx.x;
    const bool mine = (t & ~63u) < M;  // whole waves past the keys do nothing
    if constexpr (J >= NT) {
#pragma unroll
        for (u32 r = 0; r < ITEMS; ++r) {
            constexpr u32 JI = J / NT;
            if ((r & JI) || (r | JI) >= ITEMS || (r | JI) * NT >= M) continue;
            const bool up = ((r * NT) & K) == 0, less = a[r] < a[r | JI];
            const T lo = less == up ? a[r] : a[r | JI], hi = less == up ? a[r | JI] : a[r];
            a[r] = lo;
            a[r | JI] = hi;
        }
    } else {
        T b[ITEMS];
        if constexpr (J >= 64) {
#pragma unroll
            for (u32 r = 0; r < ITEMS; ++r)
                if (mine && (r == 0 || r * NT < M)) b0[t + r * NT] = a[r];
            __syncthreads();
        }
#pragma unroll
        for (u32 r = 0; r < ITEMS; ++r) {
            if (!mine || (r > 0 && r * NT >= M)) break;
            if constexpr (J >= 64) b[r] = b0[(t ^ J) + r * NT];
            else b[r] = lane_xor<J>(a[r]);
            const u32 i = t + r * NT;
            const bool low = ((i & J) == 0) == ((i & K) == 0);  // keeps the smaller
            a[r] = (a[r] < b[r]) == low ? a[r] : b[r];
        }
        if constexpr (J >= 64) {
            T *x = b0; b0 = b1; b1 = x;
        }
    }
    if constexpr (J > 1) bitonic_merge<T, NT, ITEMS, K, J / 2>(a, M, b0, b1);
}
template <class T, u32 NT, u32 ITEMS, u32 K>
__device__ __forceinline__ void bitonic_merges(T (&a)[ITEMS], u32 M, T *&b0, T *&b1) {
    bitonic_merge<T, NT, ITEMS, K, K / 2>(a, M, b0, b1);
    if constexpr (K < NT * ITEMS) {
        if (K < M) bitonic_merges<T, NT, ITEMS, K * 2>(a, M, b0, b1);
    }
}

// Sorts the n <= NT * ITEMS keys of a workgroup of NT threads in ascending
// order, key i in a[i / NT] of thread i mod NT (the largest value past n, up to
// the power of two M above n, at least 64): partners less than a wave apart
// meet by DPP and lane swaps, those a multiple of NT apart in the thread, the
// others through LDS, one barrier a step (b0, b1: M keys each, in turns; both
// are free afterwards).  A workgroup of 1024: 1000 64-bit keys 6.4 us, 256
// keys 4.1 us; with every lane exchange through LDS 10.2 and 6.5 us.
template <class T, u32 NT, u32 ITEMS>
__device__ __forceinline__ void block_bitonic(T (&a)[ITEMS], u32 n, T *b0, T *b1) {
    u32 M = 64;
    while (M < n) M <<= 1;
    bitonic_merges<T, NT, ITEMS, 2>(a, M, b0, b1);
    __syncthreads();
}

}  // namespace pma
