// analytics.hip -- BFS and PageRank straight over the gapped layout.
//
// The reference runs nvGraph on a CSR copy (test_algos.cu:44-90 PageRank,
// :136-186 BFS; test.cu:170-182 converts with to_csr_rpma first).  Here both
// read the PMA in place: row r's out-edges are the live slots between the
// markers of rows r-1 and r, i.e. slots (row_off[r], row_off[r+1]).
#include <atomic>

#include "common.hpp"
#include "kernels.hpp"

namespace pma {

static constexpr u32 INF_LEVEL = 0xFFFFFFFFu;

// the XCD this wave runs on
__device__ __forceinline__ u32 xcc_id() {
    u32 x;
    asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID, 0, 4)" : "=s"(x));
    return x & 7u;
}

__device__ __forceinline__ void slot_range(const DevState &d, u32 r, u64 &lo, u64 &hi) {
    lo = r == 0 ? 0 : (u64)d.row_off[r] + 1;
    hi = d.row_off[r + 1];
}

// ------------------------------------------------------------------ BFS
//
// Level-synchronous, top-down.  A level expands the frontier's slot ranges
// with one lane per slot, so hub vertices are split over many waves:
//   k_bfs_front   lists the frontier's non-empty rows (the entries): a row's
//                 first place in the level's slots and what to add to a place
//                 to get its slot; and the first entry of every run of
//                 BFS_RUN places;
//   k_bfs_expand  a wave per run: a bit for each entry's first place (so a
//                 place finds its entry by counting bits), then segment
//                 counts, keys and visited words, BFS_ITEMS loads in flight a
//                 lane at each step, dead lines never read.
// The sizes stand in device memory, and a front stores its own where the host
// polls, so the host keeps BFS_AHEAD levels queued past the last it knows of (a
// level after the end costs its empty launches) and nothing waits between
// levels; a copy and a wait after every level, and a fill, three kernels to
// scan and one to search before its expansion, took 100 us a level.
// A visited bitmap (V bits: 2 MB at V = 2^24, held by every XCD's L2) filters
// the edges; the levels array (32 bits per vertex) is only written.  A vertex
// is claimed by the atomic OR that sets its bit, so it enters the next
// frontier once; a plain read of a word another XCD has just changed can only
// miss bits (they go from 0 to 1), which costs an extra atomic, never a wrong
// level.
// Bound: at V = 2^22 and E = 2^26 the two large levels (80 and 70 million
// places) take 671 and 409 us this way, 140 of them for the first's keys; the
// rest are visited words that miss L1 (a miss every 6 to 8 clocks a CU, through
// L1 or past it) and atomics (6 G/s, with or without their results).  A
// workgroup per run of 2048 places, with barriers and a binary search per
// place, took 813 and 510.  Through lists (below) 300 and 290.

// per level mod 4: vertices found, and entries (high 31 bits) and places (low
// 33 bits)
struct BfsCtl {
    u64 ent[4];
    u64 scanned;  // live edges of the frontiers so far
    u32 qn[4];
    u32 depth;    // levels with a frontier
};
static_assert(sizeof(BfsCtl) <= BFS_CTL_WORDS * 4, "control words");

static constexpr u64 BFS_PLACES = (1ull << 33) - 1;
static constexpr u32 BFS_ITEMS = 4;
static constexpr u32 BFS_RUN = 64 * BFS_ITEMS;  // places per run

// Large levels of a graph of at most BFS_WINDOWS * 2^BFS_WIN_LOG vertices go
// through lists (BfsLists): the expansion's waves leave their edges'
// destinations in extents of BFS_EXT, each of one window of the bitmap; a
// workgroup of k_bfs_windows holds a window in LDS and marks the destinations of
// its share of the extents there; k_bfs_merge joins the workgroups' windows.
// The random reads meet LDS instead of L2, and nothing is claimed by atomics in
// memory: 218 us for the expansion, 76 for the windows, 8 to join them, where
// the claims in memory took 671 (80 million places; a 2^22-vertex, 2^26-edge
// search 1250 -> 800 us).  The windows cost 60 us however few destinations there
// are, as the claims do for some 8 million places.
static constexpr u32 BFS_WIN_WORDS = 1u << (BFS_WIN_LOG - 5);
static constexpr u32 BFS_EXT = 128;
static constexpr u32 BFS_WIN_GRID = 256;
static constexpr u32 BFS_WIN_EXT = 8;  // extents a wave of k_bfs_windows reads at a time
static constexpr u64 BFS_LISTED = 1ull << 22;  // places from which a level goes through lists

__device__ __forceinline__ bool bfs_listed(const BfsLists &ls, u64 ent) {
    return ls.list && (ent & BFS_PLACES) >= BFS_LISTED;
}
// extents a wave of the expansion may fill
__host__ __device__ __forceinline__ u64 bfs_extents(u64 nruns, u32 waves) {
    return (nruns + waves - 1) / waves * (BFS_RUN / BFS_EXT) + BFS_WINDOWS;
}

__global__ void k_bfs_init(u32 *levels, u32 V, u32 src, u32 *queue, BfsCtl *ctl, u32 *visited) {
    for (u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x; i < V; i += (u64)gridDim.x * blockDim.x)
        levels[i] = i == src ? 0u : INF_LEVEL;
    for (u64 w = (u64)blockIdx.x * blockDim.x + threadIdx.x; w < bfs_visited_words(V); w += (u64)gridDim.x * blockDim.x)
        visited[w] = w == (src >> 5) ? 1u << (src & 31) : 0u;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        queue[0] = src;
        for (int k = 0; k < 4; ++k) {
            ctl->ent[k] = 0;
            ctl->qn[k] = k == 0 ? 1u : 0u;
        }
        ctl->scanned = 0;
        ctl->depth = 0;
    }
}

static constexpr u32 FRONT_TPB = 1024;
static constexpr u32 FRONT_ITEMS = 4;  // vertices a lane of a sweep (one from the queue)

// Entries of a level's frontier, FRONT_TPB vertices at a time.  One atomic
// gives a chunk its entries and its places together, so places grow with
// entries whatever order the chunks come in.  A run's first place lies in one
// chunk, which finds the entry by binary search in LDS.  Bound: random reads
// of row_off (1.6 million vertices: 40 us).
__global__ __launch_bounds__(FRONT_TPB) void k_bfs_front(DevState d, u32 level, const u32 *__restrict__ q,
                                                          BfsCtl *__restrict__ ctl, u32 *__restrict__ off,
                                                          u32 *__restrict__ adj, u32 *__restrict__ runs,
                                                          BfsLists ls, u32 *__restrict__ levels, u64 *host) {
    constexpr u32 NW = FRONT_TPB / 64;
    __shared__ u32 s_off[FRONT_TPB * FRONT_ITEMS];
    __shared__ u32 s_n[NW], s_len[NW];
    __shared__ u64 s_base;
    const u32 tid = threadIdx.x, lane = lane_id(), w = tid >> 6;
    const u32 qn = ctl->qn[level & 3];
    if (blockIdx.x == 0 && tid == 0) {  // words of the level after the next: nothing reads or adds to them yet
        ctl->qn[(level + 2) & 3] = 0;
        ctl->ent[(level + 2) & 3] = 0;
        if (qn) ctl->depth = level + 1;
        __hip_atomic_store(host + 1, ctl->scanned, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        __hip_atomic_store(host + 2, (u64)(qn ? level + 1 : ctl->depth), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        __hip_atomic_store(host, (u64)(level + 1) << 32 | qn, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    // after a listed level the frontier is a bitmap, whose waves take vertices 64
    // at a time from regions far apart: neighboring hubs fall to different
    // workgroups
    const bool sweep = qn && level > 0 && bfs_listed(ls, ctl->ent[(level - 1) & 3]);
    const u32 blocks = (d.V + 63) / 64;
    const u32 items = sweep ? FRONT_ITEMS : 1;
    const u32 chunks = sweep ? (blocks + NW * FRONT_ITEMS - 1) / (NW * FRONT_ITEMS) : (qn + FRONT_TPB - 1) / FRONT_TPB;
    for (u32 c = blockIdx.x; c < chunks; c += gridDim.x) {
        u32 v[FRONT_ITEMS], lo[FRONT_ITEMS], len[FRONT_ITEMS];
        bool ok[FRONT_ITEMS];
#pragma unroll
        for (u32 k = 0; k < FRONT_ITEMS; ++k) {
            v[k] = 0;
            ok[k] = false;
            if (sweep) {
                const u64 i = ((u64)(k * NW + w) * chunks + c) * 64 + lane;
                v[k] = (u32)i;
                ok[k] = i < d.V && ((ls.fresh[i >> 5] >> (i & 31)) & 1u);
            } else if (k == 0) {
                const u64 i = (u64)c * FRONT_TPB + tid;
                ok[k] = i < qn;
                if (ok[k]) v[k] = q[i];
            }
        }
        u32 n = 0, sum = 0;
#pragma unroll
        for (u32 k = 0; k < FRONT_ITEMS; ++k) {
            u64 l = 0, h = 0;
            if (k < items && ok[k]) {
                slot_range(d, v[k], l, h);
                if (sweep) levels[v[k]] = level;
            }
            lo[k] = (u32)l;
            len[k] = (u32)(h - l);
        }
#pragma unroll
        for (u32 k = 0; k < FRONT_ITEMS; ++k) {
            n += len[k] != 0;
            sum += len[k];
        }
        const u32 ni = dpp_incl_scan32(n), li = dpp_incl_scan32(sum);
        if (lane == 63) {
            s_n[w] = ni;
            s_len[w] = li;
        }
        __syncthreads();
        u32 n0 = 0, l0 = 0, nt = 0, lt = 0;
        for (u32 x = 0; x < NW; ++x) {
            if (x == w) { n0 = nt; l0 = lt; }
            nt += s_n[x];
            lt += s_len[x];
        }
        if (tid == 0) s_base = nt ? atomicAdd((unsigned long long *)&ctl->ent[level & 3], ((u64)nt << 33) | lt) : 0;
        __syncthreads();
        const u32 eb = (u32)(s_base >> 33), pb = (u32)s_base;  // places: fewer than 2^32 slots
        u32 e = n0 + ni - n, o = l0 + li - sum;
#pragma unroll
        for (u32 k = 0; k < FRONT_ITEMS; ++k)
            if (len[k]) {
                s_off[e] = o;
                off[eb + e] = pb + o;
                adj[eb + e] = lo[k] - (pb + o);
                ++e;
                o += len[k];
            }
        __syncthreads();
        const u64 end = (u64)pb + lt;
        for (u64 r = ((u64)pb + BFS_RUN - 1) / BFS_RUN + tid; r * BFS_RUN < end; r += FRONT_TPB) {
            const u32 t = (u32)(r * BFS_RUN - pb);
            u32 x = 0, y = nt;
            while (y - x > 1) {
                const u32 m = (x + y) >> 1;
                if (s_off[m] <= t) x = m; else y = m;
            }
            runs[r] = eb + x;
        }
        __syncthreads();
    }
}

static constexpr u32 EXP_TPB = 512;
static constexpr u32 EXP_WAVES = EXP_TPB / 64;
static constexpr u32 EXP_Q = 2 * BFS_RUN;  // discovered vertices a wave holds: flushed before a run could outgrow them

__global__ __launch_bounds__(EXP_TPB) void k_bfs_expand(DevState d, u32 level, const u32 *__restrict__ off,
                                                         const u32 *__restrict__ adj, const u32 *__restrict__ runs,
                                                         u32 *__restrict__ levels, u32 *__restrict__ visited,
                                                         u32 *__restrict__ qnext, BfsCtl *__restrict__ ctl,
                                                         BfsLists ls) {
    __shared__ u32 s_adj[EXP_WAVES][BFS_RUN];
    __shared__ union {
        u32 q[EXP_Q];
        u32 b[BFS_WINDOWS][BFS_EXT + 64];  // a listed level's destinations by window
    } s_w[EXP_WAVES];
    __shared__ u32 s_first[EXP_WAVES][2 * BFS_ITEMS];  // a bit per place: an entry starts there
    __shared__ u32 s_n[EXP_WAVES], s_scanned[EXP_WAVES], s_base;
    const u32 lane = lane_id(), w = threadIdx.x >> 6;
    const u64 ent = ctl->ent[level & 3];
    const u64 total = ent & BFS_PLACES;
    const u32 nent = (u32)(ent >> 33);
    const u64 nruns = (total + BFS_RUN - 1) / BFS_RUN;
    const bool listed = bfs_listed(ls, ent);
    const u32 wave = blockIdx.x * EXP_WAVES + w;
    const u64 ext0 = wave * bfs_extents(nruns, gridDim.x * EXP_WAVES);  // this wave's extents
    u32 ne = 0, bn[BFS_WINDOWS] = {};
    // extent of the first `len` destinations of window x; the others move up
    auto put_extent = [&](u32 x, u32 len) {
        __builtin_amdgcn_wave_barrier();
        u32 *to = ls.list + (ext0 + ne) * BFS_EXT;
        for (u32 k = lane; k < len; k += 64) to[k] = s_w[w].b[x][k];
        const u32 rest = s_w[w].b[x][BFS_EXT + lane];
        if (lane == 0) ls.meta[ext0 + ne] = x << 8 | len;
        ++ne;
        __builtin_amdgcn_wave_barrier();
        s_w[w].b[x][lane] = rest;
        __builtin_amdgcn_wave_barrier();
    };
    const u64 le = ~0ull >> (63 - lane);  // this lane and those below
    const u32 Smask = (1u << d.log2S) - 1;
    const gu64 *keys = (const gu64 *)d.keys;
    u32 *next_n = &ctl->qn[(level + 1) & 3];
    u32 scanned = 0, n = 0;
    const u64 stride = (u64)gridDim.x * EXP_WAVES;
    u64 run = (u64)blockIdx.x * EXP_WAVES + w;
    // a run's first entries are loaded one run ahead
    u32 e0 = 0, p_off = 0, p_adj = 0;
    auto load = [&](u32 e) {
        const bool in = e < nent;
        p_off = in ? off[e] : ~0u;
        p_adj = in ? adj[e] : 0u;
    };
    if (run < nruns) {
        e0 = runs[run];
        load(e0 + lane);
    }
    for (; run < nruns; run += stride) {
        const bool more = run + stride < nruns;
        u32 e1 = 0;
        if (more) e1 = runs[run + stride];
        const u64 t0 = run * BFS_RUN;
        if (lane < 2 * BFS_ITEMS) s_first[w][lane] = 0;
        __builtin_amdgcn_wave_barrier();
        for (u32 k = lane;; k += 64) {
            // the first entry may begin before the run
            const bool in = e0 + k < nent && (u64)p_off < t0 + BFS_RUN;
            if (in) {
                const u32 at = p_off > t0 ? (u32)(p_off - t0) : 0u;
                s_adj[w][k] = p_adj;
                atomicOr(&s_first[w][at >> 5], 1u << (at & 31));
            }
            if (!__all(in)) break;
            load(e0 + k + 64);
        }
        __builtin_amdgcn_wave_barrier();
        u32 slot[BFS_ITEMS];
        bool ok[BFS_ITEMS];
        u32 before = 0;
#pragma unroll
        for (u32 i = 0; i < BFS_ITEMS; ++i) {
            const u64 m = (u64)s_first[w][2 * i + 1] << 32 | s_first[w][2 * i];
            const u64 t = t0 + i * 64 + lane;
            ok[i] = t < total;
            const u32 k = before + __popcll(m & le) - 1;
            slot[i] = ok[i] ? (u32)t + s_adj[w][k] : 0u;
            before += __popcll(m);
        }
        u32 live[BFS_ITEMS];
#pragma unroll
        for (u32 i = 0; i < BFS_ITEMS; ++i) live[i] = d.cnt[slot[i] >> d.log2S];  // slot 0 when !ok: in bounds
        e0 = e1;
        if (more) load(e1 + lane);
        u64 key[BFS_ITEMS];
#pragma unroll
        for (u32 i = 0; i < BFS_ITEMS; ++i) {
            u64 k = KEY_NONE;
            if (ok[i] && (slot[i] & Smask) < live[i]) k = keys[slot[i]];
            key[i] = k;
        }
        if (listed) {
#pragma unroll
            for (u32 i = 0; i < BFS_ITEMS; ++i) {
                const bool edge = key[i] != KEY_NONE;
                const u32 v = (u32)key[i], win = v >> BFS_WIN_LOG;
                scanned += edge;
#pragma unroll
                for (u32 x = 0; x < BFS_WINDOWS; ++x) {
                    const u64 m = __ballot(edge && win == x);
                    if (!m) continue;
                    if (edge && win == x) s_w[w].b[x][bn[x] + __popcll(m & le) - 1] = v;
                    bn[x] += (u32)__popcll(m);
                    if (bn[x] >= BFS_EXT) {
                        put_extent(x, BFS_EXT);
                        bn[x] -= BFS_EXT;
                    }
                }
            }
            continue;
        }
        u32 vw[BFS_ITEMS];
#pragma unroll
        for (u32 i = 0; i < BFS_ITEMS; ++i) {
            vw[i] = key[i] != KEY_NONE ? visited[(u32)key[i] >> 5] : ~0u;
            scanned += key[i] != KEY_NONE;
        }
        u32 old[BFS_ITEMS];
#pragma unroll
        for (u32 i = 0; i < BFS_ITEMS; ++i) {
            const u32 v = (u32)key[i], bit = 1u << (v & 31);
            old[i] = ~0u;
            if (!(vw[i] & bit)) old[i] = atomicOr(&visited[v >> 5], bit);
        }
#pragma unroll
        for (u32 i = 0; i < BFS_ITEMS; ++i) {
            const u32 v = (u32)key[i];
            const bool found = !((old[i] >> (v & 31)) & 1u);
            const u64 m = __ballot(found);
            if (found) {
                levels[v] = level + 1;
                s_w[w].q[n + __popcll(m & le) - 1] = v;
            }
            n += __popcll(m);
        }
        if (n > EXP_Q - BFS_RUN) {
            u32 base = 0;
            if (lane == 0) base = atomicAdd(next_n, n);
            base = (u32)__builtin_amdgcn_readfirstlane((int)base);
            __builtin_amdgcn_wave_barrier();
            for (u32 k = lane; k < n; k += 64) qnext[base + k] = s_w[w].q[k];
            __builtin_amdgcn_wave_barrier();
            n = 0;
        }
    }
    if (listed) {
#pragma unroll
        for (u32 x = 0; x < BFS_WINDOWS; ++x)
            if (bn[x]) put_extent(x, bn[x]);
        if (lane == 0) ls.ne[wave] = ne;
    }
    // what is left, with one atomic a workgroup
    scanned = wave_sum(scanned);
    if (lane == 0) {
        s_n[w] = n;
        s_scanned[w] = scanned;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        u32 sum = 0, sc = 0;
        for (u32 v = 0; v < EXP_WAVES; ++v) {
            const u32 c = s_n[v];
            s_n[v] = sum;
            sum += c;
            sc += s_scanned[v];
        }
        s_base = sum ? atomicAdd(next_n, sum) : 0u;
        if (sc) atomicAdd((unsigned long long *)&ctl->scanned, (u64)sc);
    }
    __syncthreads();
    const u32 base = s_base + s_n[w];
    for (u32 k = lane; k < n; k += 64) qnext[base + k] = s_w[w].q[k];
}

// Workgroup b: window b % windows, share b / windows of the expansion's waves.
__global__ __launch_bounds__(1024) void k_bfs_windows(u32 V, u32 level, u32 waves, const u32 *__restrict__ visited,
                                                       const BfsCtl *__restrict__ ctl, BfsLists ls) {
    extern __shared__ u32 win[];
    const u64 ent = ctl->ent[level & 3];
    if (!bfs_listed(ls, ent)) return;
    const u32 tid = threadIdx.x, lane = lane_id();
    const u32 x = blockIdx.x % ls.windows, share = blockIdx.x / ls.windows, shares = gridDim.x / ls.windows;
    const u64 words = bfs_visited_words(V), w0 = (u64)x * BFS_WIN_WORDS;
    for (u32 i0 = tid; i0 < BFS_WIN_WORDS; i0 += 1024 * 16) {
        u32 r[16];
#pragma unroll
        for (u32 k = 0; k < 16; ++k) {
            const u64 i = w0 + i0 + k * 1024;
            r[k] = visited[i < words ? i : 0];
            if (i >= words) r[k] = 0;
        }
#pragma unroll
        for (u32 k = 0; k < 16; ++k) win[i0 + k * 1024] = r[k];
    }
    __syncthreads();
    const u64 epw = bfs_extents(((ent & BFS_PLACES) + BFS_RUN - 1) / BFS_RUN, waves);
    auto mark = [&](u32 v, bool ok) {
        const u32 i = (v >> 5) & (BFS_WIN_WORDS - 1), bit = 1u << (v & 31);
        if (ok && !(win[i] & bit)) atomicOr(&win[i], bit);
    };
    // (shares beyond the last whole one have none)
    for (u32 wv = share < shares ? share + (tid >> 6) * shares : waves; wv < waves; wv += 16 * shares) {
        const u32 ne = ls.ne[wv];
        for (u32 e0 = 0; e0 < ne; e0 += 64) {
            const u32 m = e0 + lane < ne ? ls.meta[wv * epw + e0 + lane] : ~0u;
            u64 mine = __ballot(m >> 8 == x);
            while (mine) {
                u32 v[BFS_WIN_EXT][2], len[BFS_WIN_EXT];
#pragma unroll
                for (u32 k = 0; k < BFS_WIN_EXT; ++k) {
                    const u32 l = mine ? (u32)__builtin_ctzll(mine) : 0u;
                    len[k] = mine ? (u32)__builtin_amdgcn_readlane((int)m, (int)l) & 0xFFu : 0u;
                    mine &= mine - 1;
                    const u32 *from = ls.list + (wv * epw + e0 + l) * BFS_EXT;
#pragma unroll
                    for (u32 h = 0; h < 2; ++h) v[k][h] = lane + 64 * h < len[k] ? from[lane + 64 * h] : 0u;
                }
#pragma unroll
                for (u32 k = 0; k < BFS_WIN_EXT; ++k)
#pragma unroll
                    for (u32 h = 0; h < 2; ++h) mark(v[k][h], lane + 64 * h < len[k]);
            }
        }
    }
    __syncthreads();
    for (u32 i = tid; i < BFS_WIN_WORDS; i += 1024) ls.part[(u64)blockIdx.x * BFS_WIN_WORDS + i] = win[i];
}

// A thread a word: what the workgroups' windows have beyond the bitmap is the
// next frontier.
__global__ __launch_bounds__(256) void k_bfs_merge(u32 V, u32 level, u32 *__restrict__ visited,
                                                    BfsCtl *__restrict__ ctl, BfsLists ls) {
    if (!bfs_listed(ls, ctl->ent[level & 3])) return;
    const u64 words = bfs_visited_words(V);
    const u32 shares = BFS_WIN_GRID / ls.windows;
    for (u64 i = (u64)blockIdx.x * 256 + threadIdx.x; i < words; i += (u64)gridDim.x * 256) {
        const u32 x = (u32)(i >> (BFS_WIN_LOG - 5));
        const u32 *from = ls.part + (u64)x * BFS_WIN_WORDS + (i & (BFS_WIN_WORDS - 1));
        u32 now = 0;
#pragma unroll 8
        for (u32 s = 0; s < shares; ++s) now |= from[(u64)s * ls.windows * BFS_WIN_WORDS];
        const u32 was = visited[i];
        ls.fresh[i] = now & ~was;
        if (now & ~was) {
            visited[i] = now | was;
            ctl->qn[(level + 1) & 3] = 1;  // a listed level only tells none from some
        }
    }
}

hipError_t bfs_init(u32 *levels, u32 V, u32 src, u32 *queue, u32 *ctl, u32 *visited, hipStream_t st) {
    k_bfs_init<<<grid_for(V, 256, 16384), 256, 0, st>>>(levels, V, src, queue, (BfsCtl *)ctl, visited);
    return hipGetLastError();
}

u64 bfs_run_words(u64 slots) { return slots / BFS_RUN + 2; }

// Default expansion grid: every workgroup resident at once (compute units x
// workgroups per CU that fit), so the runs are shared out in one round.
static u32 bfs_expand_grid() {
    static std::atomic<u32> cached[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 1024;
    u32 g = cached[dev].load(std::memory_order_relaxed);
    if (g) return g;
    int cus = 0, per_cu = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_bfs_expand, EXP_TPB, 0) != hipSuccess || cus <= 0 ||
        per_cu <= 0)
        return 1024;
    g = (u32)(cus * per_cu);
    cached[dev].store(g, std::memory_order_relaxed);
    return g;
}

u32 bfs_list_waves() { return bfs_expand_grid() * EXP_WAVES; }
u64 bfs_list_extents(u64 slots, u32 waves) { return bfs_extents((slots + BFS_RUN - 1) / BFS_RUN, waves) * waves; }
u64 bfs_list_words(u64 extents) { return extents * BFS_EXT; }
u64 bfs_part_words() { return (u64)BFS_WIN_GRID * BFS_WIN_WORDS; }

hipError_t bfs_level(const DevState &d, const u32 *q, u32 *off, u32 *adj, u32 *runs, u32 *levels, u32 *visited,
                     u32 level, u32 *qnext, u32 *ctl, const BfsLists &ls, u64 *host, u32 expand_grid, hipStream_t st) {
    BfsCtl *c = (BfsCtl *)ctl;
    const u32 grid = expand_grid ? expand_grid : bfs_expand_grid();
    k_bfs_front<<<grid_for(d.V, FRONT_TPB, 512), FRONT_TPB, 0, st>>>(d, level, q, c, off, adj, runs, ls, levels,
                                                                    host);
    k_bfs_expand<<<grid, EXP_TPB, 0, st>>>(d, level, off, adj, runs, levels, visited, qnext, c, ls);
    if (ls.list) {
        k_bfs_windows<<<BFS_WIN_GRID, 1024, BFS_WIN_WORDS * sizeof(u32), st>>>(d.V, level, grid * EXP_WAVES, visited, c,
                                                                            ls);
        k_bfs_merge<<<grid_for(bfs_visited_words(d.V), 256, 1024), 256, 0, st>>>(d.V, level, visited, c, ls);
    }
    return hipGetLastError();
}

// ------------------------------------------------------------- PageRank
//
// nvGraph's formulation (include/pagerank.hxx:66-88): with a = alpha on
// dangling vertices and 1-alpha elsewhere,
//     pr' = alpha * A^T (pr / outdeg) + (sum_u a_u pr_u) / n,
// iterated from the uniform vector; here until the L1 change is below the
// tolerance or max_iter, then normalised by the L1 norm.
//
// Values and accumulation are FP32.  Every accumulation is compensated: an
// atomic add returns the old value, the thread recomputes the sum and its
// exact rounding error (TwoSum, Knuth TAOCP vol. 2, 4.2.2) and adds that
// error to a second FP32 accumulator, so a hub that receives millions of
// contributions keeps the precision of its partial sums.  The push goes to
// one accumulator copy per XCD (the XCD read from the hardware register), so
// the atomics of a hub are spread over eight addresses; the copies are
// summed (Kahan) when the iteration finishes.

static constexpr u32 PR_COPIES = 8;  // accumulator copies, one per XCD

// hi += x with the rounding error of that add going to lo
__device__ __forceinline__ void atomic_add2(float *hi, float *lo, float x) {
    const float old = atomicAdd(hi, x);
    const float s = old + x;
    const float bp = s - old;
    const float e = (old - (s - bp)) + (x - bp);
    if (e != 0.f) atomicAdd(lo, e);
}

// sum over a workgroup of PR_TPB threads (every thread gets it); tmp holds
// PR_TPB / 64 floats of LDS
static constexpr u32 PR_TPB = 256;
__device__ __forceinline__ float block_sum(float v, float *tmp) {
    v = wave_sum(v);
    __syncthreads();  // tmp may still be read from a previous call
    if (lane_id() == 0) tmp[threadIdx.x >> 6] = v;
    __syncthreads();
    float t = 0.f;
#pragma unroll
    for (u32 w = 0; w < PR_TPB / 64; ++w) t += tmp[w];
    return t;
}

// red layout (floats): [0,1] dangling mass hi/lo, [2,3] sum hi/lo,
// [4,5] L1 change hi/lo
static constexpr u32 PR_RED = 8;

// out-degree of every row from marker ranks (rank = live slots before)
__global__ void k_outdeg(DevState d, const u32 *__restrict__ gpre, u32 *__restrict__ outdeg) {
    const u32 Smask = (1u << d.log2S) - 1;
    for (u64 r = (u64)blockIdx.x * blockDim.x + threadIdx.x; r < d.V; r += (u64)gridDim.x * blockDim.x) {
        u64 hs = d.row_off[r + 1];
        u64 rank_hi = (u64)gpre[hs >> d.log2S] + (hs & Smask);
        u64 rank_lo = 0;
        if (r > 0) {
            u64 ls = d.row_off[r];
            rank_lo = (u64)gpre[ls >> d.log2S] + (ls & Smask) + 1;
        }
        outdeg[r] = (u32)(rank_hi - rank_lo);
    }
}

// contributions pr/outdeg, the dangling mass, and cleared accumulators
// (PR_COPIES hi copies, then PR_COPIES lo copies, V floats each)
__global__ __launch_bounds__(PR_TPB) void k_pr_prep(const float *__restrict__ pr, const u32 *__restrict__ outdeg, u32 V, float *__restrict__ c,
                          float *__restrict__ acc, u64 nclear, float *__restrict__ red) {
    float dang = 0.f;
    const u64 stride = (u64)gridDim.x * blockDim.x;
    for (u64 u = (u64)blockIdx.x * blockDim.x + threadIdx.x; u < V; u += stride) {
        u32 od = outdeg[u];
        float p = pr[u];
        c[u] = od ? p / (float)od : 0.f;
        if (!od) dang += p;
    }
    for (u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x; i < nclear; i += stride) acc[i] = 0.f;
    __shared__ float tmp[PR_TPB / 64];
    dang = block_sum(dang, tmp);
    if (threadIdx.x == 0 && dang != 0.f) atomic_add2(&red[0], &red[1], dang);
}

__global__ void k_pr_push(DevState d, const float *__restrict__ c, float *__restrict__ acc) {
    const u64 W = nseg_of(d) << d.log2S;
    const u64 V = d.V;
    float *hi = acc + (u64)xcc_id() * V;
    float *lo = hi + PR_COPIES * V;
    for (u64 t = (u64)blockIdx.x * blockDim.x + threadIdx.x; t < W; t += (u64)gridDim.x * blockDim.x) {
        u64 key = d.keys[t];
        if (key == KEY_NONE || is_marker(key)) continue;
        const u32 v = (u32)key;
        atomic_add2(&hi[v], &lo[v], c[(u32)(key >> 32)]);
    }
}

// pr' = alpha*acc + (alpha*dangling + (1-alpha)*sum(pr)) / n; L1 change and sum
__global__ __launch_bounds__(PR_TPB) void k_pr_finish(const float *__restrict__ acc, const float *__restrict__ pr, float *__restrict__ out,
                            u32 V, float alpha, const float *__restrict__ red_in, float *__restrict__ red_out) {
    const float dang = red_in[0] + red_in[1];
    const float sum_in = red_in[2] + red_in[3];
    const float gamma = (alpha * dang + (1.f - alpha) * sum_in) / (float)V;
    float dl = 0.f, sum = 0.f;
    for (u64 v = (u64)blockIdx.x * blockDim.x + threadIdx.x; v < V; v += (u64)gridDim.x * blockDim.x) {
        // Kahan sum of the copies, lo parts first (the small terms)
        float a = 0.f, comp = 0.f;
#pragma unroll
        for (u32 k = 2 * PR_COPIES; k-- > 0;) {
            float y = acc[(u64)k * V + v] - comp;
            float t = a + y;
            comp = (t - a) - y;
            a = t;
        }
        float p = alpha * a + gamma;
        out[v] = p;
        dl += fabsf(p - pr[v]);
        sum += p;
    }
    __shared__ float tmp[PR_TPB / 64];
    dl = block_sum(dl, tmp);
    sum = block_sum(sum, tmp);
    if (threadIdx.x == 0) {
        atomic_add2(&red_out[4], &red_out[5], dl);
        atomic_add2(&red_out[2], &red_out[3], sum);
    }
}

__global__ void k_pr_init(float *pr, u32 V, float *red) {
    for (u64 v = (u64)blockIdx.x * blockDim.x + threadIdx.x; v < V; v += (u64)gridDim.x * blockDim.x)
        pr[v] = 1.f / (float)V;
    if (blockIdx.x == 0 && threadIdx.x < PR_RED) red[threadIdx.x] = threadIdx.x == 2 ? 1.f : 0.f;  // sum = 1
}

__global__ void k_pr_reset(float *red_next) {
    if (threadIdx.x < PR_RED) red_next[threadIdx.x] = 0.f;
}

__global__ void k_pr_scale(float *pr, u32 V, const float *red) {
    const float inv = 1.f / (red[2] + red[3]);
    for (u64 v = (u64)blockIdx.x * blockDim.x + threadIdx.x; v < V; v += (u64)gridDim.x * blockDim.x) pr[v] *= inv;
}

hipError_t pr_outdeg(const DevState &d, u32 *gpre, u32 *scan_scratch, u32 *outdeg, hipStream_t st) {
    (void)device_excl_scan(d.cnt, nseg_of(d), gpre, scan_scratch, st);
    k_outdeg<<<grid_for(d.V, 256, 16384), 256, 0, st>>>(d, gpre, outdeg);
    return hipGetLastError();
}

u64 pr_acc_floats(u32 V) { return 2ull * PR_COPIES * V; }
u32 pr_red_floats() { return PR_RED; }

hipError_t pr_init(float *pr, u32 V, float *red, hipStream_t st) {
    k_pr_init<<<grid_for(V, 256, 16384), 256, 0, st>>>(pr, V, red);
    return hipGetLastError();
}

// one iteration: pr -> out; red holds (dangling, sum) of pr on entry and
// (dangling of out, sum of out, L1 change) on exit in red_next
hipError_t pr_iterate(const DevState &d, const float *pr, const u32 *outdeg, float *c, float *acc, float *out,
                      float alpha, float *red, float *red_next, hipStream_t st) {
    const u32 V = d.V;
    k_pr_reset<<<1, 64, 0, st>>>(red_next);
    k_pr_prep<<<grid_for(pr_acc_floats(V), PR_TPB, PR_GRID), PR_TPB, 0, st>>>(pr, outdeg, V, c, acc, pr_acc_floats(V),
                                                                         red);
    k_pr_push<<<grid_for(nseg_of(d) << d.log2S, 256, 65536), 256, 0, st>>>(d, c, acc);
    k_pr_finish<<<grid_for(V, PR_TPB, PR_GRID), PR_TPB, 0, st>>>(acc, pr, out, V, alpha, red, red_next);
    return hipGetLastError();
}

hipError_t pr_scale(float *pr, u32 V, const float *red, hipStream_t st) {
    k_pr_scale<<<grid_for(V, 256, 16384), 256, 0, st>>>(pr, V, red);
    return hipGetLastError();
}

// ------------------------------------------------- binned edges (PageRank)
//
// The push above sends every edge's contribution to a random destination in
// HBM: one returning atomic per edge on a 64 MB vector, which no L2 holds.
// Binning the edges by destination (propagation blocking: Beamer, Asanovic,
// Patterson, "Reducing PageRank communication via propagation blocking",
// IPDPS 2017) keeps the random adds in LDS.  The graph does not change during
// a call, so the edges are binned once, not their contributions every
// iteration:
//   count    the slot array is cut into parts of 2^part_log slots; the edges
//            of each (bin, part) are counted and the bin-major exclusive scan
//            of the counts fixes where each goes;
//   bin      each part's workgroup writes its edges into its bins' runs, one
//            word each: source relative to the part's first row, destination
//            relative to the bin.  Runs are padded to groups of words and each
//            group has the part's first row beside it.  A group is PB_CHUNK
//            words, or one word, without padding, where runs are short or their
//            padding would pass 32-bit offsets (pr_bins_plan);
// and an iteration is one kernel (k_pr_iter): a workgroup takes a chunk of a
// bin's edges, reads the source's contribution (a run's sources ascend, so
// the lanes of a wave share lines and the workgroups of an XCD sweep the
// vector together), adds it to the destination in LDS, and finishes the bin's
// vertices: rank, next contribution, dangling mass, L1 change.

static constexpr u32 PB_BIN_LOG = 13;  // destination vertices per bin
static constexpr u32 PB_BIN = 1u << PB_BIN_LOG;
static constexpr u32 PB_MAX_BINS = 16384;  // LDS cursors of the bin pass: 64 KB
static constexpr u32 PB_TPB = 1024;
static constexpr u32 PB_ITEMS = 8;
static constexpr u32 PB_MAX_PART_LOG = 18;         // slots per part (log2): see pb_word
static constexpr u32 PB_MAX_PARTS = 1u << (32 - PB_MAX_PART_LOG);
static constexpr u32 PB_CHUNK = 8;                // words per group and staged chunk (32 B, one HBM sector)
static constexpr u32 PB_STAGE_MAX_BINS = 2048;    // staged bin pass LDS: 40 B per bin
static constexpr u32 PBS_TPB = 512;               // staged bin pass: two workgroups per CU (80 KB LDS each)
static constexpr u32 PBS_ITEMS = 8;
static constexpr u32 PRI_TPB = 1024;              // iteration: two workgroups of 64 KB of LDS fill a CU's waves
static constexpr u32 PRI_ITEMS = 8;

// Lanes holding a live edge of the same bin form runs (adjacent lanes; keys
// are sorted, so a row's edges to one bin are adjacent).  Returns the lane
// that leads this lane's run, and for a leader the run's length in `len`.
__device__ __forceinline__ u32 bin_run(bool valid, u32 bin, u32 &len) {
    const u32 lane = lane_id();
    const u32 bb = valid ? bin : 0xFFFFFFFFu;
    const u32 prev = __shfl_up(bb, 1, 64);
    const u32 next = __shfl_down(bb, 1, 64);
    const u64 starts = __ballot(valid && (lane == 0 || prev != bb));
    const u64 ends = __ballot(valid && (lane == 63 || next != bb));
    // the sentinel bits keep both masks non-zero; a valid lane's own run
    // bits are the highest start at or below it and the lowest end at or above
    const u32 lead = 63 - (u32)__clzll((starts & ((2ull << lane) - 1ull)) | 1ull);
    const u32 end = (u32)__builtin_ctzll((ends & ~((1ull << lane) - 1ull)) | (1ull << 63));
    len = end - lane + 1;
    return lead;
}

// PB_ITEMS slots t0 + i * PB_TPB + threadIdx.x of a part ending at p1: the
// live ones' keys, KEY_NONE elsewhere.  All segment counts are loaded first
// (clamped, unconditional), then the keys with exec-masked global loads, so a
// thread has PB_ITEMS loads in flight per phase and dead lines are not read.
template <u32 TPB = PB_TPB, u32 ITEMS = PB_ITEMS>
__device__ __forceinline__ void pb_load(const DevState &d, u64 t0, u64 p1, u64 (&key)[ITEMS]) {
    const u32 Smask = (1u << d.log2S) - 1;
    const gu64 *keys = (const gu64 *)d.keys;
    u32 live[ITEMS];
#pragma unroll
    for (u32 i = 0; i < ITEMS; ++i) {
        const u64 t = t0 + (u64)i * TPB + threadIdx.x;
        live[i] = d.cnt[(t < p1 ? t : p1 - 1) >> d.log2S];
    }
#pragma unroll
    for (u32 i = 0; i < ITEMS; ++i) {
        const u64 t = t0 + (u64)i * TPB + threadIdx.x;
        u64 k = KEY_NONE;
        if (t < p1 && (u32)(t & Smask) < live[i]) k = keys[t];
        key[i] = k;
    }
}

__device__ __forceinline__ bool pb_edge(u64 key) { return key != KEY_NONE && !is_marker(key); }
// An edge in its bin: its source relative to the part's first row, and its
// destination within the bin.  Every row has its marker in a slot, so a part
// of 2^18 slots holds edges of at most 2^18 + 1 rows: 19 bits over the bin's
// 13, and no edge gives the padding word.
static constexpr u32 PB_PAD = 0xFFFFFFFFu;
static_assert((1ull << PB_MAX_PART_LOG) + 1 < (1ull << (32 - PB_BIN_LOG)) - 1, "a source fits above the destination");
__device__ __forceinline__ u32 pb_word(u64 key, u32 row0) {
    return (((u32)(key >> 32) - row0) << PB_BIN_LOG) | ((u32)key & (PB_BIN - 1));
}

// the row that slot p lies in (rows whose marker slots are below p), by one
// whole wave: 64 pivots a step
__device__ __forceinline__ u32 row_of_slot(const DevState &d, u64 p) {
    const u32 lane = lane_id();
    u32 lo = 0, hi = d.V;  // first r with row_off[r + 1] >= p, V if none
    while (lo < hi) {
        const u32 step = (hi - lo + 63) / 64;
        const u64 q = (u64)lo + (u64)lane * step;
        const u64 below = __ballot(q < hi && d.row_off[q + 1] < p);  // a prefix of the lanes
        const u32 c = (u32)__popcll(below);
        if (c == 0) return lo;
        const u32 nlo = lo + (c - 1) * step + 1;
        hi = min((u64)lo + (u64)c * step, (u64)hi);
        lo = nlo;
    }
    return lo;
}

// pb_load in separate phases, for a loop that prefetches its next step:
// the segment counts, then the keys (after the counts)
template <u32 TPB, u32 ITEMS>
__device__ __forceinline__ void pb_counts(const DevState &d, u64 t0, u64 p1, u32 (&live)[ITEMS]) {
#pragma unroll
    for (u32 i = 0; i < ITEMS; ++i) {
        const u64 t = t0 + (u64)i * TPB + threadIdx.x;
        live[i] = d.cnt[(t < p1 ? t : p1 - 1) >> d.log2S];
    }
}

template <u32 TPB, u32 ITEMS>
__device__ __forceinline__ void pb_keys(const DevState &d, u64 t0, u64 p1, const u32 (&live)[ITEMS],
                                        u64 (&key)[ITEMS]) {
    const u32 Smask = (1u << d.log2S) - 1;
    const gu64 *keys = (const gu64 *)d.keys;
#pragma unroll
    for (u32 i = 0; i < ITEMS; ++i) {
        const u64 t = t0 + (u64)i * TPB + threadIdx.x;
        u64 k = KEY_NONE;
        if (t < p1 && (u32)(t & Smask) < live[i]) k = keys[t];
        key[i] = k;
    }
}

// count[bin * P + part] = live edges of `part` into `bin`, rounded up to whole
// groups (and clears the iterations' reductions)
__global__ __launch_bounds__(PB_TPB) void k_pb_count(DevState d, u32 part_log, u32 P, u32 NB, u32 group,
                                                     u32 *__restrict__ count, PrSlot *slots) {
    extern __shared__ u32 pb_lds[];
    if (blockIdx.x == 0 && threadIdx.x < PR_SLOTS) slots[threadIdx.x] = PrSlot{0.0, 0.0, 0.0};
    for (u32 b = threadIdx.x; b < NB; b += PB_TPB) pb_lds[b] = 0;
    __syncthreads();
    const u64 W = nseg_of(d) << d.log2S;
    const u64 p0 = (u64)blockIdx.x << part_log;
    const u64 p1 = min(W, p0 + (1ull << part_log));
    for (u64 t0 = p0; t0 < p1; t0 += (u64)PB_TPB * PB_ITEMS) {
        u64 key[PB_ITEMS];
        pb_load(d, t0, p1, key);
#pragma unroll
        for (u32 i = 0; i < PB_ITEMS; ++i) {
            const bool valid = pb_edge(key[i]);
            const u32 bin = (u32)key[i] >> PB_BIN_LOG;
            u32 len;
            const u32 lead = bin_run(valid, bin, len);
            if (valid && lead == lane_id()) atomicAdd(&pb_lds[bin], len);
        }
    }
    __syncthreads();
    for (u32 b = threadIdx.x; b < NB; b += PB_TPB)
        count[(u64)b * P + blockIdx.x] = (pb_lds[b] + group - 1) & ~(group - 1);
}

// words[off[bin * P + part] + rank] = pb_word(edge)
// Phases per step: all key loads, all cursor adds, then the stores, so each
// thread keeps PB_ITEMS loads in flight at a time.  G: words of a group (of
// one, the row stands beside its word).
template <u32 G>
__global__ __launch_bounds__(PB_TPB) void k_pb_bin(DevState d, u32 part_log, u32 P, u32 NB, const u32 *__restrict__ off,
                                                   u32 *__restrict__ words, u32 *__restrict__ rows, u64 room) {
    extern __shared__ u32 pb_lds[];
    __shared__ u32 s_row0;
    for (u32 b = threadIdx.x; b < NB; b += PB_TPB) pb_lds[b] = off[(u64)b * P + blockIdx.x];
    if (threadIdx.x < 64) {
        const u32 r = row_of_slot(d, (u64)blockIdx.x << part_log);
        if (threadIdx.x == 0) s_row0 = r;
    }
    __syncthreads();
    const u32 row0 = s_row0;
    const u64 W = nseg_of(d) << d.log2S;
    const u64 p0 = (u64)blockIdx.x << part_log;
    const u64 p1 = min(W, p0 + (1ull << part_log));
    const u32 lane = lane_id();
    for (u64 t0 = p0; t0 < p1; t0 += (u64)PB_TPB * PB_ITEMS) {
        u64 key[PB_ITEMS];
        pb_load(d, t0, p1, key);
        u32 lead[PB_ITEMS], base[PB_ITEMS];
#pragma unroll
        for (u32 i = 0; i < PB_ITEMS; ++i) {
            const bool valid = pb_edge(key[i]);
            u32 len;
            lead[i] = bin_run(valid, (u32)key[i] >> PB_BIN_LOG, len);
            base[i] = 0;
            if (valid && lead[i] == lane) base[i] = atomicAdd(&pb_lds[(u32)key[i] >> PB_BIN_LOG], len);
            if (!valid) lead[i] = lane;
        }
#pragma unroll
        for (u32 i = 0; i < PB_ITEMS; ++i) {
            const u32 b0 = __shfl(base[i], lead[i], 64);
            const u64 pos = (u64)b0 + (lane - lead[i]);
            if (pb_edge(key[i]) && pos < room) {
                if (G == 1) {
                    ((uint2 *)words)[pos] = make_uint2(pb_word(key[i], row0), row0);
                } else {
                    words[pos] = pb_word(key[i], row0);
                    if (pos % G == 0) rows[pos / G] = row0;
                }
            }
        }
    }
    __syncthreads();
    // a run's last group is filled up
    for (u32 b = threadIdx.x; b < NB; b += PB_TPB)
        for (u64 pos = pb_lds[b]; pos % G && pos < room; ++pos) words[pos] = PB_PAD;
}

// Staged form of the bin pass (bins <= PB_STAGE_MAX_BINS): a bin's words
// reach HBM only as whole aligned chunks of PB_CHUNK words (32 B), so no
// partly written line is evicted from L2 and written twice.  Per step, phase by phase:
//   1. ranks: each edge takes rank r on its bin's fill counter (run-aggregated);
//   2. r < PB_CHUNK goes to the bin's LDS chunk, r inside a further complete
//      chunk straight to HBM (a run's lanes are adjacent: coalesced), the
//      rest waits;
//   3. full LDS chunks are written out and the bin's position advances;
//   4. the waiting edges start the next LDS chunk.
// At the end of the part each bin's last chunk is filled up with PB_PAD.
__global__ __launch_bounds__(PBS_TPB) void k_pb_bin_staged(DevState d, u32 part_log, u32 P, u32 NB,
                                                          const u32 *__restrict__ off,
                                                          u32 *__restrict__ words, u32 *__restrict__ rows, u64 room) {
    extern __shared__ uint4 pb_stage[];
    __shared__ u32 s_row0;
    u32 *buf = (u32 *)pb_stage;                           // NB * PB_CHUNK staged words
    u32 *fill = buf + (u64)NB * PB_CHUNK;                 // staged words per bin (< PB_CHUNK between steps)
    u32 *gpos = fill + NB;                                // word index of the bin's LDS chunk in HBM
    if (threadIdx.x < 64) {
        const u32 r = row_of_slot(d, (u64)blockIdx.x << part_log);
        if (threadIdx.x == 0) s_row0 = r;
    }
    for (u32 b = threadIdx.x; b < NB; b += PBS_TPB) {
        fill[b] = 0;
        gpos[b] = off[(u64)b * P + blockIdx.x];
    }
    __syncthreads();
    const u32 row0 = s_row0;
    const u64 W = nseg_of(d) << d.log2S;
    const u64 p0 = (u64)blockIdx.x << part_log;
    const u64 p1 = min(W, p0 + (1ull << part_log));
    const u32 lane = lane_id();
    // the next step's loads go out one phase ahead of their use: counts
    // during the ranking, keys during the placement (the barriers wait for
    // LDS only)
    constexpr u64 STEP = (u64)PBS_TPB * PBS_ITEMS;
    u32 live_n[PBS_ITEMS];
    u64 key_n[PBS_ITEMS];
    pb_counts<PBS_TPB, PBS_ITEMS>(d, p0, p1, live_n);
    pb_keys<PBS_TPB, PBS_ITEMS>(d, p0, p1, live_n, key_n);
    for (u64 t0 = p0; t0 < p1; t0 += STEP) {
        u64 key[PBS_ITEMS];
#pragma unroll
        for (u32 i = 0; i < PBS_ITEMS; ++i) key[i] = key_n[i];
        const bool more = t0 + STEP < p1;  // uniform
        if (more) pb_counts<PBS_TPB, PBS_ITEMS>(d, t0 + STEP, p1, live_n);
        u32 rank[PBS_ITEMS];
#pragma unroll
        for (u32 i = 0; i < PBS_ITEMS; ++i) {
            const bool valid = pb_edge(key[i]);
            u32 len;
            u32 lead = bin_run(valid, (u32)key[i] >> PB_BIN_LOG, len);
            u32 base = 0;
            if (valid && lead == lane) base = atomicAdd(&fill[(u32)key[i] >> PB_BIN_LOG], len);
            if (!valid) lead = lane;
            rank[i] = __shfl(base, lead, 64) + (lane - lead);
        }
        __syncthreads();
        if (more) pb_keys<PBS_TPB, PBS_ITEMS>(d, t0 + STEP, p1, live_n, key_n);
        u32 full[PBS_ITEMS];
        u32 wait = 0;
#pragma unroll
        for (u32 i = 0; i < PBS_ITEMS; ++i) {
            full[i] = 0;
            if (!pb_edge(key[i])) continue;
            const u32 bin = (u32)key[i] >> PB_BIN_LOG;
            const u32 word = pb_word(key[i], row0);
            full[i] = fill[bin] & ~(PB_CHUNK - 1);
            if (rank[i] < PB_CHUNK) {
                buf[bin * PB_CHUNK + rank[i]] = word;
            } else if (rank[i] < full[i]) {
                const u64 pos = (u64)gpos[bin] + rank[i];
                if (pos < room) {
                    words[pos] = word;
                    if (pos % PB_CHUNK == 0) rows[pos / PB_CHUNK] = row0;
                }
            } else {
                wait |= 1u << i;
            }
        }
        __syncthreads();
        for (u32 b = threadIdx.x; b < NB; b += PBS_TPB) {
            const u32 F = fill[b];
            if (F >= PB_CHUNK) {
                const u64 pos = gpos[b];
                if (pos + PB_CHUNK <= room) {
                    const uint4 *src = (const uint4 *)(buf + b * PB_CHUNK);
                    uint4 *dst = (uint4 *)(words + pos);
#pragma unroll
                    for (u32 k = 0; k < PB_CHUNK / 4; ++k) dst[k] = src[k];
                    rows[pos / PB_CHUNK] = row0;
                }
                gpos[b] = (u32)(pos + (F & ~(PB_CHUNK - 1)));
                fill[b] = F & (PB_CHUNK - 1);
            }
        }
        __syncthreads();
#pragma unroll
        for (u32 i = 0; i < PBS_ITEMS; ++i)
            if (wait & (1u << i)) {
                const u32 bin = (u32)key[i] >> PB_BIN_LOG;
                buf[bin * PB_CHUNK + (rank[i] - full[i])] = pb_word(key[i], row0);
            }
        // the next step's ranks read fill (settled before the last barrier);
        // its LDS chunk writes come after its first barrier
    }
    __syncthreads();
    for (u32 b = threadIdx.x; b < NB; b += PBS_TPB) {
        const u32 F = fill[b];
        const u64 pos = gpos[b];
        if (F && pos + PB_CHUNK <= room) {
            for (u32 k = 0; k < PB_CHUNK; ++k) words[pos + k] = k < F ? buf[b * PB_CHUNK + k] : PB_PAD;
            rows[pos / PB_CHUNK] = row0;
        }
    }
}

// chunks before each bin (cb[NB]: all): ceil(words of the bin / chunk), at
// least one, so that every bin has a workgroup to finish its vertices; and
// before it, the chunks of bins of several (their partial sums): cb[NB + 1 + b]
__global__ __launch_bounds__(1024) void k_pb_chunks(const u32 *__restrict__ off, u32 P, u32 NB, u32 chunk,
                                                    u32 *__restrict__ cb) {
    __shared__ u64 tmp[1024 / 64 + 1];
    u64 carry = 0;
    for (u32 b0 = 0; b0 < NB; b0 += 1024) {
        const u32 b = b0 + threadIdx.x;
        u64 v = 0;
        if (b < NB) {
            const u32 len = off[(u64)(b + 1) * P] - off[(u64)b * P];
            const u32 n = len ? (len - 1) / chunk + 1 : 1u;
            v = n | (n > 1 ? (u64)n << 32 : 0ull);
        }
        u64 tot;
        const u64 ex = block_excl_scan<1024, u64>(v, tot, tmp) + carry;
        if (b < NB) {
            cb[b] = (u32)ex;
            cb[NB + 1 + b] = (u32)(ex >> 32);
        }
        carry += tot;
    }
    if (threadIdx.x == 0) cb[NB] = (u32)carry;
}

// Sums of contributions are kept in 64 bits, in floating or in fixed point of
// PR_FIX fractional bits.  FP64 takes a contribution of any size whole.  Fixed
// point does so from 2^(23 - PR_FIX) on, and then its adds are exact; a sum stays
// below 2, as the ranks of a vector sum to 1 (the recurrence keeps it).  LDS adds
// integers faster where many lanes meet on one address, until the reads of the
// contributions hide that: 10^7 edges on 6*10^5 vertices 78 us an iteration, FP64
// 94; 3.4*10^7 on 2^21 104 and 109; 6.4*10^7 on 2^22 the same.  So integers take the
// sums where no contribution can be smaller (pr_fits_fixed).
static constexpr u32 PR_FIX = 63;
// A rank is at least an equal share of (1 - alpha) of the mass, a contribution
// at least that over the largest out-degree; a hundredth of it is more than
// roundings take.
bool pr_fits_fixed(u32 V, u64 degree, float alpha) {
    return (1.0 - (double)alpha) * 0.99 * (double)(1ull << (PR_FIX - 23)) >= (double)V * (double)degree;
}
// x to a word of LDS
template <bool FIXED>
__device__ __forceinline__ void pr_add(u64 *sum, float x) {
    if constexpr (FIXED) {
        const u32 bits = __float_as_uint(x), e = bits >> 23;  // x is 0, or of [2^(23 - PR_FIX), 2)
        const u64 m = ((u64)((bits & 0x7FFFFFu) | 0x800000u)) << (PR_FIX - 23);  // mantissa, of value 1 at e = 127
        atomicAdd((unsigned long long *)sum, (unsigned long long)(m >> min(127u - min(e, 127u), 63u)));
    } else {
        typedef __attribute__((address_space(3))) double lds_double;
        (void)__builtin_amdgcn_ds_atomic_fadd_f64((lds_double *)sum, (double)x);
    }
}
template <bool FIXED>
__device__ __forceinline__ double pr_sum(u64 sum) {
    return FIXED ? (double)sum * (0.5 / (double)(1ull << (PR_FIX - 1))) : __longlong_as_double((long long)sum);
}

// the host's word: (iteration, its L1 change)
__device__ __forceinline__ void pr_report(const PrSlot &s, u32 it, u64 *host) {
    __hip_atomic_store(host, ((u64)it << 32) | __float_as_uint((float)s.delta), __ATOMIC_RELEASE,
                       __HIP_MEMORY_SCOPE_SYSTEM);
}

__device__ __forceinline__ u32 wave_max(u32 v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = max(v, (u32)__shfl_xor((int)v, o, 64));
    return v;
}
static __device__ __forceinline__ double wave_sum_d(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// adds three per-thread sums of the workgroup (PRI_TPB threads at most) to a
// reduction slot; `lds` holds 3 doubles a wave
__device__ __forceinline__ void pr_reduce(double dang, double sum, double delta, PrSlot *to, double *lds) {
    dang = wave_sum_d(dang); sum = wave_sum_d(sum); delta = wave_sum_d(delta);
    const u32 wv = threadIdx.x >> 6, nw = blockDim.x >> 6;
    if (lane_id() == 0) { lds[3 * wv] = dang; lds[3 * wv + 1] = sum; lds[3 * wv + 2] = delta; }
    __syncthreads();
    if (threadIdx.x < 3) {
        double t = 0.0;
        for (u32 w = 0; w < nw; ++w) t += lds[3 * w + threadIdx.x];
        double *at = threadIdx.x == 0 ? &to->dang : (threadIdx.x == 1 ? &to->sum : &to->delta);
        if (t != 0.0) unsafeAtomicAdd(at, t);  // native 64-bit float atomic on device memory
    }
}

// start vector 1/V, out-degrees (from marker ranks), contributions, dangling
// mass, and each workgroup's largest out-degree (PR_GRID words after the slots:
// an atomic maximum by every wave took 26 us)
__global__ __launch_bounds__(PR_TPB) void k_pr_start(DevState d, const u32 *__restrict__ gpre,
                                                     u32 *__restrict__ outdeg, float *__restrict__ pr,
                                                     float *__restrict__ c0, float *__restrict__ c1, PrSlot *slot) {
    __shared__ double lds[3 * PR_TPB / 64];
    __shared__ u32 s_most[PR_TPB / 64];
    u32 most = 0;
    const u32 V = d.V, Smask = (1u << d.log2S) - 1;
    const float p = 1.f / (float)V;
    double dang = 0.0;
    for (u64 r = (u64)blockIdx.x * blockDim.x + threadIdx.x; r < V; r += (u64)gridDim.x * blockDim.x) {
        const u64 hs = d.row_off[r + 1];
        const u64 ls = r > 0 ? d.row_off[r] : 0u;
        const u64 hi = (u64)gpre[hs >> d.log2S] + (hs & Smask);
        const u64 lo = r > 0 ? (u64)gpre[ls >> d.log2S] + (ls & Smask) + 1 : 0ull;
        const u32 od = (u32)(hi - lo);
        outdeg[r] = od;
        pr[r] = p;
        c0[r] = od ? p / (float)od : 0.f;
        if (!od) dang += p;
        most = max(most, od);
    }
    most = wave_max(most);
    if (lane_id() == 0) s_most[threadIdx.x >> 6] = most;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        c0[V] = c1[V] = 0.f;  // the padding words' source
        slot->sum = 1.0;
    }
    pr_reduce(dang, 0.0, 0.0, slot, lds);  // (a barrier inside)
    if (threadIdx.x == 0) {
        for (u32 w = 0; w < PR_TPB / 64; ++w) most = max(most, s_most[w]);
        ((u32 *)(slot + PR_SLOTS))[blockIdx.x] = most;
    }
}

// Iteration `it` (from 1) is two kernels.  It reads the masses of iteration
// it - 1 from its slot and leaves its own in slot it (the ring's next slot is
// cleared).  Once an iteration's L1 change is below tol, the ones queued
// behind it return at once, which lets the host queue an iteration ahead; the
// first kernel reports the change of the one before it to the host's word.

// a vertex's new rank pr' = alpha * sum + gamma, gamma = (alpha * dangling +
// (1 - alpha) * sum(pr)) / n, and what the next iteration needs of it
struct PrMass {
    double dang, sum, delta;
};
__device__ __forceinline__ void pr_vertex(u32 v, double acc, float alpha, double gamma, const float *pr, float *out,
                                          const u32 *outdeg, float *cnext, PrMass &m) {
    const float p = (float)((double)alpha * acc + gamma);
    const u32 od = outdeg[v];
    m.delta += (double)fabsf(p - pr[v]);
    m.sum += (double)p;
    if (!od) m.dang += (double)p;
    out[v] = p;
    cnext[v] = od ? p / (float)od : 0.f;
}
__device__ __forceinline__ double pr_gamma(const PrSlot &prev, float alpha, u32 V) {
    return ((double)alpha * prev.dang + (1.0 - (double)alpha) * prev.sum) / (double)V;
}

// Chunk k of a bin's edges (cb = chunks before each bin), in groups of G words.  A bin of one chunk
// is finished here; the chunks of a larger one leave their sums in partial,
// for k_pr_join.  (Joining them by 64-bit atomics on a vector in HBM instead
// took 850 us an iteration, against 25 us.)
// Bound: the random reads of the contributions through L2 (one per edge whose
// line no other lane asks for), then the edge stream (4.5 B an edge).  6.4e7
// edges on 2^22 vertices: 195 us an iteration and 30 us for the joins, against
// 1340 us when every iteration binned contributions and summed them by LDS
// compare-and-swap; with 8-byte edges 235 us.  The LDS adds are hidden: without
// them the kernel takes the same time.
template <u32 G, bool FIXED>
__global__ __launch_bounds__(PRI_TPB) void k_pr_iter(const u32 *__restrict__ words,
                                                     const u32 *__restrict__ rows, const u32 *__restrict__ off, u32 P,
                                                     u32 NB, const u32 *__restrict__ cb, u32 chunk,
                                                     const float *__restrict__ c, float *__restrict__ cnext,
                                                     const float *__restrict__ pr, float *__restrict__ out,
                                                     const u32 *__restrict__ outdeg, u32 V, float alpha, float tol,
                                                     u32 it, PrSlot *slots, u32 starts, double *__restrict__ partial,
                                                     u64 *__restrict__ host) {
    extern __shared__ u64 pb_acc[];  // PB_BIN sums
    __shared__ double red[3 * PRI_TPB / 64];
    const PrSlot &prev = slots[(it - 1) % PR_SLOTS];
    if (blockIdx.x == 0 && threadIdx.x == 0 && it > 1) pr_report(prev, it - 1, host);
    if (blockIdx.x == 0 && it == 1 && threadIdx.x < 64) {
        // the largest out-degree, for the host's choice of later iterations
        u32 most = 0;
        for (u32 i = threadIdx.x; i < starts; i += 64) most = max(most, ((const u32 *)(slots + PR_SLOTS))[i]);
        most = wave_max(most);
        if (threadIdx.x == 0) __hip_atomic_store(host + 1, (u64)most, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    if (it > 1 && (float)prev.delta < tol) return;
    if (blockIdx.x == 0 && threadIdx.x == 0) slots[(it + 1) % PR_SLOTS] = PrSlot{0.0, 0.0, 0.0};
    const u32 k = blockIdx.x;
    if (k >= cb[NB]) return;  // the grid is an upper bound
    u32 b = 0, z = NB;        // last b with cb[b] <= k
    while (z - b > 1) {
        const u32 m = (b + z) >> 1;
        if (cb[m] <= k) b = m; else z = m;
    }
    const u32 nch = cb[b + 1] - cb[b];
    const u64 e1 = off[(u64)(b + 1) * P];
    const u64 s0 = (u64)off[(u64)b * P] + (u64)(k - cb[b]) * chunk;
    const u64 s1 = min(e1, s0 + chunk);
    const u32 v0 = b << PB_BIN_LOG, nv = min(PB_BIN, V - v0);
    for (u32 v = threadIdx.x; v < PB_BIN; v += PRI_TPB) pb_acc[v] = 0ull;
    __syncthreads();
    for (u64 i0 = s0; i0 < s1; i0 += (u64)PRI_TPB * PRI_ITEMS) {
        u32 e[PRI_ITEMS], row0[PRI_ITEMS];
#pragma unroll
        for (u32 r = 0; r < PRI_ITEMS; ++r) {
            const u64 i = i0 + (u64)r * PRI_TPB + threadIdx.x;
            const u64 j = i < s1 ? i : s1 - 1;  // unconditional loads: all of them in flight together
            if (G == 1) {
                const uint2 w = ((const uint2 *)words)[j];
                e[r] = w.x;
                row0[r] = w.y;
            } else {
                e[r] = words[j];
                row0[r] = rows[j / G];
            }
            if (i >= s1) e[r] = PB_PAD;
        }
        float x[PRI_ITEMS];
#pragma unroll
        for (u32 r = 0; r < PRI_ITEMS; ++r) x[r] = c[e[r] == PB_PAD ? V : row0[r] + (e[r] >> PB_BIN_LOG)];
#pragma unroll
        for (u32 r = 0; r < PRI_ITEMS; ++r) pr_add<FIXED>(&pb_acc[e[r] & (PB_BIN - 1)], x[r]);
    }
    __syncthreads();
    if (nch > 1) {
        double *to = partial + (u64)(cb[NB + 1 + b] + (k - cb[b])) * PB_BIN;
        for (u32 v = threadIdx.x; v < nv; v += PRI_TPB) to[v] = pr_sum<FIXED>(pb_acc[v]);
        return;
    }
    const double gamma = pr_gamma(prev, alpha, V);
    PrMass m{0.0, 0.0, 0.0};
    for (u32 v = threadIdx.x; v < nv; v += PRI_TPB)
        pr_vertex(v0 + v, pr_sum<FIXED>(pb_acc[v]), alpha, gamma, pr, out, outdeg, cnext, m);
    pr_reduce(m.dang, m.sum, m.delta, &slots[it % PR_SLOTS], red);
}

// the bins of several chunks: PB_BIN / PRI_TPB workgroups a bin, a thread a
// vertex, the chunks' sums read PRI_ITEMS at a time
__global__ __launch_bounds__(PRI_TPB) void k_pr_join(u32 NB, const u32 *__restrict__ cb, const double *__restrict__ partial,
                                                     float *__restrict__ cnext, const float *__restrict__ pr,
                                                     float *__restrict__ out, const u32 *__restrict__ outdeg, u32 V,
                                                     float alpha, float tol, u32 it, PrSlot *slots) {
    __shared__ double red[3 * PRI_TPB / 64];
    constexpr u32 WPB = PB_BIN / PRI_TPB;
    const PrSlot &prev = slots[(it - 1) % PR_SLOTS];
    if (it > 1 && (float)prev.delta < tol) return;
    const u32 b = blockIdx.x / WPB;
    const u32 k0 = cb[NB + 1 + b], k1 = k0 + (cb[b + 1] - cb[b]);
    if (k1 - k0 == 1) return;
    const u32 w = (blockIdx.x % WPB) * PRI_TPB + threadIdx.x;  // vertex within the bin
    const u32 v = (b << PB_BIN_LOG) + w;
    PrMass m{0.0, 0.0, 0.0};
    if (v < V) {
        double acc = 0.0;
        u32 k = k0;
        for (; k + PRI_ITEMS <= k1; k += PRI_ITEMS) {
            double t[PRI_ITEMS];
#pragma unroll
            for (u32 r = 0; r < PRI_ITEMS; ++r) t[r] = partial[(u64)(k + r) * PB_BIN + w];
#pragma unroll
            for (u32 r = 0; r < PRI_ITEMS; ++r) acc += t[r];
        }
        for (; k < k1; ++k) acc += partial[(u64)k * PB_BIN + w];
        pr_vertex(v, acc, alpha, pr_gamma(prev, alpha, V), pr, out, outdeg, cnext, m);
    }
    pr_reduce(m.dang, m.sum, m.delta, &slots[it % PR_SLOTS], red);
}

// rank = p / sum(p) of iteration `it`, and its report to the host
__global__ void k_pr_norm(const float *pr, float *rank, u32 V, const PrSlot *slot, u32 it, u64 *host) {
    if (blockIdx.x == 0 && threadIdx.x == 0) pr_report(*slot, it, host);
    const double inv = 1.0 / slot->sum;
    for (u64 v = (u64)blockIdx.x * blockDim.x + threadIdx.x; v < V; v += (u64)gridDim.x * blockDim.x)
        rank[v] = (float)((double)pr[v] * inv);
}

bool pr_bins_fit(u32 V) { return ((u64)V + PB_BIN - 1) / PB_BIN <= PB_MAX_BINS; }

// the groups' rows follow the words (groups of one word: stand beside them)
static u64 pr_bins_rows_at(const PrBins &b) { return (b.words + b.group - 1) / b.group * b.group; }
u64 pr_bins_edge_words(const PrBins &b) { return pr_bins_rows_at(b) / b.group * (b.group + 1) + b.group; }

PrBins pr_bins_plan(const DevState &d, u64 edges) {
    PrBins b{};
    const u64 W = nseg_of(d) << d.log2S;
    u32 lw = 0;
    while ((1ull << lw) < W) ++lw;
    // about 1024 parts, of at least one step of the bin pass
    b.part_log = std::max<u32>(std::max<u32>(d.log2S, 12), lw > 10 ? lw - 10 : 0);
    b.part_log = std::min(b.part_log, PB_MAX_PART_LOG);
    b.parts = (u32)((W + (1ull << b.part_log) - 1) >> b.part_log);
    b.bins = (u32)(((u64)d.V + PB_BIN - 1) / PB_BIN);
    // Every run that holds an edge is padded to whole groups, and the offsets
    // of the words are 32-bit sums: runs whose padding could pass them, or could
    // take more memory than a row beside every word (8 B an edge), go unpadded.
    // First iteration and each further one, unpadded against padded: 1.8*10^7
    // edges on 2^24 vertices 1044 + 377 us (988 + 372), 4*10^6 562 + 195 (626 +
    // 199), 4*10^6 on 2^22 214 + 72 (273 + 118).
    b.group = PB_CHUNK;
    b.words = std::min<u64>(edges * PB_CHUNK, edges + (u64)(PB_CHUNK - 1) * b.bins * b.parts);
    if (b.words >= 1ull << 32 || pr_bins_edge_words(b) > 2 * edges) {
        b.group = 1;
        b.words = edges;  // with a marker a row in 2^32 slots at most
    }
    b.staged = b.group == PB_CHUNK && b.bins <= PB_STAGE_MAX_BINS;
    // about two rounds of chunks over the workgroups the device holds (two a
    // CU): more chunks have more sums to join, fewer leave a tail
    b.chunk = (u32)((std::max<u64>(8192, edges / 1024) + 1023) / 1024 * 1024);
    b.max_multi = (u32)(2 * (b.words / b.chunk));  // chunks of bins of several
    b.max_chunks = (u32)(b.words / b.chunk) + b.bins;
    return b;
}

u64 pr_bins_count_words(const PrBins &b) { return (u64)b.bins * b.parts + 1; }

hipError_t pr_bins_edges(const DevState &d, const PrBins &b, u32 *off, u32 *cb, u32 *words, u32 *scan_scratch,
                         PrSlot *slots, hipStream_t st) {
    if (b.parts > PB_MAX_PARTS || b.bins > PB_MAX_BINS || b.bins == 0) return hipErrorInvalidValue;
    k_pb_count<<<b.parts, PB_TPB, b.bins * sizeof(u32), st>>>(d, b.part_log, b.parts, b.bins, b.group, off, slots);
    hipError_t e = device_excl_scan(off, (u64)b.bins * b.parts, off, scan_scratch, st);
    if (e != hipSuccess) return e;
    k_pb_chunks<<<1, 1024, 0, st>>>(off, b.parts, b.bins, b.chunk, cb);
    u32 *rows = words + pr_bins_rows_at(b);
    if (b.staged)
        k_pb_bin_staged<<<b.parts, PBS_TPB, b.bins * (PB_CHUNK + 2) * sizeof(u32), st>>>(d, b.part_log, b.parts, b.bins,
                                                                                        off, words, rows, b.words);
    else if (b.group == PB_CHUNK)
        k_pb_bin<PB_CHUNK><<<b.parts, PB_TPB, b.bins * sizeof(u32), st>>>(d, b.part_log, b.parts, b.bins, off, words,
                                                                         rows, b.words);
    else
        k_pb_bin<1><<<b.parts, PB_TPB, b.bins * sizeof(u32), st>>>(d, b.part_log, b.parts, b.bins, off, words, rows,
                                                                  b.words);
    return hipGetLastError();
}

hipError_t pr_bins_start(const DevState &d, u32 *gpre, u32 *scan_scratch, u32 *outdeg, float *pr, float *c0, float *c1,
                         PrSlot *slots, hipStream_t st) {
    hipError_t e = device_excl_scan(d.cnt, nseg_of(d), gpre, scan_scratch, st);
    if (e != hipSuccess) return e;
    k_pr_start<<<grid_for(d.V, PR_TPB, PR_GRID), PR_TPB, 0, st>>>(d, gpre, outdeg, pr, c0, c1, slots);
    return hipGetLastError();
}

u64 pr_bins_partial_words(const PrBins &b) { return std::max<u64>(1, (u64)b.max_multi * PB_BIN); }

hipError_t pr_bins_iterate(const DevState &d, const PrBins &b, const u32 *words, const u32 *off, const u32 *cb,
                           const float *c, float *cnext, const float *pr, float *out, const u32 *outdeg, float alpha,
                           float tol, u32 it, bool fixed, PrSlot *slots, double *partial, u64 *host, hipStream_t st) {
    const auto iter = b.group == PB_CHUNK ? (fixed ? k_pr_iter<PB_CHUNK, true> : k_pr_iter<PB_CHUNK, false>)
                                          : (fixed ? k_pr_iter<1, true> : k_pr_iter<1, false>);
    iter<<<b.max_chunks, PRI_TPB, PB_BIN * sizeof(u64), st>>>(
        words, words + pr_bins_rows_at(b), off, b.parts, b.bins, cb, b.chunk, c, cnext, pr, out, outdeg, d.V, alpha, tol, it,
        slots, grid_for(d.V, PR_TPB, PR_GRID), partial, host);
    if (b.max_multi)
        k_pr_join<<<b.bins * (PB_BIN / PRI_TPB), PRI_TPB, 0, st>>>(b.bins, cb, partial, cnext, pr, out, outdeg, d.V,
                                                                   alpha, tol, it, slots);
    return hipGetLastError();
}

hipError_t pr_bins_norm(const float *pr, float *rank, u32 V, u32 it, const PrSlot *slots, u64 *host, hipStream_t st) {
    k_pr_norm<<<grid_for(V, 256, 16384), 256, 0, st>>>(pr, rank, V, &slots[it % PR_SLOTS], it, host);
    return hipGetLastError();
}

}  // namespace pma
