// sort.hip -- batch packing and sorting on gfx950, and the device-wide u32
// exclusive scan used across the library.
//
// Replaces thrust::sort_by_key over the batch (rpma.cuh:1557,
// gpma.cuh:751).  The batch key src<<32|dst and its operation are packed
// into ((src << vbits | dst) << 1 | op), vbits = ceil(log2 V), with the PMA id
// above it for a group and the request order between key and operation for a
// merged sequence, so equal keys end up ordered delete before insert, earlier
// request before later; the dedup that follows keeps the last of each run.
// Two paths by batch size:
//   <= 2^19 keys   sample-split sort: two kernels, buckets chosen from a
//                  sample, each sorted by a bitonic network;
//   larger         LSD radix, one kernel per 7/8-bit digit (decoupled
//                  look-back), the digit counts of every pass taken at pack;
//                  also smaller batches found too skewed for the buckets.
#include <atomic>

#include "common.hpp"
#include "kernels.hpp"
#include "begin.hpp"

namespace pma {

// ------------------------------------------------- one kernel per pass
//
// Batches of more than 512K keys sort by LSD radix with digits of DB = 7 or 8 bits
// (six passes for the 41 bits of a lone PMA with 2^20 vertices), one kernel
// each, over tiles of OS_TPB * ITEMS keys: the pack kernel counts the digits of
// every pass at once (global digit totals); a pass kernel ranks its tile in
// LDS, publishes the tile's digit counts, reads the counts of the tiles before
// it (decoupled look-back, Merrill & Garland, "Single-pass Parallel Prefix Scan
// with Decoupled Look-back", NVR-2016-002), brings the tile into digit order in
// LDS and writes it out, a digit's keys side by side.  A published word with
// OS_PRE set carries the count of this tile and every tile before it in bits
// 0..30 (a batch has fewer than 2^31 keys); without it, this tile's count plus
// one; 0 means not yet published.
//
// Bound: HBM and the look-back's latency.  Small digits make a tile's keys of
// one digit a run of 32 to 64 keys (256 to 512 B).  2*10^6 keys of 41 bits:
// six passes of 17.6 us; four passes over 11-bit digits, written from registers
// with two keys a digit and tile, took 43 us each.  8.4*10^6 keys of 41 bits:
// 38 us to pack and six passes of 55 us (2.4 TB/s); 8-bit passes of a
// histogram, a scan and a scatter kernel took 550 us in all.
//
// Tile t waits only on tiles < t.  Workgroups are dispatched in index order,
// so every tile it waits on is running or done, unless something else holds the
// compute units that the next one in order would get; the wait is bounded
// (OS_SPIN_LIMIT rounds), after which the batch is flagged FLAG_SORT_STALL and
// changes nothing.  The host then runs it again with tiles numbered as their
// workgroups start (ORDERED: a counter a pass), where every tile that is waited
// on has its workgroup, whatever else runs.  That makes a pass of 2*10^6 keys 19.8
// us instead of 17.6 and one of 8.4*10^6 57.9 instead of 55.2, so not at first.

static constexpr int OS_TPB = 1024;  // large tiles: few tiles, short look-back walks
static constexpr u32 OS_PRE = 1u << 31;
static constexpr u32 OS_SPIN_LIMIT = 1u << 20;
static constexpr u32 OS_MAX_R = 256;
// copies of the digit totals: their atomics meet on few lines otherwise
static constexpr u32 OS_COPIES = 8;
static constexpr u32 OS_GH_WORDS = SORT_MAX_PASSES * OS_MAX_R * OS_COPIES;
// digit totals, then the passes' tile counters, to whole lines (look-back rows
// that straddle them cost 5 us of a pass of 8.4*10^6 keys)
static constexpr u32 OS_ZERO_WORDS = OS_GH_WORDS + 64;
static_assert(SORT_MAX_PASSES <= 64, "a counter a pass");
static constexpr u32 OS_PACK_GRID = 512;
static constexpr int OS_LOOK = 32;   // look-back loads in flight per thread

__device__ __forceinline__ u32 os_load(const u32 *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void os_store(u32 *p, u32 v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Pack (keys with src or dst >= V raise FLAG_INVALID_KEY) and count the digits of all npass passes:
// gh[(copy * npass + p) * R + d] += keys whose pass-p digit is d (gh zeroed by
// the caller); also clears the tiles' look-back rows for the first pass.  Few
// workgroups take several tiles each, so that their counts reach memory once.
template <int DB>
__global__ __launch_bounds__(OS_TPB) void k_pack_count(const BatchSeg *__restrict__ segs, u32 nsegs, u64 n,
                                                        const u64 *n_dev, u32 pshift, u32 sbits, u64 *__restrict__ out,
                                                        u32 *__restrict__ flags, u32 lo_bit, u32 npass, u32 items,
                                                        u32 ntiles, u32 *__restrict__ gh, u32 *__restrict__ look0) {
    constexpr u32 R = 1u << DB;
    __shared__ u32 h[SORT_MAX_PASSES * R];
    if (n_dev) n = *n_dev;
    for (u32 i = threadIdx.x; i < npass * R; i += OS_TPB) h[i] = 0;
    __syncthreads();
    bool bad = false;
    for (u32 t = blockIdx.x; t < ntiles; t += gridDim.x) {
        if (threadIdx.x < R) look0[(u64)t * R + threadIdx.x] = 0;
        const u64 base = (u64)t * items * OS_TPB + threadIdx.x;
        if (base >= n) continue;
        u32 s = source_of(segs, nsegs, base);
        BatchSeg sg = segs[s];
        for (u32 r = 0; r < items; ++r) {
            u64 i = base + (u64)r * OS_TPB;
            if (i >= n) break;
            while (i >= sg.off + sg.n) sg = segs[++s];
            const u64 p = pack_element(sg, i, pshift, sbits, bad);
            out[i] = p;
            for (u32 q = 0; q < npass; ++q) atomicAdd(&h[q * R + ((u32)(p >> (lo_bit + q * DB)) & (R - 1))], 1u);
        }
    }
    if (__any(bad) && lane_id() == 0) atomicOr(flags, FLAG_INVALID_KEY);
    __syncthreads();
    u32 *to = gh + (u64)(blockIdx.x % OS_COPIES) * npass * R;
    for (u32 i = threadIdx.x; i < npass * R; i += OS_TPB) {
        u32 v = h[i];
        if (v) atomicAdd(&to[i], v);
    }
}

// One pass over bits [shift, shift + DB).  Tile t = keys [t*T, t*T + T),
// T = OS_TPB * ITEMS; wave w holds the 64*ITEMS consecutive keys from
// t*T + w*64*ITEMS, one per lane per round, so (wave, round, lane) order is
// input order and the ranking is stable.  gh: the pass's digit totals, copies
// gstride apart.  ORDERED: tiles by next_tile, else by workgroup.
template <int DB, int ITEMS, bool ORDERED>
__global__ __launch_bounds__(OS_TPB) void k_os_pass(const u64 *__restrict__ in, u64 *__restrict__ out, u64 n,
                                                     const u64 *n_dev, u32 shift, const u32 *__restrict__ gh,
                                                     u32 gstride, u32 *__restrict__ next_tile, u32 *__restrict__ look,
                                                     u32 *__restrict__ look_next, u32 *__restrict__ flags,
                                                     u32 spin_limit) {
    constexpr u32 R = 1u << DB;
    constexpr u32 NW = OS_TPB / 64;
    constexpr u32 DW = R / 64;  // waves that hold the digits
    extern __shared__ u64 os_lds[];
    u64 *buf = os_lds;  // the tile in digit order
    // per-wave digit counts, then per-wave offsets (a tile has at most 2^13 keys)
    unsigned short(*whist)[R] = (unsigned short(*)[R])(buf + OS_TPB * ITEMS);
    __shared__ u32 lofs[R];  // the tile's keys of smaller digits
    __shared__ u32 gofs[R];  // a digit's first place in the batch, less lofs
    __shared__ u32 sums[2][DW];
    if (n_dev) n = *n_dev;
    const u32 tid = threadIdx.x;
    u32 t = blockIdx.x;
    if (ORDERED) {
        __shared__ u32 s_tile;
        if (tid == 0) s_tile = atomicAdd(next_tile, 1u);
        __syncthreads();
        t = s_tile;
    }
    if (look_next && tid < R) look_next[(u64)t * R + tid] = 0;
    const u64 tbase = (u64)t * OS_TPB * ITEMS;
    if (tbase >= n) return;  // whole workgroup: grids sized for a capacity
    const u32 lane = lane_id();
    const u32 w = tid >> 6;
    const u64 lt = (1ull << lane) - 1ull;

    u64 key[ITEMS];
    const u64 wbase = tbase + (u64)w * 64 * ITEMS + lane;
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        u64 i = wbase + (u64)r * 64;
        key[r] = i < n ? in[i] : 0ull;
    }
    u32 gv = 0;  // batch-wide total of digit tid
    if (tid < R) {
#pragma unroll
        for (u32 c = 0; c < OS_COPIES; ++c) gv += gh[(u64)c * gstride + tid];
    }
    for (u32 i = tid; i < NW * R / 2; i += OS_TPB) ((u32 *)whist)[i] = 0;
    __syncthreads();

    // rank inside the wave: lanes of equal digit found with DB ballots; the
    // wave's running count of each digit lives in whist[w] (one wave reads
    // and then updates its own row, in order)
    u32 rk[ITEMS];
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const bool valid = wbase + (u64)r * 64 < n;
        const u32 dg = (u32)(key[r] >> shift) & (R - 1);
        u64 peers = __ballot(valid);
#pragma unroll
        for (int b = 0; b < DB; ++b) {
            u64 bb = __ballot((dg >> b) & 1u);
            peers &= ((dg >> b) & 1u) ? bb : ~bb;
        }
        const u32 below = __popcll(peers & lt);
        const u32 before = whist[w][dg];
        __builtin_amdgcn_wave_barrier();
        if (valid && below == 0) whist[w][dg] = before + __popcll(peers);
        __builtin_amdgcn_wave_barrier();
        rk[r] = before + below;
    }
    __syncthreads();

    // digit tid: offsets of the waves, the tile's count, published at once,
    // and the scans of the tile's counts and of the totals
    u32 cnt = 0, li = 0, gi = 0;
    if (tid < R) {
        u32 c[NW];
#pragma unroll
        for (u32 v = 0; v < NW; ++v) c[v] = whist[v][tid];
#pragma unroll
        for (u32 v = 0; v < NW; ++v) {
            whist[v][tid] = (unsigned short)cnt;
            cnt += c[v];
        }
        os_store(&look[(u64)t * R + tid], t == 0 ? OS_PRE | cnt : cnt + 1);
        li = dpp_incl_scan32(cnt);
        gi = dpp_incl_scan32(gv);
        if (lane == 63) {
            sums[0][w] = li;
            sums[1][w] = gi;
        }
    }
    __syncthreads();
    if (tid < R) {
        for (u32 v = 0; v < w; ++v) {
            li += sums[0][v];
            gi += sums[1][v];
        }
        lofs[tid] = li - cnt;
    }
    __syncthreads();

    // the tile in digit order
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const u32 dg = (u32)(key[r] >> shift) & (R - 1);
        if (wbase + (u64)r * 64 < n) buf[lofs[dg] + whist[w][dg] + rk[r]] = key[r];
    }

    // look-back: keys of digit tid in tiles < t
    if (tid < R) {
        u32 excl = 0;
        int p = (int)t - 1;
        bool stalled = false;
        for (u32 spin = 0; p >= 0; ++spin) {
            u32 s[OS_LOOK];
            // unconditional loads (row 0 stands in past the first tile) so
            // that all of them are in flight together
#pragma unroll
            for (int k = 0; k < OS_LOOK; ++k) {
                const int q = p - k;
                s[k] = os_load(&look[(u64)(q > 0 ? q : 0) * R + tid]);
            }
            // consume predecessors in order until one is unpublished (read it
            // again next round) or carries the prefix of all before it (done);
            // branch-free so that s stays in registers
            int q = p;
            bool go = true;
            u32 acc = 0;
#pragma unroll
            for (int k = 0; k < OS_LOOK; ++k) {
                const u32 v = s[k];
                const bool pre = v >> 31;
                const bool use = go && q >= 0 && v != 0;
                acc += use ? (pre ? v & ~OS_PRE : v - 1) : 0u;
                q = use ? (pre ? -1 : q - 1) : q;
                go = use && !pre;
            }
            excl += acc;
            p = q;
            if (p >= 0 && spin >= spin_limit) {
                stalled = true;
                break;
            }
        }
        if (stalled) atomicOr(flags, FLAG_SORT_STALL);
        if (t != 0) os_store(&look[(u64)t * R + tid], OS_PRE | (excl + cnt));
        gofs[tid] = (gi - gv) + excl - (li - cnt);
    }
    __syncthreads();

    const u32 m = (u32)min((u64)(OS_TPB * ITEMS), n - tbase);
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const u32 i = tid + r * OS_TPB;
        if (i >= m) break;
        const u64 k = buf[i];
        u32 pos = gofs[(u32)(k >> shift) & (R - 1)] + i;
        if (pos >= n) pos = (u32)n - 1;  // only after a stall (flagged): stay in bounds
        out[pos] = k;
    }
}

// ------------------------------------------------------- sample-split sort
//
// Batches of up to SS_MAX_N keys sort in two kernels, whatever their key
// width.  k_ss_split: every workgroup draws the same regular sample of the
// batch (SS_OVER packed keys a bucket), sorts it (bitonic, on 32-bit
// projections), and takes its quantiles as the splitters of nb buckets
// (rounded down to a key boundary, so that equal keys of any request order and
// operation share a bucket); then it packs its tile, assigns each key to its
// bucket, and writes the tile back grouped by bucket (tile-major: no global
// offsets are needed), with its per-bucket counts and offsets.  k_ss_bucket:
// one workgroup per bucket gathers the bucket's keys from every tile into
// registers, sorts them by a bitonic network (lane swaps within a wave, LDS
// between waves), and writes them at the bucket's offset.  A sample-chosen
// split keeps buckets even under R-MAT skew, where a split on the top key bits
// puts a hub's keys in one bucket.  A bucket beyond the workgroup's SB_CAP keys
// is read for the bits on which its keys differ (AND / OR of the keys), 3 us a
// chunk of SB_CAP: if that is one key, its last element is written for all (the
// update asks only for that one); else the bucket is gathered and LSD-radix-sorted
// through global memory on those bits, chunk by chunk, with wave64 ranking (the
// k_os_pass scheme), 8 us a chunk and pass.  A splitter that is repeated (a
// projection of more than an average bucket) has a bucket of its own, so that a
// key repeated some thousand times is not mixed with others.  A batch with a
// projection of SS_SKEW_KEYS keys or more (a hub of a graph of so many vertices
// that its edges share projections), or SS_SKEW_SAME copies of one key, is not
// sorted but flagged FLAG_SORT_SKEW: the kernels after it do nothing, and the host
// runs it again with the passes above, 50 us later.  Batches over 2^20 vertices:
// 4*10^5 keys, one key half of them, 197 us (1660 by one workgroup on mixed
// buckets); 10^5 121 (473); 32 requests of 4*10^5 of one key 235 (1240), of 10^5
// 162 (350).
//
// Bound: the sample's sort in every tile (vector issue: 1024 samples 5 us, 2048
// 10 us with one tile a compute unit) and the largest bucket.  10^5 R-MAT keys:
// 13 us + 12 us with 512 buckets of 2 samples each; 256 buckets of 4: 10.6 +
// 15; of 8: 16 + 10; of 128 buckets, ranked by counting 256 samples, and 8-bit
// radix passes in LDS (an earlier form): 10.5 + 26.  3.2*10^5 keys: 22 + 26,
// against 14 + 5 * 15 in the one-kernel passes below.

static constexpr int SS_TPB = 1024;
static constexpr u32 SS_PYR = 4;          // pyramid chunks a workgroup sums side by side
static constexpr u32 SS_MAX_TILES = 256;  // a tile a compute unit: every tile sorts the sample
static constexpr u32 SS_MAX_BUCKETS = 1024;
static constexpr u32 SS_LSEGS = 128;                 // sources staged in LDS
static constexpr u32 SS_OVER = 2;                   // sample keys per bucket
static constexpr u32 SS_MAX_SAMPLE = SS_MAX_BUCKETS * SS_OVER;
static constexpr int SS_SITEMS = (int)((SS_MAX_SAMPLE + SS_TPB - 1) / SS_TPB);
static constexpr u64 SS_MAX_N = 1ull << 19;
static constexpr int SB_TPB = 1024;                 // bucket sort workgroup
static constexpr int SB_ITEMS = 4;
static constexpr u32 SB_CAP = SB_TPB * SB_ITEMS;    // keys sorted in LDS
static constexpr u32 SB_NW = SB_TPB / 64;
// a tile's count entry: offset << 16 | count, bit 31 on bucket 0's entry
// when the tile met an invalid key
static constexpr u32 SS_BAD = 1u << 31;
// and bit 30 on bucket 0's entry of tile 0 when the sample says that one
// projection holds SS_SKEW_KEYS keys or more, or as many as SS_SKEW_SAME of
// which all are one key
static constexpr u32 SS_SKEW = 1u << 30;
static constexpr u32 SS_SKEW_KEYS = 6144;
static constexpr u32 SS_SKEW_SAME = 160000;
// keys a thread: 1 up to 2^18 keys, 2 above
static int ss_items(u64 n) { return n <= (u64)SS_MAX_TILES * SS_TPB ? 1 : 2; }
static u32 ss_tiles(u64 n) { return (u32)((n + ss_items(n) * SS_TPB - 1) / (ss_items(n) * SS_TPB)); }
static_assert(SS_MAX_N <= 2ull * SS_MAX_TILES * SS_TPB && 2 * SS_TPB < (1 << 14),
              "the tiles hold a batch, and their offsets and counts stay below the marks");

// buckets of a batch of n keys, a power of two: of at most 256 keys on average
// up to 2^18 keys, so that the largest of R-MAT keys (about four times the
// average) still sorts with one key a thread
static u32 ss_buckets(u64 n) {
    u32 nb = 1;
    while (nb < SS_MAX_BUCKETS && (u64)nb * 256 < n) nb <<= 1;
    return nb;
}

// Splitters and bucket choice work on 32-bit projections of the packed
// keys, x >> psh with psh >= the bits below the key (request order,
// operation): equal keys project equally, so they share a bucket, and any
// non-decreasing splitters give a correct split.
// FIRST: a lone PMA's batch of at most FIRST sources, whose first work (status,
// update index) one more workgroup, past the tiles, does here instead of a
// kernel of its own, and the next ones the count pyramid's chunk levels the last
// batch left owing, SS_PYR chunks each (its top levels follow in the bucket
// kernel); the sources come from the kernel arguments.  (A chunk is eleven
// barriers: one by a whole workgroup, two of which fill a compute unit, took the
// kernel to 32 us over 2^23 segments; 21 with four side by side.)  A tile that
// met an invalid key marks its count of bucket 0 (bit 31): the bucket
// kernel raises the flag, after the status is cleared.
template <u32 FIRST, int ITEMS>
__global__ __launch_bounds__(SS_TPB) void k_ss_split(const BatchSeg *__restrict__ segs, u32 nsegs, u64 n,
                                                      const u64 *n_dev, u32 pshift, u32 sbits, u32 psh, u32 nb,
                                                      u64 *__restrict__ tmp, u32 *__restrict__ bc,
                                                      SegArgs<FIRST ? FIRST : 1> in, Group g, Status *status, u32 *wfirst) {
    constexpr u32 TILE = SS_TPB * ITEMS;
    __shared__ union {
        struct {
            u32 smp[2][SS_MAX_SAMPLE], spl[SS_MAX_BUCKETS], cnt[SS_MAX_BUCKETS], base[SS_MAX_BUCKETS];
        };
        u32 pyr[FIRST ? SS_PYR : 1][PYR_CH + PYR_CH / 2];
    } L;
    u32(*const smp)[SS_MAX_SAMPLE] = L.smp, *const spl = L.spl, *const cnt = L.cnt, *const base = L.base;
    __shared__ BatchSeg lsegs[FIRST ? FIRST : SS_LSEGS];
    if (n_dev) n = *n_dev;
    const u32 t = blockIdx.x;
    const u32 ntiles = (u32)((n + TILE - 1) / TILE);
    const u32 tid = threadIdx.x;
    if (FIRST) {
        if (t >= ntiles) {
            if (t == ntiles)
                batch_first_work(g, status, 0, nullptr, 0, wfirst, nullptr);
            else {
                const u32 q = tid / (SS_TPB / SS_PYR);
                pyr_chunk(pma_of(g, 0), (u64)(t - ntiles - 1) * SS_PYR + q, L.pyr[q], L.pyr[q] + PYR_CH,
                          tid % (SS_TPB / SS_PYR), SS_TPB / SS_PYR);
            }
            return;
        }
        if (tid < in.n) lsegs[tid] = in.s[tid];
        __syncthreads();
        segs = lsegs;
    }
    if (t >= ntiles) return;  // whole workgroup: grids sized for a capacity
    if (!FIRST && nsegs <= SS_LSEGS) {
        // the sources in LDS: a key's is found by a search over them
        constexpr u32 W = sizeof(BatchSeg) / 8;
        for (u32 i = tid; i < nsegs * W; i += SS_TPB) ((u64 *)lsegs)[i] = ((const u64 *)segs)[i];
        __syncthreads();
        segs = lsegs;
    }

    // the tile's keys and the sample key are loaded first, all in flight
    // while the sample is ranked
    bool bad = false;
    const u64 tbase = (u64)t * TILE;
    u64 key[ITEMS];
    bool valid[ITEMS];
    {
        const u64 i0 = tbase + tid;
        u32 s = source_of(segs, nsegs, i0 < n ? i0 : n - 1);
        BatchSeg sg = segs[s];
#pragma unroll
        for (int r = 0; r < ITEMS; ++r) {
            const u64 i = i0 + (u64)r * SS_TPB;
            valid[r] = i < n;
            key[r] = 0;
            if (valid[r]) {
                while (i >= sg.off + sg.n) sg = segs[++s];
                key[r] = pack_element(sg, i, pshift, sbits, bad);
            }
        }
    }
    // the sample's projections, sorted; its quantiles are the splitters
    const u32 ns = nb * SS_OVER;
    u32 sm[SS_SITEMS];
    u64 sx[SS_SITEMS];
#pragma unroll
    for (int r = 0; r < SS_SITEMS; ++r) {
        const u32 i = tid + r * SS_TPB;
        sm[r] = ~0u;
        sx[r] = 0;
        if (i < ns) {
            const u64 p = ((2ull * i + 1) * n) / (2ull * ns);
            bool ignore = false;
            sx[r] = pack_element(segs[source_of(segs, nsegs, p)], p, pshift, sbits, ignore);
            sm[r] = (u32)(sx[r] >> psh);
        }
    }
    if (tid < SS_MAX_BUCKETS) cnt[tid] = 0;
    block_bitonic<u32, SS_TPB, SS_SITEMS>(sm, ns, smp[0], smp[1]);
#pragma unroll
    for (int r = 0; r < SS_SITEMS; ++r) {
        const u32 i = tid + r * SS_TPB;
        if (i < ns && i > 0 && i % SS_OVER == 0) spl[i / SS_OVER - 1] = sm[r];
    }
    __syncthreads();

    // bucket = number of splitters <= the key's projection, or one less where
    // that is a repeated splitter
    auto bucket_of = [&](u32 x) {
        u32 lo = 0, hi = nb - 1;
        while (lo < hi) {
            const u32 mid = (lo + hi) >> 1;
            if (spl[mid] <= x) lo = mid + 1; else hi = mid;
        }
        return lo >= 2 && spl[lo - 2] == x ? lo - 1 : lo;
    };
    u32 bk[ITEMS], loc[ITEMS];
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        bk[r] = bucket_of((u32)(key[r] >> psh));
        loc[r] = valid[r] ? atomicAdd(&cnt[bk[r]], 1u) : 0u;
    }
    const bool tbad = __syncthreads_or(bad);
    bool skew = false;
    if (t == 0) {
        // splitters `far` apart are 2 * far samples apart
        static_assert(SS_OVER == 2, "sample keys a splitter");
        auto holds = [&](u32 keys) {
            const u32 far = (u32)(((u64)keys * nb + n - 1) / n);
            return tid + far < nb - 1 && spl[tid] == spl[tid + far];
        };
        const bool many = holds(SS_SKEW_KEYS);
        if (__syncthreads_or(many)) {
            // the lowest and the highest of the samples' key bits below the projection
            u32 *least = smp[0], *most = smp[1];
            if (tid < nb) {
                least[tid] = ~0u;
                most[tid] = 0;
            }
            __syncthreads();
#pragma unroll
            for (int r = 0; r < SS_SITEMS; ++r)
                if (tid + r * SS_TPB < ns) {
                    const u32 b = bucket_of((u32)(sx[r] >> psh));
                    const u32 low = (u32)((sx[r] & ((1ull << psh) - 1)) >> (1 + sbits));
                    atomicMin(&least[b], low);
                    atomicMax(&most[b], low);
                }
            __syncthreads();
            const u32 b = many ? bucket_of(spl[tid]) : 0u;
            skew = __syncthreads_or(many && (least[b] != most[b] || holds(SS_SKEW_SAME)));
        }
    }
    if (tid < 64) {
        // exclusive scan of the bucket counts, four a lane
        constexpr u32 PER = SS_MAX_BUCKETS / 64;
        u32 c[PER], sum = 0;
#pragma unroll
        for (u32 k = 0; k < PER; ++k) {
            c[k] = PER * tid + k < nb ? cnt[PER * tid + k] : 0u;
            sum += c[k];
        }
        u32 ex = wave_incl_scan(sum) - sum;
#pragma unroll
        for (u32 k = 0; k < PER; ++k) {
            if (PER * tid + k < nb) base[PER * tid + k] = ex;
            ex += c[k];
        }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < ITEMS; ++r)
        if (valid[r]) tmp[tbase + base[bk[r]] + loc[r]] = key[r];
    static_assert(SS_MAX_BUCKETS <= (u32)SS_TPB, "one bucket a thread");
    if (tid < nb)
        bc[(u64)tid * ntiles + t] =
            (base[tid] << 16) | cnt[tid] | (tid == 0 && tbad ? SS_BAD : 0u) | (tid == 0 && skew ? SS_SKEW : 0u);
}

// Keys of a workgroup are spread over every wave: with R = ceil(m / SB_TPB)
// rounds, wave w holds keys w*64R + r*64 + lane (r < R), so a bucket of up
// to SB_TPB keys is ranked in one round by all waves at once.
__device__ __forceinline__ u32 sb_rounds(u32 m) { return (m + SB_TPB - 1) / SB_TPB; }
__device__ __forceinline__ u32 sb_index(u32 w, u32 r, u32 lane, u32 R) { return w * (64 * R) + r * 64 + lane; }

// One LSD pass over the (up to SB_CAP) keys x[] of the workgroup, digit
// (x >> shift) & 255: returns each key's rank inside the chunk (stable, in
// the order of sb_index) in rk[] and leaves in dofs[d] the chunk's exclusive
// count of smaller digits, in whist[w][d] the keys of digit d in waves
// before w.  Every thread of the workgroup calls it.
__device__ __forceinline__ void sb_rank(const u64 (&x)[SB_ITEMS], u32 m, u32 R, u32 shift, u32 (*whist)[256],
                                        u32 *dofs, u32 *stmp, u32 (&rk)[SB_ITEMS]) {
    const u32 lane = lane_id();
    const u32 w = threadIdx.x >> 6;
    const u64 lt = (1ull << lane) - 1ull;
    for (u32 i = threadIdx.x; i < SB_NW * 256; i += SB_TPB) (&whist[0][0])[i] = 0;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < SB_ITEMS; ++r) {
        if (r >= (int)R || sb_index(w, r, 0, R) >= m) break;  // the rest of this wave's rounds are empty
        const u32 j = sb_index(w, r, lane, R);
        const bool valid = j < m;
        const u32 dg = (u32)(x[r] >> shift) & 255u;
        u64 peers = __ballot(valid);
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            const u64 bb = __ballot((dg >> b) & 1u);
            peers &= ((dg >> b) & 1u) ? bb : ~bb;
        }
        const u32 below = __popcll(peers & lt);
        const u32 before = whist[w][dg];
        __builtin_amdgcn_wave_barrier();
        if (valid && below == 0) whist[w][dg] = before + __popcll(peers);
        __builtin_amdgcn_wave_barrier();
        rk[r] = before + below;
    }
    __syncthreads();
    // the first four waves: digit d = thread; its count per wave turns into
    // the prefix of the waves before, its total into a wave-wide DPP scan
    u32 total = 0, inc = 0;
    if (threadIdx.x < 256) {
        const u32 d = threadIdx.x;
        u32 c[SB_NW];
#pragma unroll
        for (u32 v = 0; v < SB_NW; ++v) c[v] = whist[v][d];
#pragma unroll
        for (u32 v = 0; v < SB_NW; ++v) {
            whist[v][d] = total;
            total += c[v];
        }
        inc = dpp_incl_scan32(total);
        if (lane == 63) stmp[w] = inc;
    }
    __syncthreads();
    if (threadIdx.x < 256) {
        u32 pre = 0;
        for (u32 v = 0; v < w; ++v) pre += stmp[v];
        dofs[threadIdx.x] = pre + inc - total;
    }
    __syncthreads();
}

// ks: bits below the key (request order, operation).
// top: one more workgroup, past the buckets, sums the lone PMA's pyramid
// top levels (after the split kernel's chunk levels)
__global__ __launch_bounds__(SB_TPB) void k_ss_bucket(const u64 *__restrict__ tmp, u64 *__restrict__ out,
                                                       u64 *__restrict__ aux, u64 n, const u64 *n_dev, u32 tile, u32 nb, u32 ks,
                                                       const u32 *__restrict__ bc, u32 *__restrict__ flags,
                                                       bool top, DevState topd) {
    // the bucket's sort, or an oversized bucket's radix passes, or the
    // pyramid's top levels
    __shared__ union {
        u64 kb[2][SB_CAP];
        struct {
            u32 whist[SB_NW][256], dofs[256], run[256];
        };
        u32 pyr[2 * PYR_TOP_LDS];
    } L;
    __shared__ u32 toff[SS_MAX_TILES + 1], tb[SS_MAX_TILES];
    __shared__ u32 stmp[SB_NW + 1];
    __shared__ u64 red[3][SB_NW];
    u32(*const whist)[256] = L.whist;
    u32 *const dofs = L.dofs, *const run = L.run;
    if (n_dev) n = *n_dev;
    const u32 b = blockIdx.x;
    const u32 tid = threadIdx.x;
    const u32 ntiles = (u32)((n + tile - 1) / tile);
    if (top && b == nb) {
        pyr_top_levels(topd, L.pyr);
        return;
    }
    if (b >= nb || ntiles == 0) return;
    const bool skew = bc[0] & SS_SKEW;
    // where the bucket lies in each tile and inside the bucket; its offset in
    // the batch is the sum of its offsets in the tiles (a tile's keys of the
    // buckets before it)
    constexpr u32 TW = SS_MAX_TILES / 64;  // waves that hold the tiles' entries
    static_assert(SS_MAX_TILES % 64 == 0 && SS_MAX_TILES <= SB_TPB, "one entry a thread");
    __shared__ u32 sums[2][TW];
    u32 e = 0, inc = 0;
    if (tid < SS_MAX_TILES) {
        e = tid < ntiles ? bc[(u64)b * ntiles + tid] : 0u;
        inc = dpp_incl_scan32(e & 0xFFFFu);
        const u32 off = wave_sum((e & ~(SS_BAD | SS_SKEW)) >> 16);
        if (lane_id() == 63) {
            sums[0][tid >> 6] = inc;
            sums[1][tid >> 6] = off;
        }
    }
    __syncthreads();
    if (b == 0 && (e & SS_BAD)) atomicOr(flags, FLAG_INVALID_KEY);
    if (skew) {
        if (b == 0 && tid == 0) atomicOr(flags, FLAG_SORT_SKEW);
        return;
    }
    u32 m = 0, pre = 0;
    u64 obase = 0;
#pragma unroll
    for (u32 w = 0; w < TW; ++w) {
        if (w < tid >> 6) pre += sums[0][w];
        m += sums[0][w];
        obase += sums[1][w];
    }
    if (tid < ntiles) {
        toff[tid] = inc - (e & 0xFFFFu) + pre;
        tb[tid] = (e & ~(SS_BAD | SS_SKEW)) >> 16;
    }
    if (tid == 0) toff[ntiles] = m;
    if (m == 0) return;
    __syncthreads();
    const u32 lane = lane_id();
    const u32 w = tid >> 6;
    auto addr_of = [&](u32 j) -> u64 {
        u32 lo = 0, hi = ntiles;  // last tile with toff <= j
        while (hi - lo > 1) {
            const u32 mid = (lo + hi) >> 1;
            if (toff[mid] <= j) lo = mid; else hi = mid;
        }
        return (u64)lo * tile + tb[lo] + (j - toff[lo]);
    };

    if (m <= SB_CAP) {
        // gather (addresses first, then the loads), and a bitonic sort
        u64 x[SB_ITEMS];
        {
            u64 ad[SB_ITEMS];
#pragma unroll
            for (int r = 0; r < SB_ITEMS; ++r) {
                const u32 j = r * SB_TPB + tid;
                ad[r] = j < m ? addr_of(j) : ~0ull;
            }
#pragma unroll
            for (int r = 0; r < SB_ITEMS; ++r) x[r] = ad[r] != ~0ull ? tmp[ad[r]] : ~0ull;
        }
        block_bitonic<u64, SB_TPB, SB_ITEMS>(x, m, L.kb[0], L.kb[1]);
#pragma unroll
        for (int r = 0; r < SB_ITEMS; ++r) {
            const u32 j = r * SB_TPB + tid;
            if (j < m) out[obase + j] = x[r];
        }
        return;
    }

    // beyond the LDS: the bits that vary, and the last key in order
    u64 andv = ~0ull, orv = 0, last = 0;
    constexpr u32 FLY = 16;  // loads of a thread in flight
    for (u32 j0 = tid; j0 < m; j0 += SB_TPB * FLY) {
        u64 x[FLY];
#pragma unroll
        for (u32 r = 0; r < FLY; ++r) x[r] = tmp[addr_of(min(j0 + r * SB_TPB, m - 1))];
#pragma unroll
        for (u32 r = 0; r < FLY; ++r) {
            andv &= x[r];
            orv |= x[r];
            last = max(last, x[r]);
        }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        andv &= __shfl_xor(andv, o, 64);
        orv |= __shfl_xor(orv, o, 64);
        last = max(last, (u64)__shfl_xor(last, o, 64));
    }
    if (lane == 0) { red[0][w] = andv; red[1][w] = orv; red[2][w] = last; }
    __syncthreads();
    andv = ~0ull;
    orv = 0;
#pragma unroll
    for (u32 q = 0; q < SB_NW; ++q) { andv &= red[0][q]; orv |= red[1][q]; last = max(last, red[2][q]); }
    if (((andv ^ orv) >> ks) == 0) {
        // one key: its last element decides, and the ones before it only have to
        // be that key's, so it stands for all
        for (u32 j = tid; j < m; j += SB_TPB) out[obase + j] = last;
        return;
    }
    // several: gathered into the output range, then LSD passes over the bits
    // that vary, chunk by chunk through global memory (from the output range to
    // aux and back); each digit's running offset carries across the chunks, which
    // are taken in order (stable)
    for (u32 j = tid; j < m; j += SB_TPB) out[obase + j] = tmp[addr_of(j)];
    __syncthreads();  // makes the gather's stores visible to the workgroup
    const u64 diff = andv ^ orv;
    const u32 lo_bit = diff ? (u32)__builtin_ctzll(diff) : 64u;
    const u32 hi_bit = diff ? 64u - (u32)__builtin_clzll(diff) : 0u;
    u64 *src = out + obase, *dst = aux + obase;
    for (u32 shift = lo_bit; shift < hi_bit; shift += 8) {
        // digit totals of the bucket, then their exclusive scan as the start
        for (u32 i = tid; i < SB_NW * 256; i += SB_TPB) (&whist[0][0])[i] = 0;
        __syncthreads();
        for (u32 j = tid; j < m; j += SB_TPB) atomicAdd(&whist[0][(u32)(src[j] >> shift) & 255u], 1u);
        __syncthreads();
        {
            const u32 c = tid < 256 ? whist[0][tid] : 0u;
            u32 tot;
            const u32 ex = block_excl_scan<SB_TPB, u32>(c, tot, stmp);
            if (tid < 256) run[tid] = ex;
        }
        __syncthreads();
        for (u32 c0 = 0; c0 < m; c0 += SB_CAP) {
            const u32 mc = m - c0 < SB_CAP ? m - c0 : SB_CAP;
            const u32 R = sb_rounds(mc);
            u64 x[SB_ITEMS];
            u32 rk[SB_ITEMS];
#pragma unroll
            for (int r = 0; r < SB_ITEMS; ++r) {
                const u32 j = r < (int)R ? sb_index(w, r, lane, R) : mc;
                x[r] = j < mc ? src[c0 + j] : 0ull;
            }
            sb_rank(x, mc, R, shift, whist, dofs, stmp, rk);
#pragma unroll
            for (int r = 0; r < SB_ITEMS; ++r) {
                const u32 j = r < (int)R ? sb_index(w, r, lane, R) : mc;
                if (j < mc) {
                    const u32 dg = (u32)(x[r] >> shift) & 255u;
                    dst[run[dg] + whist[w][dg] + rk[r]] = x[r];
                }
            }
            __syncthreads();
            // the chunk's count of digit d: the next digit's chunk offset
            // minus this one's
            if (tid < 256) run[tid] += (tid + 1 < 256 ? dofs[tid + 1] : mc) - dofs[tid];
            __syncthreads();
        }
        u64 *t2 = src; src = dst; dst = t2;
        __syncthreads();
    }
    if (src != out + obase)
        for (u32 j = tid; j < m; j += SB_TPB) out[obase + j] = src[j];
}

// ------------------------------------------------------ device-wide scan

static constexpr int SC_TPB = 256;
static constexpr int SC_ITEMS = 8;
static constexpr int SC_TILE = SC_TPB * SC_ITEMS;

__global__ __launch_bounds__(SC_TPB) void k_scan_reduce(const u32 *__restrict__ in, u64 n, u32 *__restrict__ part) {
    u64 base = (u64)blockIdx.x * SC_TILE;
    u32 sum = 0;
#pragma unroll
    for (int r = 0; r < SC_ITEMS; ++r) {
        u64 i = base + (u64)r * SC_TPB + threadIdx.x;
        if (i < n) sum += in[i];
    }
    __shared__ u32 tmp[SC_TPB / 64 + 1];
    u32 tot;
    block_excl_scan<SC_TPB, u32>(sum, tot, tmp);
    if (threadIdx.x == 0) part[blockIdx.x] = tot;
}

// exclusive scan of part[0..np) in place by one workgroup; part[np] = total
__global__ __launch_bounds__(1024) void k_scan_partials(u32 *__restrict__ part, u32 np) {
    __shared__ u32 tmp[1024 / 64 + 1];
    u32 carry = 0;
    for (u32 b = 0; b < np; b += 1024) {
        u32 i = b + threadIdx.x;
        u32 v = i < np ? part[i] : 0;
        u32 tot;
        u32 ex = block_excl_scan<1024, u32>(v, tot, tmp);
        if (i < np) part[i] = carry + ex;
        carry += tot;
    }
    if (threadIdx.x == 0) part[np] = carry;
}

__global__ __launch_bounds__(SC_TPB) void k_scan_down(const u32 *__restrict__ in, u64 n, const u32 *__restrict__ part,
                                                      u32 *__restrict__ out) {
    __shared__ u32 tile[SC_TILE];
    __shared__ u32 tmp[SC_TPB / 64 + 1];
    u64 base = (u64)blockIdx.x * SC_TILE;
#pragma unroll
    for (int r = 0; r < SC_ITEMS; ++r) {
        u64 i = base + (u64)r * SC_TPB + threadIdx.x;
        tile[r * SC_TPB + threadIdx.x] = i < n ? in[i] : 0;
    }
    __syncthreads();
    // each thread owns SC_ITEMS consecutive entries
    u32 loc[SC_ITEMS];
    u32 sum = 0;
#pragma unroll
    for (int r = 0; r < SC_ITEMS; ++r) { loc[r] = tile[threadIdx.x * SC_ITEMS + r]; sum += loc[r]; }
    u32 tot;
    u32 ex = block_excl_scan<SC_TPB, u32>(sum, tot, tmp) + part[blockIdx.x];
#pragma unroll
    for (int r = 0; r < SC_ITEMS; ++r) { tile[threadIdx.x * SC_ITEMS + r] = ex; ex += loc[r]; }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < SC_ITEMS; ++r) {
        u64 i = base + (u64)r * SC_TPB + threadIdx.x;
        if (i < n) out[i] = tile[r * SC_TPB + threadIdx.x];
    }
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) out[n] = part[gridDim.x];
}

u64 scan_scratch_words(u64 n) { return (n + SC_TILE - 1) / SC_TILE + 2; }

// out[0..n) = exclusive prefix of in, out[n] = total.  out may alias in.
hipError_t device_excl_scan(const u32 *in, u64 n, u32 *out, u32 *scratch, hipStream_t st) {
    u32 nb = (u32)((n + SC_TILE - 1) / SC_TILE);
    if (nb == 0) nb = 1;
    k_scan_reduce<<<nb, SC_TPB, 0, st>>>(in, n, scratch);
    k_scan_partials<<<1, 1024, 0, st>>>(scratch, nb);
    k_scan_down<<<nb, SC_TPB, 0, st>>>(in, n, scratch, out);
    return hipGetLastError();
}

// ------------------------------------------------------------ radix driver

// Keys a thread in a tile of the one-kernel passes: 4 up to one tile per CU, 8
// beyond, for longer runs and fewer tiles to look back over (2*10^6 keys: 17.6
// against 19.9 us a pass; 8.4*10^6: 55 and 54).
static constexpr u64 OS_SMALL_N = 1ull << 20;
static u32 os_items(u64 n) { return n <= OS_SMALL_N ? 4 : 8; }

// Fault injection for the failure-path tests: so many radix sorts whose tiles do
// not wait for the ones before them.
static std::atomic<u64> g_stalls{0};
void inject_sort_stalls(u64 sorts) { g_stalls.store(sorts, std::memory_order_relaxed); }
static bool injected_stall() {
    u64 c = g_stalls.load(std::memory_order_relaxed);
    while (c && !g_stalls.compare_exchange_weak(c, c - 1, std::memory_order_relaxed)) {
    }
    return c != 0;
}

// digit width for a sort over `width` bits: as many passes as 8-bit digits take
static u32 os_digit_bits(u32 width) { return (width + 7) / 8 * 7 >= width ? 7 : 8; }

// of any batch of up to n keys (never less for more keys: a reserved scratch
// serves the smaller batches too, whose tiles may be smaller and more)
u64 sort_scratch_words(u64 n) {
    auto tiles = [](u64 keys, u64 tile) { return (keys + tile - 1) / tile; };
    const u64 small = std::min<u64>(n, OS_SMALL_N), ss = std::min<u64>(n, SS_MAX_N);
    const u64 look = std::max(tiles(small, 4 * OS_TPB), n > OS_SMALL_N ? tiles(n, 8 * OS_TPB) : 0);
    const u64 split = ss_buckets(ss) * std::min<u64>(SS_MAX_TILES, tiles(ss, SS_TPB));
    return OS_ZERO_WORDS + std::max<u64>(2 * OS_MAX_R * look, split);
}

u32 sort_zero_words() { return OS_ZERO_WORDS; }

template <int DB, int ITEMS>
static u64 *os_sort(const BatchSeg *segs, u32 nsegs, u64 n, const u64 *n_dev, u32 pshift, u32 sbits, u32 lo_bit,
                    u32 npass, u64 *k0, u64 *k1, u32 *scratch, u32 *flags, bool ordered, hipStream_t st) {
    const u32 spin_limit = !n_dev && injected_stall() ? 0u : OS_SPIN_LIMIT;  // (a captured graph keeps its limit)
    const auto pass = ordered ? k_os_pass<DB, ITEMS, true> : k_os_pass<DB, ITEMS, false>;
    constexpr u32 R = 1u << DB;
    constexpr u64 tile = (u64)ITEMS * OS_TPB;
    const u32 ntiles = (u32)((n + tile - 1) / tile);
    u32 *gh = scratch;
    u32 *look[2] = {scratch + OS_ZERO_WORDS, scratch + OS_ZERO_WORDS + (u64)ntiles * R};
    k_pack_count<DB><<<std::min(ntiles, OS_PACK_GRID), OS_TPB, 0, st>>>(segs, nsegs, n, n_dev, pshift, sbits, k0, flags,
                                                                       lo_bit, npass, ITEMS, ntiles, gh, look[0]);
    u64 *src = k0, *dst = k1;
    const size_t lds = tile * sizeof(u64) + (size_t)(OS_TPB / 64) * R * sizeof(unsigned short);
    for (u32 q = 0; q < npass; ++q) {
        const u32 shift = lo_bit + q * DB;
        u32 *nxt = q + 1 < npass ? look[(q + 1) & 1] : nullptr;
        pass<<<ntiles, OS_TPB, lds, st>>>(src, dst, n, n_dev, shift, gh + q * R, npass * R, scratch + OS_GH_WORDS + q,
                                          look[q & 1], nxt, flags, spin_limit);
        u64 *t = src; src = dst; dst = t;
    }
    return src;
}

// Packs a group batch (n elements from nsegs sources) and sorts the packed
// keys on bits [lo_bit, hi_bit): the first histogram is taken while packing.
// With n_dev the kernels read the element count from device memory and n
// is only a capacity that sizes the grids (graph replays).  The first
// sort_zero_words() words of `scratch` must be zero on entry (the batch's
// first kernel clears them).
u64 *pack_and_sort(const BatchSeg *segs, u32 nsegs, u64 n, const u64 *n_dev, u32 pshift, u32 sbits, u32 lo_bit,
                   u32 hi_bit, u64 *k0, u64 *k1, u64 *k2, u32 *scratch, u32 *flags, SortBy by, hipStream_t st) {
    if (n == 0) return k0;
    if (n <= SS_MAX_N && by == SortBy::SIZE) {
        // sample-split sort: k1 holds the tiles grouped by bucket, k0 the
        // result, k2 the second buffer of oversized buckets; the tiles'
        // bucket counts go to the scratch after its cleared words
        const u32 nb = ss_buckets(n);
        const u32 ntiles = ss_tiles(n);
        u32 *bc = scratch + OS_ZERO_WORDS;
        const u32 ks = 1 + sbits;
        const u32 psh = hi_bit > 32 + ks ? hi_bit - 32 : ks;
        if (ss_items(n) == 1)
            k_ss_split<0, 1><<<ntiles, SS_TPB, 0, st>>>(segs, nsegs, n, n_dev, pshift, sbits, psh, nb, k1, bc,
                                                             SegArgs<1>{}, Group{}, nullptr, nullptr);
        else
            k_ss_split<0, 2><<<ntiles, SS_TPB, 0, st>>>(segs, nsegs, n, n_dev, pshift, sbits, psh, nb, k1, bc,
                                                             SegArgs<1>{}, Group{}, nullptr, nullptr);
        k_ss_bucket<<<nb, SB_TPB, 0, st>>>(k1, k0, k2, n, n_dev, (u32)ss_items(n) * SS_TPB, nb, ks, bc, flags, false,
                                           DevState{});
        return k0;
    }
    const u32 width = hi_bit - lo_bit;
    const u32 db = os_digit_bits(width);
    const u32 npass = (width + db - 1) / db;
    const bool big = os_items(n) == 8;
    const auto sort = db == 7 ? (big ? os_sort<7, 8> : os_sort<7, 4>) : (big ? os_sort<8, 8> : os_sort<8, 4>);
    return sort(segs, nsegs, n, n_dev, pshift, sbits, lo_bit, npass, k0, k1, scratch, flags, by == SortBy::ORDERED_TILES,
                st);
}

bool sort_carries_first(u64 n, u32 nsegs) { return n > 0 && n <= SS_MAX_N && nsegs <= ARG_SEGS; }

// The sample-split sort of a lone PMA's batch of at most SS_MAX_N keys from at
// most ARG_SEGS sources, with the batch's first work (batch_begin without its
// sort-scratch clearing, which the sample-split sort does not need) in one
// more workgroup of the split kernel, pyr_chunks more for the pyramid's
// chunk levels the last batch left owing, and one more of the bucket kernel
// for the pyramid's top levels.  Sources beyond INLINE_SEGS in the arguments
// instead of a copy of them, a kernel for the first work and two for the
// pyramid: 32 requests of 5000 + 5000 keys on 2^25 edges 212 -> 194 us.
template <u32 N>
static void ss_split_first(u32 grid, const Group &g, Status *status, u32 *wfirst, const BatchSeg *segs, u32 nsegs,
                           u64 n, u32 pshift, u32 sbits, u32 psh, u32 nb, u64 *tmp, u32 *bc, hipStream_t st) {
    static_assert(sizeof(SegArgs<N>) + sizeof(Group) + 128 <= 4096, "kernel arguments");
    const SegArgs<N> in = seg_args<N>(segs, nsegs);
    if (ss_items(n) == 1)
        k_ss_split<N, 1><<<grid, SS_TPB, 0, st>>>(nullptr, nsegs, n, nullptr, pshift, sbits, psh, nb, tmp, bc, in, g,
                                                  status, wfirst);
    else
        k_ss_split<N, 2><<<grid, SS_TPB, 0, st>>>(nullptr, nsegs, n, nullptr, pshift, sbits, psh, nb, tmp, bc, in, g,
                                                  status, wfirst);
}

u64 *pack_and_sort_first(const Group &g, Status *status, u32 *wfirst, const BatchSeg *segs, u32 nsegs, u64 n,
                         u32 pshift, u32 sbits, u32 hi_bit, u64 *k0, u64 *k1, u64 *k2, u32 *scratch, u32 pyr_chunks,
                         hipStream_t st) {
    const u32 nb = ss_buckets(n);
    u32 *bc = scratch + OS_ZERO_WORDS;
    const u32 ks = 1 + sbits;
    const u32 psh = hi_bit > 32 + ks ? hi_bit - 32 : ks;
    const u32 grid = ss_tiles(n) + 1 + (pyr_chunks + SS_PYR - 1) / SS_PYR;
    if (nsegs <= INLINE_SEGS)
        ss_split_first<INLINE_SEGS>(grid, g, status, wfirst, segs, nsegs, n, pshift, sbits, psh, nb, k1, bc, st);
    else
        ss_split_first<ARG_SEGS>(grid, g, status, wfirst, segs, nsegs, n, pshift, sbits, psh, nb, k1, bc, st);
    k_ss_bucket<<<nb + 1, SB_TPB, 0, st>>>(k1, k0, k2, n, nullptr, (u32)ss_items(n) * SS_TPB, nb, ks, bc, &status->flags,
                                           true, g.one);
    return k0;
}

}  // namespace pma
