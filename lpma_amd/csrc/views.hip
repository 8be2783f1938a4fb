// views.hip -- read paths over the gapped layout: compacted export (the
// parity surface), the reference's CSR convention, edge-membership queries,
// neighbor-list reads, and an on-device invariant checker.
#include <mutex>

#include "common.hpp"
#include "kernels.hpp"
#include "begin.hpp"

namespace pma {

// Compacted export.  With p = rank of a live slot among live slots (from the
// segment counts):
//   all_keys[p] = key                          (get_data_rpma, rpma.cuh:1735-1761)
//   edge_keys[p - src] = key, row_std[src+1] = p - src for src's marker
//                                              (standard CSR, markers excluded)
//   csr_col[p] = dst, or src for a marker; csr_row[src+1] = p + 1
//                                              (to_csr_rpma, rpma.cuh:2192-2295)
// The segments are shared out to at most EX_TILES workgroups; a first kernel
// sums every tile's counts, and a workgroup of the second adds up the sums
// before its own and scans its counts EX_SUB segments at a time.
// Bound: HBM.  8.4*10^6 edges in 2^19 segments: 5 + 34 us (3.9 TB/s of lines
// read, 2.1 written); a three-kernel scan of the counts and a slot a thread
// took 13 + 38.
static constexpr u32 EX_TPB = 256;
static constexpr u32 EX_TILES = 1024;
static constexpr u32 EX_SUB = 512;
static constexpr u32 EX_LOADS = 8;

static u32 export_tile(u64 nseg) { return (u32)std::max<u64>(8, nseg / EX_TILES); }  // segments

__global__ __launch_bounds__(EX_TPB) void k_export_sums(const u32 *__restrict__ cnt, u64 nseg, u32 tile,
                                                         u32 *__restrict__ sums) {
    __shared__ u32 s[EX_TPB / 64];
    const u64 s0 = (u64)blockIdx.x * tile;
    u32 c = 0;
#pragma unroll 4
    for (u32 i = threadIdx.x; i < tile; i += EX_TPB) c += s0 + i < nseg ? cnt[s0 + i] : 0u;
    c = wave_sum(c);
    if (lane_id() == 0) s[threadIdx.x >> 6] = c;
    __syncthreads();
    if (threadIdx.x == 0) {
        u32 sum = 0;
        for (u32 w = 0; w < EX_TPB / 64; ++w) sum += s[w];
        sums[blockIdx.x] = sum;
    }
}

__global__ __launch_bounds__(EX_TPB) void k_export(DevState d, u32 tile, const u32 *__restrict__ sums,
                                                    u64 *__restrict__ edge_keys, u32 *__restrict__ row_std,
                                                    u64 *__restrict__ all_keys, u32 *__restrict__ csr_row,
                                                    u32 *__restrict__ csr_col) {
    __shared__ u32 pre[EX_SUB + 1];  // live slots of the sub-tile's segments before each
    __shared__ u32 tmp[EX_TPB / 64 + 1];
    const u64 nseg = nseg_of(d);
    const u32 S = 1u << d.log2S, tid = threadIdx.x;
    if (blockIdx.x == 0 && tid == 0) {
        if (row_std) row_std[0] = 0;
        if (csr_row) csr_row[0] = 0;
    }
    u32 part = 0;
#pragma unroll
    for (u32 k = 0; k < EX_TILES / EX_TPB; ++k) {
        const u32 i = k * EX_TPB + tid;
        part += i < blockIdx.x ? sums[i] : 0u;
    }
    u32 base;
    (void)block_excl_scan<EX_TPB, u32>(part, base, tmp);
    const u64 end = min((u64)(blockIdx.x + 1) * tile, nseg);
    for (u64 s0 = (u64)blockIdx.x * tile; s0 < end; s0 += EX_SUB) {
        const u32 n = (u32)min((u64)EX_SUB, end - s0);
        constexpr u32 PT = EX_SUB / EX_TPB;
        u32 c[PT], sum = 0;
#pragma unroll
        for (u32 k = 0; k < PT; ++k) {
            const u32 i = tid * PT + k;
            c[k] = i < n ? d.cnt[s0 + i] : 0u;
            sum += c[k];
        }
        u32 total;
        u32 x = base + block_excl_scan<EX_TPB, u32>(sum, total, tmp);
        base += total;
#pragma unroll
        for (u32 k = 0; k < PT; ++k) {
            pre[tid * PT + k] = x;
            x += c[k];
        }
        if (tid == EX_TPB - 1) pre[EX_SUB] = x;
        __syncthreads();
        for (u32 t0 = tid; t0 < n * S; t0 += EX_TPB * EX_LOADS) {
            u64 key[EX_LOADS];
            u32 p[EX_LOADS];
#pragma unroll
            for (u32 k = 0; k < EX_LOADS; ++k) {
                const u32 t = t0 + k * EX_TPB, seg = t >> d.log2S;
                key[k] = KEY_NONE;
                p[k] = 0;
                if (t < n * S) {
                    p[k] = pre[seg] + (t & (S - 1));
                    if (p[k] < pre[seg + 1]) key[k] = d.keys[(s0 << d.log2S) + t];
                }
            }
#pragma unroll
            for (u32 k = 0; k < EX_LOADS; ++k) {
                if (key[k] == KEY_NONE) continue;
                const u32 src = (u32)(key[k] >> 32);
                if (all_keys) all_keys[p[k]] = key[k];
                if (is_marker(key[k]) && src < d.V) {
                    if (row_std) row_std[src + 1] = p[k] - src;
                    if (csr_col) csr_col[p[k]] = src;
                    if (csr_row) csr_row[src + 1] = p[k] + 1;
                } else {
                    if (edge_keys && p[k] >= src) edge_keys[p[k] - src] = key[k];
                    if (csr_col) csr_col[p[k]] = (u32)key[k];
                }
            }
        }
        __syncthreads();
    }
}

u64 export_scratch_words() { return EX_TILES; }

hipError_t export_compacted(const DevState &d, u32 *sums, u64 *edge_keys, u32 *row_std, u64 *all_keys, u32 *csr_row,
                            u32 *csr_col, hipStream_t st) {
    const u64 nseg = nseg_of(d);
    const u32 tile = export_tile(nseg);
    const u32 tiles = (u32)((nseg + tile - 1) / tile);
    k_export_sums<<<tiles, EX_TPB, 0, st>>>(d.cnt, nseg, tile, sums);
    k_export<<<tiles, EX_TPB, 0, st>>>(d, tile, sums, edge_keys, row_std, all_keys, csr_row, csr_col);
    return hipGetLastError();
}

// ------------------------------------------- export without allocation
//
// The compacted export's scratch (the tiles' sums) in a static device array,
// for callers that may not allocate (graph capture, serving loops).  Every
// call on a device shares that device's copy: calls that overlap on one device
// race.  Nothing in it needs clearing: every word is written before it is read.

static constexpr u64 EXPORT_STATIC_MAX_SEGS = 1ull << 21;  // what callers are promised (the scratch would serve any)
static __device__ __align__(256) u32 scratch[EX_TILES];

static constexpr int EXPORT_STATIC_MAX_DEVICES = 64;
static u32 *g_scratch_ptr[EXPORT_STATIC_MAX_DEVICES];
static std::mutex g_scratch_mu;

// The device address of `scratch` on `device` (the current device), found
// once per device; the host-side name of the array is not a device address.
hipError_t export_scratch_setup(int device) {
    if (device < 0 || device >= EXPORT_STATIC_MAX_DEVICES) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> g(g_scratch_mu);
    if (g_scratch_ptr[device]) return hipSuccess;
    void *p = nullptr;
    hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    g_scratch_ptr[device] = (u32 *)p;
    return hipSuccess;
}

u64 export_static_max_segments() { return EXPORT_STATIC_MAX_SEGS; }

hipError_t export_compacted_static(int device, const DevState &d, u64 *edge_keys, u32 *row_std, hipStream_t st) {
    if (nseg_of(d) > EXPORT_STATIC_MAX_SEGS) return hipErrorInvalidValue;
    hipError_t e = export_scratch_setup(device);
    if (e != hipSuccess) return e;
    return export_compacted(d, g_scratch_ptr[device], edge_keys, row_std, nullptr, nullptr, nullptr, st);
}

// Exact edge membership (edge_query_rpma / edge_query_kernel,
// rpma.cuh:2090-2190): 1 when the key is a live edge, 0 otherwise
// (row markers and out-of-range keys are not edges).
__global__ __launch_bounds__(256) void k_edge_query(DevState d, const u64 *__restrict__ q, u64 n,
                                                     u32 *__restrict__ res) {
    for (u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (u64)gridDim.x * blockDim.x) {
        u64 key = q[i];
        u32 src = (u32)(key >> 32), dst = (u32)key;
        u32 r = 0;
        if (src < d.V && dst < d.V) {
            u32 s = locate_segment(d.sep, d.H, key);
            r = segment_holds(d, s, key) ? 1u : 0u;
        }
        res[i] = r;
    }
}

// Many queries: a workgroup stages every 2^(H - EQ_TAB_LOG)-th separator in
// LDS, so a query's first EQ_TAB_LOG levels cost no memory request.  Each lane
// then narrows its own query down to 16 separators, and later 16 slots, by a
// few probes; those 16 words, one 128-byte line, are read by the query's row
// of 16 lanes at once, query after query, one request each (a lane that went
// on alone would ask for the line again at every step: 13 requests a query
// instead of 6, and slower than the 4-ary search at 148 against 110 us).
static constexpr u32 EQ_TAB_LOG = 12;
static constexpr u32 EQ_TPB = 1024;
static constexpr u32 EQ_GRID = 512;  // two workgroups a CU

__global__ __launch_bounds__(EQ_TPB) void k_edge_query_staged(DevState d, const u64 *__restrict__ q, u64 n,
                                                               u32 *__restrict__ res) {
    __shared__ u64 tab[1u << EQ_TAB_LOG];
    const u32 tl = min(d.H, EQ_TAB_LOG), sh = d.H - tl;
    for (u32 i = threadIdx.x; i < (1u << tl); i += EQ_TPB) tab[i] = d.sep[(u64)i << sh];
    __syncthreads();
    const u32 sw = min(16u, 1u << sh), S = 1u << d.log2S, kw = min(16u, S);
    for (u64 i0 = (u64)blockIdx.x * EQ_TPB; i0 < n; i0 += (u64)gridDim.x * EQ_TPB) {
        const u64 i = i0 + threadIdx.x;
        const u64 key = i < n ? q[i] : 0ull;
        u32 at = 0;  // separator 0 is 0: never above a key
        for (u32 h = (1u << tl) >> 1; h; h >>= 1) at += tab[at + h] <= key ? h : 0u;
        at <<= sh;
        for (u32 h = (1u << sh) >> 1; h >= 16; h >>= 1) at += d.sep[at + h] <= key ? h : 0u;
        u64 v[8], w[8];
        u32 c = 0;
        row_lines<0>(d.sep, at, sw, v);
        row_lines<8>(d.sep, at, sw, w);
        row_counts<0, true>(v, key, c);
        row_counts<8, true>(w, key, c);
        // (a gap word counts for no key but KEY_NONE, which is no edge)
        at += min(c, sw) - 1;
        // the segment's keys, then gaps that hold the largest key: lines whose
        // last word is below the key are passed over
        u64 base = (u64)at << d.log2S;
        for (u32 h = S >> 1; h >= 16; h >>= 1) base += d.keys[base + h - 1] < key ? h : 0u;
        c = 0;
        row_lines<0>(d.keys, base, kw, v);
        row_lines<8>(d.keys, base, kw, w);
        row_counts<0, false>(v, key, c);
        row_counts<8, false>(w, key, c);
        if (i < n) res[i] = c && (u32)(key >> 32) < d.V && (u32)key < d.V ? 1u : 0u;
    }
}

// Staging pays once a workgroup has several hundred queries.  Over 2^19
// segments of 32 slots: 131072 queries 17.4 us staged, 16.2 us alone; 262144:
// 22.5 against 33; 10^6: 60 against 110; 4*10^6: 187 against 405.  Over 2^14:
// 10.4 against 11.4, 10.9 / 17.0, 30 / 59, 94 / 213.
static constexpr u64 EQ_STAGED_MIN = 3ull << 16;

hipError_t edge_query(const DevState &d, const u64 *q, u64 n, u32 *res, hipStream_t st) {
    if (n == 0) return hipSuccess;
    if (n >= EQ_STAGED_MIN)
        k_edge_query_staged<<<grid_for(n, EQ_TPB, EQ_GRID), EQ_TPB, 0, st>>>(d, q, n, res);
    else
        k_edge_query<<<grid_for(n, 256, 16384), 256, 0, st>>>(d, q, n, res);
    return hipGetLastError();
}

// Neighbor lists (query_rpma, rpma.cuh:1827-2036, without the time window):
// row r's edges are the live slots strictly between the markers of rows
// r-1 and r, i.e. slots (row_off[r], row_off[r+1]) (from slot 0 for r = 0).
__device__ __forceinline__ void row_range(const DevState &d, u32 r, u64 &lo, u64 &hi) {
    lo = r == 0 ? 0 : (u64)d.row_off[r] + 1;
    hi = d.row_off[r + 1];
}

// Live edges of this lane's row r (0 when !ok), from the segment counts: a
// segment's live slots are its first ones and both markers are live, so a row
// inside one segment has no gaps, and one over several has the rest of its
// first segment's live slots, every live slot of the middle ones, and the
// slots before its marker in the last.  A wave sums a long row together.  Every
// lane of the wave active.
__device__ __forceinline__ u32 row_live(const DevState &d, u32 r, bool ok) {
    const u32 Smask = (1u << d.log2S) - 1;
    u64 lo = 0, hi = 0;
    if (ok) row_range(d, r, lo, hi);
    const u32 a = (u32)(lo >> d.log2S), b = (u32)(hi >> d.log2S);
    u32 c = (u32)(hi - lo);
    if (a != b) {
        c = d.cnt[a] - ((u32)lo & Smask) + ((u32)hi & Smask);
        if (b - a <= 8)
            for (u32 k = a + 1; k < b; ++k) c += d.cnt[k];
    }
    const u32 lane = lane_id();
    for (u64 m = __ballot(b - a > 8); m; m &= m - 1) {
        const int l = __builtin_ctzll(m);
        const u32 x = (u32)__builtin_amdgcn_readlane((int)a, l), y = (u32)__builtin_amdgcn_readlane((int)b, l);
        u32 sum = 0;
#pragma unroll 4
        for (u32 k = x + 1 + lane; k < y; k += 64) sum += d.cnt[k];
        sum = wave_sum(sum);
        if (lane == (u32)l) c += sum;
    }
    return c;
}

__global__ __launch_bounds__(256) void k_nbr_count(DevState d, const u32 *__restrict__ srcs, u64 n,
                                                    u32 *__restrict__ len) {
    for (u64 i0 = (u64)blockIdx.x * 256; i0 < n; i0 += (u64)gridDim.x * 256) {
        const u64 i = i0 + threadIdx.x;
        const u32 r = i < n ? srcs[i] : 0xFFFFFFFFu;
        const u32 c = row_live(d, r, r < d.V);
        if (i < n) len[i] = c;
    }
}

// Offsets of the rows' neighbor lists: counts and their exclusive prefix, the
// total stored where the host polls for it.  A workgroup takes `per` rows; with
// several, each leaves its sum in the place of its first offset (which is 0
// within the workgroup) and adds it to `word` with its arrival (bits 48 up),
// and the last to arrive turns the sums into bases, which k_nbr_base adds to
// the offsets after them.  `word` is 0 between calls.
// Bound: latency (row offsets, then counts; 512 rows: 6 us with the launch).
static constexpr u32 NBR_TPB = 1024;  // also the most workgroups: one base a thread
static constexpr u64 NBR_DONE = 1ull << 63;

__global__ __launch_bounds__(NBR_TPB) void k_nbr_offsets(DevState d, const u32 *__restrict__ srcs, u64 n, u64 per,
                                                          u32 *__restrict__ offs, u64 *__restrict__ word,
                                                          u64 *__restrict__ host) {
    __shared__ u64 tmp[NBR_TPB / 64 + 1];
    __shared__ u64 s_total;
    __shared__ u32 s_last;
    const u32 t = threadIdx.x;
    const u64 first = blockIdx.x * per;
    u64 carry = 0;
    for (u64 k = 0; k < per && first + k < n; k += NBR_TPB) {
        const u64 i = first + k + t;
        const u32 r = i < n ? srcs[i] : 0xFFFFFFFFu;
        const u64 c = row_live(d, r, r < d.V);
        u64 total;
        const u64 x = carry + block_excl_scan<NBR_TPB, u64>(c, total, tmp);
        carry += total;
        if (i < n && (i != first || gridDim.x == 1)) offs[i] = (u32)x;
        __syncthreads();
    }
    if (gridDim.x > 1) {
        if (t == 0) {
            __hip_atomic_store(&offs[first], (u32)carry, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            const u64 old = __hip_atomic_fetch_add(word, (1ull << 48) | carry, __ATOMIC_RELAXED,
                                                   __HIP_MEMORY_SCOPE_AGENT);
            s_last = (old >> 48) == gridDim.x - 1;
            s_total = (old & ((1ull << 48) - 1)) + carry;
        }
        __syncthreads();
        if (!s_last) return;
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        carry = s_total;
        u32 sum = 0;
        if (t < gridDim.x) sum = __hip_atomic_load(&offs[t * per], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        u32 total;
        const u32 x = block_excl_scan<NBR_TPB, u32>(sum, total, (u32 *)tmp);
        if (t < gridDim.x) offs[t * per] = x;
        if (t == 0) __hip_atomic_store(word, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (t == 0) {
        offs[n] = (u32)carry;
        __hip_atomic_store(host, NBR_DONE | carry, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

__global__ __launch_bounds__(NBR_TPB) void k_nbr_base(u64 n, u64 per, u32 *__restrict__ offs) {
    const u64 i = (u64)blockIdx.x * NBR_TPB + threadIdx.x;
    const u64 first = (u64)blockIdx.x * NBR_TPB / per * per;
    if (i < n && i != first) offs[i] += offs[first];
}

// A wave per row, NBR_LOADS rounds of 64 slots in flight (one at a time left a
// row of 20000 slots 300 memory latencies).
static constexpr u32 NBR_LOADS = 4;

__global__ void k_nbr_gather(DevState d, const u32 *__restrict__ srcs, u64 n, const u32 *__restrict__ offs,
                             u32 *__restrict__ out) {
    const u64 waves = ((u64)gridDim.x * blockDim.x) >> 6;
    const u32 lane = lane_id();
    for (u64 i = ((u64)blockIdx.x * blockDim.x + threadIdx.x) >> 6; i < n; i += waves) {
        u32 r = srcs[i];
        if (r >= d.V) continue;
        u64 lo, hi;
        row_range(d, r, lo, hi);
        u64 o = offs[i];
        for (u64 t0 = lo; t0 < hi; t0 += 64 * NBR_LOADS) {
            u64 key[NBR_LOADS];
#pragma unroll
            for (u32 k = 0; k < NBR_LOADS; ++k) {
                const u64 t = t0 + k * 64 + lane;
                key[k] = t < hi ? d.keys[t] : KEY_NONE;
            }
#pragma unroll
            for (u32 k = 0; k < NBR_LOADS; ++k) {
                const bool live = key[k] != KEY_NONE;
                const u64 m = __ballot(live);
                if (live) out[o + __popcll(m & ((1ull << lane) - 1ull))] = (u32)key[k];
                o += __popcll(m);
            }
        }
    }
}

hipError_t neighbor_count(const DevState &d, const u32 *srcs, u64 n, u32 *len, hipStream_t st) {
    if (n == 0) return hipSuccess;
    k_nbr_count<<<grid_for(n, 256, 16384), 256, 0, st>>>(d, srcs, n, len);
    return hipGetLastError();
}

hipError_t neighbor_offsets(const DevState &d, const u32 *srcs, u64 n, u32 *offs, u64 *word, u64 *host,
                            hipStream_t st) {
    const u64 blocks = std::max<u64>(1, (n + NBR_TPB - 1) / NBR_TPB);
    const u64 per = (blocks + NBR_TPB - 1) / NBR_TPB * NBR_TPB;
    const u32 grid = (u32)std::max<u64>(1, (n + per - 1) / per);
    k_nbr_offsets<<<grid, NBR_TPB, 0, st>>>(d, srcs, n, per, offs, word, host);
    if (grid > 1) k_nbr_base<<<(u32)blocks, NBR_TPB, 0, st>>>(n, per, offs);
    return hipGetLastError();
}

bool neighbor_total(u64 word, u64 &total) {
    total = word & ~NBR_DONE;
    return word & NBR_DONE;
}

hipError_t neighbor_gather(const DevState &d, const u32 *srcs, u64 n, const u32 *offs, u32 *out, hipStream_t st) {
    if (n == 0) return hipSuccess;
    k_nbr_gather<<<grid_for(n * 64, 256, 16384), 256, 0, st>>>(d, srcs, n, offs, out);
    return hipGetLastError();
}

// Invariants of the layout, one thread per segment; err[0] counts
// violations: a segment's live keys are front-packed, strictly increasing,
// inside [sep[s], sep[s+1]); its count matches; a marker's slot is its row
// offset.  (The reference has no such checker; its only checks are the
// host-side comparisons in test_update_rpma.cu:131-165.)
__global__ void k_check(DevState d, u32 *err) {
    const u64 nseg = nseg_of(d);
    const u32 S = 1u << d.log2S;
    u32 bad = 0;
    for (u64 s = (u64)blockIdx.x * blockDim.x + threadIdx.x; s < nseg; s += (u64)gridDim.x * blockDim.x) {
        const u64 *seg = d.keys + (s << d.log2S);
        u32 c = d.cnt[s];
        if (c > S) { ++bad; continue; }
        u64 lo = d.sep[s];
        u64 hi = s + 1 < nseg ? d.sep[s + 1] : KEY_NONE;
        if (s == 0 && lo != 0) ++bad;
        if (hi < lo) ++bad;
        for (u32 l = 0; l < S; ++l) {
            u64 k = seg[l];
            if (l < c) {
                if (k == KEY_NONE) ++bad;
                if (k < lo || (s + 1 < nseg && k >= hi)) ++bad;
                if (l > 0 && k <= seg[l - 1]) ++bad;
                if (is_marker(k)) {
                    u32 r = (u32)(k >> 32);
                    if (r >= d.V || d.row_off[r + 1] != (u32)((s << d.log2S) + l)) ++bad;
                }
            } else if (k != KEY_NONE) {
                ++bad;
            }
        }
    }
    if (bad) atomicAdd(err, bad);
}

hipError_t check_invariants(const DevState &d, u32 *err, hipStream_t st) {
    k_check<<<grid_for(nseg_of(d), 256, 16384), 256, 0, st>>>(d, err);
    return hipGetLastError();
}

}  // namespace pma
