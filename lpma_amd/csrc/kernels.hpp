// kernels.hpp -- host-side launchers of the HIP kernels (one per phase).
#pragma once
#include "common.hpp"

namespace pma {

// sort.hip
u64 scan_scratch_words(u64 n);
hipError_t device_excl_scan(const u32 *in, u64 n, u32 *out, u32 *scratch, hipStream_t st);
u64 sort_scratch_words(u64 n);
u32 sort_zero_words();
// how a batch is sorted: as its size asks, by radix passes (after
// FLAG_SORT_SKEW), or by radix passes whose tiles cannot wait for one that has
// not started (after FLAG_SORT_STALL)
enum class SortBy { SIZE, RADIX, ORDERED_TILES };
// k0, k1, k2: n keys each (k2 only for batches of up to 2^19 keys, as the
// second buffer of an oversized bucket).  A batch that comes back unsorted has
// FLAG_SORT_SKEW or FLAG_SORT_STALL in flags
u64 *pack_and_sort(const BatchSeg *segs, u32 nsegs, u64 n, const u64 *n_dev, u32 pshift, u32 sbits, u32 lo_bit,
                   u32 hi_bit, u64 *k0, u64 *k1, u64 *k2, u32 *scratch, u32 *flags, SortBy by, hipStream_t st);
// the next `sorts` radix sorts give up waiting at once (tests)
void inject_sort_stalls(u64 sorts);

// update.hip
struct BatchBufs {
    u64 *ukey;     // n: decoded keys of the sorted batch
    u64 *useg;     // n: run key pid << 32 | segment (| RK_OP for inserts, RK_SKIP without effect); duplicates RK_NONE
    u64 *ckey;     // n: compacted effective updates (sorted by pid, key)
    u64 *cseg;     // n: their run keys
    i32 *pd;       // n+1: exclusive prefix of +1 (insert) / -1 (delete)
    u32 *rlevel;   // n: chosen level per run start
    uint4 *rwin;   // n: per run start, its chosen window's update range [u0, u1) and counts C, M
    u64 *part;     // LOC_GROUPS + nblocks: (count, delta) of groups of locate blocks, then of each block
    Work *work[NUM_CLASSES];  // n each
    u32 *lchunk;   // n+1: chunk prefix over large windows
    u64 *lmbase;   // n: merged-scratch base per large window
    u32 *lhdr;     // 4: large windows, chunks
    u32 *wfirst;   // WFIRST_N + 1: first compacted update per index-level window (lone PMA)
    Status *status;
};

// batch descriptors small enough to travel as kernel arguments
static constexpr u32 INLINE_SEGS = 4;
template <u32 N>
struct SegArgs {
    BatchSeg s[N];
    u32 n;
};
using InlineSegs = SegArgs<INLINE_SEGS>;
static constexpr u32 ARG_SEGS = 64;  // of the sort's and the batch's first kernel (3 KB of arguments)
template <u32 N>
inline SegArgs<N> seg_args(const BatchSeg *segs, u32 n) {
    SegArgs<N> a = {};
    for (u32 k = 0; k < n; ++k) a.s[k] = segs[k];
    a.n = n;
    return a;
}

// sort.hip: a lone PMA's batch of at most 2^19 keys from at most ARG_SEGS
// sources (segs: on the host, passed as kernel arguments) is sorted with the batch's first work (batch_begin's, without clearing the
// sort scratch) carried by the sort kernels: no batch_begin launch, and the
// pyramid's pyr_chunks chunk levels owed by the last batch summed there too
bool sort_carries_first(u64 n, u32 nsegs);
u64 *pack_and_sort_first(const Group &g, Status *status, u32 *wfirst, const BatchSeg *segs, u32 nsegs, u64 n,
                         u32 pshift, u32 sbits, u32 hi_bit, u64 *k0, u64 *k1, u64 *k2, u32 *scratch, u32 pyr_chunks,
                         hipStream_t st);

// A lone PMA's batch of at most SMALL_MAX_N keys from inline sources, from its
// keys to the elected windows in one kernel, with the pyramid's levels owed by
// the last batch (chunks: its chunk levels, 0 if none) summed beside it; the
// outcome goes to the status and to `early`.  arrive: two words, zero.
static constexpr u32 SMALL_MAX_N = 2048;
static constexpr u32 SMALL_ARRIVE_WORDS = 2;
hipError_t small_batch(const Group &g, const BatchBufs &b, const InlineSegs &in, u64 n, u32 chunks, u32 *arrive,
                       EarlyOut *early, hipStream_t st);

u32 locate_blocks(u64 n);
// most groups of locate blocks
static constexpr u32 LOC_GROUPS = 1024;
// also clears zero[0, nzero) (the sort's digit totals) and the locate groups,
// resets the update index and, given at most ARG_SEGS sources of the host's in
// `hsegs`, stores them in segs
hipError_t batch_begin(const Group &g, const BatchBufs &b, const BatchSeg *hsegs, u32 nsegs, BatchSeg *segs, u32 *zero,
                       u32 nzero, hipStream_t st);
// the batch's outcome (words of it, in b.status and after) into pinned memory,
// then *seq = epoch
hipError_t report_outcome(const BatchBufs &b, u32 words, u32 *host, u64 *seq, u32 epoch, hipStream_t st);
hipError_t locate_and_compact(const Group &g, const u64 *pk, u64 n, const BatchBufs &b, hipStream_t st);
// fixed grids for graph replays (work counts read on the device)
hipError_t rebalance_fixed(const Group &g, const BatchBufs &b, u32 runs_cap, u64 *merged, hipStream_t st);
hipError_t density_check(const Group &g, u64 n, const BatchBufs &b, hipStream_t st);
hipError_t elect_windows(const Group &g, u64 n, const BatchBufs &b, hipStream_t st);
// zeroes the work counts of the status (before a repeated election)
hipError_t reset_work_counts(Status *status, hipStream_t st);
hipError_t rebalance_lds(const Group &g, const BatchBufs &b, int cls, u32 grid, hipStream_t st, hipEvent_t e0 = nullptr,
                         hipEvent_t e1 = nullptr);
// with events (timing): the launch records its own start and end in them
hipError_t rebalance_seg(const Group &g, const BatchBufs &b, u64 windows, hipStream_t st, hipEvent_t e0 = nullptr,
                         hipEvent_t e1 = nullptr);
// single-segment and one-wave windows in one launch (a lone PMA's early
// rebalance), its grid sized for at most `bound` windows, the counts read
// from the status on the device (queued before the host knows them); first
// stores the batch's outcome in `early` when given
hipError_t rebalance_seg_wave_bound(const Group &g, const BatchBufs &b, u64 bound, EarlyOut *early, hipStream_t st,
                                    hipEvent_t e0 = nullptr, hipEvent_t e1 = nullptr);
u32 seg_lanes_log2(u32 log2S, int slots_log2);
hipError_t group_pyramid(const Group &g, u32 nblocks, hipStream_t st);
u32 pyramid_blocks(u32 H);

// global (multi-workgroup) window path, in place, and the full rebuild
hipError_t rebalance_large(const Group &g, const BatchBufs &b, u64 *merged, u32 grid, hipStream_t st);
// ubeg: nseg + 1 words of scratch
// root rebuild / resize of PMA pid: its keys after the batch (updates [u0, u1)
// of the compacted batch) from src's arrays straight into dst's, spread evenly
// (index: rebuild_index_words(src) words of scratch for the per-chunk update
// starts and ranks; merged: room for the live keys to rebuild by merging them,
// which pays where rebuild_merges(), or null)
bool rebuild_merges(u64 live, u64 updates);
hipError_t rebuild_scatter(const DevState &src, const DevState &dst, u32 pid, u32 u0, u32 u1, const BatchBufs &b,
                           u64 live, u64 m, u32 *index, u64 *merged, hipStream_t st);
u64 rebuild_index_words(const DevState &src);
hipError_t rebuild_spread(const DevState &dst, const u64 *merged, u64 m, hipStream_t st);
hipError_t window_spread(const DevState &t, u64 a, u32 L, const u64 *merged, u64 m, u64 *stats, int cls_slot,
                         hipStream_t st);
hipError_t rebuild_pyramid(const DevState &d, bool full, hipStream_t st);
hipError_t make_markers(u64 *out, u32 V, hipStream_t st);
hipError_t fill_u32(u32 *p, u64 n, u32 v, hipStream_t st);
hipError_t fill_u64(u64 *p, u64 n, u64 v, hipStream_t st);
hipError_t copy_device(void *dst, const void *src, u64 bytes, hipStream_t st);

// gen_dev.hip
hipError_t gen_rmat_device(u32 scale, u64 n, double a, double b, double c, u64 seed, u64 *out, hipStream_t st);

// views.hip
u64 export_scratch_words();
hipError_t export_compacted(const DevState &d, u32 *sums, u64 *edge_keys, u32 *row_std, u64 *all_keys, u32 *csr_row,
                            u32 *csr_col, hipStream_t st);
// the export with its scratch in a static device array (no allocation);
// setup finds the array's address on the current device
hipError_t export_scratch_setup(int device);
u64 export_static_max_segments();
hipError_t export_compacted_static(int device, const DevState &d, u64 *edge_keys, u32 *row_std, hipStream_t st);
hipError_t edge_query(const DevState &d, const u64 *q, u64 n, u32 *res, hipStream_t st);
hipError_t neighbor_count(const DevState &d, const u32 *srcs, u64 n, u32 *len, hipStream_t st);
hipError_t neighbor_offsets(const DevState &d, const u32 *srcs, u64 n, u32 *offs, u64 *word, u64 *host,
                            hipStream_t st);
bool neighbor_total(u64 word, u64 &total);  // of the word neighbor_offsets stores for the host
hipError_t neighbor_gather(const DevState &d, const u32 *srcs, u64 n, const u32 *offs, u32 *out, hipStream_t st);
hipError_t check_invariants(const DevState &d, u32 *err, hipStream_t st);

// analytics.hip
__host__ __device__ __forceinline__ u64 bfs_visited_words(u64 V) { return (V + 31) / 32; }
static constexpr u32 BFS_CTL_WORDS = 32;  // a search's sizes on the device
static constexpr u32 BFS_AHEAD = 2;       // levels queued past the last one whose frontier the host knows
hipError_t bfs_init(u32 *levels, u32 V, u32 src, u32 *queue, u32 *ctl, u32 *visited, hipStream_t st);
u64 bfs_run_words(u64 slots);
// a search's large levels through lists (list null: none)
static constexpr u32 BFS_WIN_LOG = 20;  // vertices of a window of the bitmap: 128 KB of LDS
static constexpr u32 BFS_WINDOWS = 4;   // what a wave of the expansion has LDS for; larger graphs go without lists
static constexpr u64 BFS_LIST_SLOTS = 1ull << 24;
struct BfsLists {
    u32 *list;   // destinations, in extents
    u32 *meta;   // an extent's window and length
    u32 *ne;     // extents of each wave of the expansion
    u32 *part;   // the workgroups' windows
    u32 *fresh;  // the next frontier's bits
    u32 windows;
};
u32 bfs_list_waves();  // of the default expansion
u64 bfs_list_extents(u64 slots, u32 waves);
u64 bfs_list_words(u64 extents);
u64 bfs_part_words();
// host: pinned; [0] level + 1 and the size of its frontier (low half; 1 for any
// after a level through lists), stored last; [1] live edges scanned and [2]
// levels with a frontier before it
hipError_t bfs_level(const DevState &d, const u32 *q, u32 *off, u32 *adj, u32 *runs, u32 *levels, u32 *visited,
                     u32 level, u32 *qnext, u32 *ctl, const BfsLists &ls, u64 *host, u32 expand_grid, hipStream_t st);
hipError_t pr_outdeg(const DevState &d, u32 *gpre, u32 *scan_scratch, u32 *outdeg, hipStream_t st);
hipError_t pr_init(float *pr, u32 V, float *red, hipStream_t st);
u64 pr_acc_floats(u32 V);
u32 pr_red_floats();
hipError_t pr_iterate(const DevState &d, const float *pr, const u32 *outdeg, float *c, float *acc, float *out,
                      float alpha, float *red, float *red_next, hipStream_t st);
hipError_t pr_scale(float *pr, u32 V, const float *red, hipStream_t st);
// binned edges: geometry of one PageRank call
struct PrBins {
    u32 part_log;    // slots per part (log2)
    u32 parts;       // parts of the slot array (<= 2^14)
    u32 bins;        // destination bins of 8192 vertices
    u32 chunk;       // edge words per chunk of an iteration
    u32 max_chunks;  // bound on the chunks of all bins (the iteration's grid)
    u32 max_multi;   // bound on the chunks of bins of several chunks
    u32 staged;      // bin pass stages whole 32-byte chunks in LDS
    u32 group;       // words that share a row; a run is padded to whole groups
    u64 words;       // room for the edge words, padding included
};
// masses of one iteration, in a ring of PR_SLOTS
struct PrSlot {
    double dang, sum, delta;
};
static constexpr u32 PR_SLOTS = 4;
static constexpr u32 PR_GRID = 2048;  // workgroups of vector passes: few enough for one atomic each
static constexpr u64 PR_SLOT_WORDS = PR_SLOTS * sizeof(PrSlot) / 8 + PR_GRID / 2;  // and the workgroups' largest out-degrees
bool pr_bins_fit(u32 V);
PrBins pr_bins_plan(const DevState &d, u64 edges);
u64 pr_bins_count_words(const PrBins &b);
u64 pr_bins_edge_words(const PrBins &b);
// bins the edges (off: pr_bins_count_words, cb: 2 bins + 1, words: pr_bins_edge_words)
hipError_t pr_bins_edges(const DevState &d, const PrBins &b, u32 *off, u32 *cb, u32 *words, u32 *scan_scratch,
                         PrSlot *slots, hipStream_t st);
// after pr_bins_edges: start vector and contributions (c0, c1: V + 1)
hipError_t pr_bins_start(const DevState &d, u32 *gpre, u32 *scan_scratch, u32 *outdeg, float *pr, float *c0, float *c1,
                         PrSlot *slots, hipStream_t st);
// iteration `it` = 1, 2, ...; does nothing once an earlier L1 change is below
// tol.  (it - 1) << 32 | its L1 change reaches `host`; pr_bins_norm reports the
// last one's.  The first leaves the largest out-degree in host[1].  fixed: sums in
// fixed point, where pr_fits_fixed says of a bound on the out-degrees that they
// are exact.
bool pr_fits_fixed(u32 V, u64 degree, float alpha);
u64 pr_bins_partial_words(const PrBins &b);
hipError_t pr_bins_iterate(const DevState &d, const PrBins &b, const u32 *words, const u32 *off, const u32 *cb,
                           const float *c, float *cnext, const float *pr, float *out, const u32 *outdeg, float alpha,
                           float tol, u32 it, bool fixed, PrSlot *slots, double *partial, u64 *host, hipStream_t st);
hipError_t pr_bins_norm(const float *pr, float *rank, u32 V, u32 it, const PrSlot *slots, u64 *host, hipStream_t st);

}  // namespace pma
