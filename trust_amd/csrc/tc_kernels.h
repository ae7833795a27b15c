// Device-side structures and launch wrappers of the counting kernels.
// Shared by tc_kernels.hip (device code) and the host engine.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace trust {

// Work tiers.  A vertex u is counted by exactly one tier.
//   spill: whole workgroup, hash table in HBM (table too big for any LDS)
//   big:   whole workgroup of the large-LDS launch, table in LDS
//   hub:   whole workgroup of the main launch, table in LDS
//   wave:  one wavefront, table in its LDS slice
enum Tier : int { kTierSpill = 0, kTierBig = 1, kTierHub = 2, kTierWave = 3, kTierNone = 4 };
constexpr int kNumTiers = 4;
constexpr int kWave = 64;
constexpr int kMinTableLg = 6;       // smallest table: 64 slots
constexpr int kPlanBlocks = 2048;    // planning workgroups, at most
constexpr int kMaxChunks = 256;      // 64-neighbour chunks balanced per group vertex
// Probe windows in flight per wave (the probe walk's batch): four, or six
// with kProbeDeep.  Six keep more loads in flight where the probed lists are
// long (the short-side walk: R-MAT 26 count 3% faster, R-MAT 24 2%) and
// waste more lookups on partial batches where they are short (Chung-Lu with
// the reference walk 13% slower, the 10k ER/BA batch 4%).
constexpr int kUnroll = 4;
constexpr int kUnrollDeep = 6;
// int32 offsets (and 32-bit byte offsets into adj) are used when a CSR holds
// fewer than kMaxEdges32 ids; larger ones keep int64 offsets.
constexpr long long kMaxEdges32 = 1ll << 30;

// Kernel modes: count triangles, count + per-vertex instrumentation, or
// gather only (the same loads, every hash lookup replaced by a checksum of
// the loaded ids: the load path alone, used as the roofline denominator).
constexpr int kModeCount = 0, kModeInstr = 1, kModeGather = 2;
// kModeBatch: kModeCount plus per-graph attribution (TcArgs::graph_*)
constexpr int kModeBatch = 3;
// OR-ed into kModeCount or kModeGather at enqueue/launch: the deep probe walk
constexpr int kProbeDeep = 16;

// Device control block: queue cursors, list bounds and results.  Cleared
// by a fill kernel before a run.
//
// Each work queue is split over several counters, each on its own 128-byte
// line: one address sustains only about 87 M atomics/s (11.5 ns each), and a
// line that many waves wait for also holds up the other accesses of its
// memory channel (in a count of R-MAT 16, whose 38k vertices take an atomic
// each, vertices of two neighbours took 13 us at the end of a launch).  The
// workgroup tiers hand out 8, the wave tier 32 shards.
constexpr int kXcds = 8;  // each with its own L2
constexpr int kWaveShards = 32;
constexpr int kGroupShards = 8;
constexpr int kShardStride = 32;  // unsigned ints per counter line
// The results are summed per workgroup and added to one of kSumLines lines,
// for the same reason: 8192 waves adding to one count and one probe total
// took 190 us at the end of a launch in which every wave had work.
constexpr int kSumLines = 16;
struct alignas(128) TcSum {
    unsigned long long count, probes;
};
struct alignas(128) TcCtl {
    unsigned long long count;       // triangles       (totals: host side,
    unsigned long long probes;      // hash lookups (W) fold_ctl)
    long long list_begin[8];        // tier t occupies list[list_begin[t], list_begin[t+1])
    int extra[8];                   // of them, positions beyond a vertex's first (group_parts)
    unsigned long long rebuilds;    // tables rebuilt with linear probing after a cuckoo attempt
    TcSum sums[kSumLines];          // triangles and hash lookups, by workgroup
    // queue cursors; the results stand before them (the allocation-free entry
    // copies no more than those to the host, kCtlHead bytes)
    alignas(128) unsigned int wave_next[kWaveShards * kShardStride];
    unsigned int group_next[kTierWave][kGroupShards * kShardStride];  // by tier
};
// Bytes of a control block that hold results (list bounds, sums).
constexpr size_t kCtlHead = offsetof(TcCtl, wave_next);
// Vertices of the wave tier.
inline long long wave_vertices(const TcCtl &h)
{
    return h.list_begin[kTierWave + 1] - h.list_begin[kTierWave] - h.extra[kTierWave];
}
// Vertices of the workgroup tiers with LDS tables (big and hub).
inline long long group_vertices(const TcCtl &h)
{
    return h.list_begin[kTierHub + 1] - h.list_begin[kTierBig] - h.extra[kTierBig] - h.extra[kTierHub];
}
// Totals of a control block copied back to the host.
inline void fold_ctl(TcCtl &h)
{
    for (const TcSum &x : h.sums) {
        h.count += x.count;
        h.probes += x.probes;
    }
}

// Three CSR views: the hash source (N+(u) that is tabled), the walk (the v
// in N+(u) whose lists are probed) and the probe rows (N+(v)).  For an
// unpartitioned graph all three are the same arrays; for a 2D tile job they
// are tiles (i,j), (i,k) and (k,j).
// A walk entry of an index: the start of the list it probes and that
// list's length, read together with one load and written with one store.
template <typename OffT>
struct alignas(2 * sizeof(OffT)) WalkEntry {
    OffT start;
    int32_t deg;
};

template <typename OffT>
struct TcArgs {
    const OffT *begH;
    const int32_t *adjH;
    const OffT *begW;        // row u of the walk is adjW[begW[u], endW[u])
    const OffT *endW;
    const int32_t *adjW;
    const OffT *begP;
    const int32_t *adjP;
    const int32_t *list;     // vertices grouped by tier (see TcCtl::list_begin)
    int32_t *spill_mem;      // HBM hash tables, spill_slots ints per workgroup
    long long spill_slots;
    int spill_groups;        // workgroups that own an HBM table
    int spill_tier;          // tier counted with HBM tables here, or -1
    int group_tier;          // tier counted by whole workgroups with the LDS table, or -1
    int wave_tier;           // tier counted by single waves, or -1
    int table_words;         // LDS ints for tables (group table = all of it)
    int group_lg;            // log2 of the group table capacity
    int wave_slots;          // LDS ints per wave table
    int wave_lg;
    int chunk_group;         // vertices per grab, spill/group tiers
    int chunk_wave;          // vertices per grab, wave tier (0: chosen by the kernel, -1: all alike)
    int part_entries;        // walk entries of a workgroup-tier part (0: vertices are whole)
    int wave_part;           // walk entries of a wave-tier part (0: vertices are whole)
    int pack_rows;           // rows a pack of the wave tier may hold (0, 1: no packs)
    int tag_shift;           // bits of an id (a pack's keys are id | row << tag_shift)
    int rank;
    int nranks;
    int force_linear;        // 1: linear-probing tables only (no cuckoo); 2: every cuckoo
                             // table is rebuilt with linear probing (a forced failure)
    // batch of graphs (nullable): graph g owns vertices [vbase[g], vbase[g+1])
    const long long *graph_vbase;
    // graph_page[p] = the graph holding vertex min(p << shift, V - 1)
    const int *graph_page;
    int graph_page_shift;
    int ngraphs;
    unsigned long long *graph_counts;  // per-graph triangles
    unsigned long long *graph_done;    // per-graph completion (wall-clock ticks)
    unsigned long long *graph_t0;      // earliest workgroup start (wall-clock ticks)
    TcCtl *ctl;
    unsigned long long *instr_cycles;  // per vertex (instrumented kernel only)
    unsigned long long *instr_probes;
    // Walk entries stored as the start and length of the list they probe
    // (nullable; a walk index).  Then adjW is not read.
    const WalkEntry<OffT> *entW;
};

// Planner parameters for the degree split.
template <typename OffT>
struct PlanArgs {
    const OffT *begH;
    const OffT *begW;
    const OffT *endW;
    long long V;
    int same_csr;       // H, W, P are one CSR: skip d+ < 2 as the reference does
    int hub_threshold;  // walk degree above which the workgroup tier is used
    int wave_lg;        // log2 of a wave table
    int hub_lg;         // log2 of the main launch's group table
    int big_lg;         // log2 of the large-LDS launch's table (0: no such launch)
    int force_spill;
    int wave_only;
    int part_entries;   // see group_parts (0: vertices stay whole)
    int wave_part;      // see wave_parts
    int32_t *list;      // V + list_extra(walk entries) positions
    int *block_counts;  // kPlanBlocks x 2 kNumTiers
    int per_block;      // set by launch_plan
    TcCtl *ctl;
};

constexpr size_t kPlanScratch = sizeof(int) * 2 * kNumTiers * kPlanBlocks;  // PlanArgs::block_counts

// What a stream of many counts keeps of each control block.
struct TcTotals {
    unsigned long long count, probes, rebuilds;
};

// Launch wrappers (tc_kernels.hip).  All launches go on `stream`.
// totals[i] = those of ctl[i], i < n
hipError_t launch_totals(const TcCtl *ctl, int n, TcTotals *totals, hipStream_t stream);
template <typename OffT>
hipError_t launch_plan(PlanArgs<OffT> p, hipStream_t stream);
template <typename OffT>
// big: the large-LDS launch (spill + big tiers), else the main launch.
hipError_t launch_count(const TcArgs<OffT> &a, int blocks, int threads, size_t lds_bytes,
                        int mode, bool big, hipStream_t stream);
template <typename OffT>
hipError_t count_occupancy(int threads, size_t lds_bytes, int mode, bool big, int *blocks_per_cu);
hipError_t launch_copy(const int4 *src, int4 *dst, long long n, int blocks, hipStream_t stream);
// every one of `blocks` workgroups reads src[0, n) `reps` times (sink: blocks words)
hipError_t launch_read(const int4 *src, long long n, int reps, int blocks, unsigned *sink,
                       hipStream_t stream);
hipError_t launch_offsets_to_i32(const int64_t *src, int32_t *dst, long long n,
                                 hipStream_t stream);
hipError_t launch_fill_u32(uint32_t *dst, uint32_t value, long long n, hipStream_t stream);

// Exclusive scan of a[i] (+ b[i] when b is not null), i < n, into
// out[0, n], out[n] = the total; bsum holds scan_blocks(n) + 1 long longs
// (walk_index.hip).  Launches only.
long long scan_blocks(long long n);
template <typename OutT>
hipError_t launch_scan(const int *a, const int *b, long long n, long long *bsum, OutT *out,
                       hipStream_t stream);

// Builds the walk rows of the short-side walk for an oriented CSR (the walk
// view of the three-view kernel) with one global atomic per in-entry to
// count its row and one to claim its slot: the build for graphs with too
// many target bins for the binned build (walk_index.hip).  Row x = the v in
// N+(x) with d+(v) <= d+(x), then the u with u -> x and d+(u) < d+(x), rows
// with d+ < 2 contributing nothing.  cnt: 2V ints of scratch; bsum:
// scan_blocks(V) + 1 long longs; begX: V + 1 offsets; entX: up to E (the
// start and length d+ of the entry's list in adj).  Launches only.
template <typename OffT>
hipError_t launch_side_build(const OffT *beg, const int32_t *adj, long long V, int *cnt,
                             long long *bsum, OffT *begX, WalkEntry<OffT> *entX,
                             hipStream_t stream);
// rowX[at] = the row x whose entries [begX[x], begX[x+1]) hold position at.
template <typename OffT>
hipError_t launch_side_rows(const OffT *begX, long long V, int32_t *rowX, hipStream_t stream);
// Start index of the reference walk: for e < E, entR[e] = {begP[adj[e]],
// its list length}.  Launches only.
template <typename OffT>
hipError_t launch_start_index(const OffT *begP, const int32_t *adj, long long E,
                              WalkEntry<OffT> *entR, hipStream_t stream);
// stats[0] = probes of the reference walk, stats[1] = of the short-side walk
// (stats: 2 unsigned long longs, cleared here).
template <typename OffT>
hipError_t launch_side_stats(const OffT *beg, const int32_t *adj, long long V,
                             unsigned long long *stats, hipStream_t stream);
// The short-side walk is chosen by default when it makes at most this share
// of the reference walk's probes (its lists are shorter, so a probe costs
// more; measured break-even near 0.45-0.5 on R-MAT).  Probes that the dense
// core takes over cost next to nothing and are left out of the share: on
// R-MAT graphs of 20 to 80 pairs per vertex they are two thirds of the walk.
// Index and count by the reference walk, by the short one with its core:
// scale 19, 32 pairs per vertex 3.25, 1.81 ms; scale 20, 22 pairs 4.56, 2.37
// ms; 80 pairs 38.5, 11.1 ms; scale 18, 48 pairs 2.47, 1.58 ms.
constexpr double kShortWalkShare = 0.45;

// Parts of the workgroup tiers.  One vertex's walk can hold a good share of a
// graph's probes, and the workgroup that takes it counts on when all others
// are done (R-MAT 20, 2 G probes by the short-side walk: 3.45 ms with whole
// vertices, 2.5 ms in parts; R-MAT 24 the same either way).  A vertex of
// more than part_entries walk entries (four times as many in the large-LDS
// launch, whose workgroups are four times as large) fills one list position
// per part, and each part builds the vertex's table for itself.
// part_entries is 1/16384 of the walk, so that no part outlasts the count's
// average workgroup and the list holds at most kGroupExtra more positions; at
// least 128, below which building the table costs more than the part's walk.
// Parts cut a row by position, so a rank's share of a count has none where its
// walk is a built index (each build leaves a row's entries in another order).
constexpr int kBigPartLg = 2;
constexpr long long kGroupExtra = 16384;
inline int walk_part_entries(long long walk_entries)
{
    if (walk_entries <= 0)
        return 0;
    int lg = 7;
    while (lg < 28 && (kGroupExtra << lg) < walk_entries)
        lg++;
    return 1 << lg;
}
__host__ __device__ inline int group_parts(int dW, int part_entries, int tier)
{
    if (part_entries <= 0)
        return 1;
    const int e = part_entries << (tier == kTierBig ? kBigPartLg : 0);
    return dW > e ? (dW + e - 1) / e : 1;
}

// Parts of the wave tier.  In a graph of up to some ten million walk entries
// the waves that take a vertex of 30 to 100 neighbours are the last to end
// (R-MAT 16: by 150 us of 240).  There a vertex fills a list position per
// `each` walk entries, a 131072nd of the walk (16 parts per wave) and 16 at
// least; the parts beyond the first stand before the tier's vertices and are
// chunks of their own, but in a batch, whose chunks are alike (there parts cost
// and give: counts of 9 batches of 5 to 400 graphs took 0.92 to 1.15 times as
// long as with whole vertices).  From 13 M entries on `each` passes the degree that
// sends a vertex to a workgroup.  Counts with whole vertices, with parts:
// R-MAT 16 241, 155 us; R-MAT 18 775, 570 us; R-MAT 19 1650, 1080 us.
// The position holds the part's number above kPartShift bits of the vertex,
// so a vertex has at most kMaxWaveParts.
constexpr int kPartShift = 26;
constexpr int kMaxWaveParts = 32;
constexpr long long kWaveExtra = 131072;
inline int walk_wave_part(long long walk_entries, long long V)
{
    if (walk_entries <= 0 || walk_entries >= (8 << 20) || V > (1 << kPartShift))
        return 0;
    const long long e = (walk_entries + kWaveExtra - 1) / kWaveExtra;
    return e < 16 ? 16 : (int)e;
}
__host__ __device__ inline int wave_parts(int dW, int each)
{
    if (each <= 0 || dW <= each)
        return 1;
    const int n = (dW + each - 1) / each;
    return n < kMaxWaveParts ? n : kMaxWaveParts;
}
// List positions beyond one per vertex, for walks of up to `entries` entries:
// a vertex fills fewer than one per part's entries.
constexpr long long kMaxExtra = kGroupExtra + kWaveExtra;
inline long long list_extra(long long entries)
{
    const long long g = entries >> 7, w = entries >> 4;
    return (g < kGroupExtra ? g : kGroupExtra) + (w < kWaveExtra ? w : kWaveExtra);
}

// Packs of the wave tier (tc_kernels.hip): ids below `ids` leave the upper
// bits of a 32-bit key for the row's number; the largest number is left out,
// since with all ids' bits set it would be the empty slot's mark.
inline void pack_limits(long long ids, int wave_lg, int *rows, int *shift)
{
    int bits = 1;
    while (bits < 31 && (1ll << bits) < ids)
        bits++;
    *shift = bits;
    const long long most = (1ll << (32 - bits)) - 1;
    // a pack holds up to 64 keys: its table needs 128 slots
    *rows = wave_lg < 7 || most < 2 ? 0 : most < kWave ? (int)most : kWave;
}

// Per-wave LDS ints after the tables: a 64-int mark array, then the wave's
// graph state of the batch mode.
constexpr int kMarkStride = kWave + 8;
// LDS ints besides the tables: per-wave marks, misc words, chunk totals.
inline int lds_extra_words(int threads)
{
    return (threads / kWave) * kMarkStride + 8 + kMaxChunks + 8;
}

// log2 of the smallest table for a hash source of degree d: >= 2d slots, >= 64.
inline int host_table_lg(long long d)
{
    int lg = kMinTableLg;
    while ((1ll << lg) < 2 * d)
        lg++;
    return lg;
}

}  // namespace trust
