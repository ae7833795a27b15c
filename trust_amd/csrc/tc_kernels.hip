// gfx950 kernels for TRUST's vertex-centric hashed triangle count.
//
// Count = sum_u sum_{v in N+(u)} |N+(u) & N+(v)| over a degree-oriented CSR
// (reference semantics: Without-graph-partition/TC.cu:230-600; partitioned
// three-tile form: With-graph-partition/TC.cu:630-973).
//
// Design (MI355X-first, not a translation of the CUDA kernel):
//  * wave64 throughout.  A vertex is counted by one wavefront (wave tier),
//    by a whole workgroup with an LDS table (hub tier in the main launch,
//    big tier in a large-LDS launch) or by a whole workgroup with an HBM
//    table (spill tier).  Tables hold >= 2 slots per key, so they never
//    overflow (the reference drops entries past 100 per bucket,
//    TC.cu:293-301).  They are bucketed two-choice cuckoo tables: a lookup
//    is two 8-byte reads and branch-free compares, so no lane's probe chain
//    stalls its wave (the reference's linear_search scans a bucket,
//    TC.cu:70-110).  A vertex whose cuckoo insertion fails falls back to
//    linear probing, whose loops end at an empty slot.
//  * The probe walk takes 64 neighbours v of u at a time: lanes load
//    (beg[v], deg v), an inclusive wave scan (DPP row_shr / row_bcast) lays
//    the 64 lists end to end, and each 64-wide window of that concatenation
//    is one coalesced load per lane.  A batch of kU windows (four, or six
//    for the short-side walk's long lists) is in flight per wave before
//    any hash lookup, so each lane has kU independent loads outstanding.  The segment owning each lane is found with a
//    64-entry LDS mark array and a wave max-scan; a window inside a single
//    list skips that and reads its base with one readlane.  This replaces
//    the reference's per-lane skip loop with its 32-lane __shfl_sync
//    resynchronisation (TC.cu:513-541) and its 16x64 CTA walk that is only
//    correct at 1024 threads (TC.cu:330-359).
//  * A workgroup vertex splits its probe windows evenly over its waves
//    (per-chunk window counts, a prefix, then units of windows pulled from
//    an LDS counter), so no wave idles while another walks a long list.
//  * Persistent workgroups pull chunks of vertices from per-tier atomic
//    queues (the reference's G_INDEX counters, TC.cu:405-422,560-577);
//    logical rank r of P takes chunks c with c % P == r (TC.cu:259,433).
//  * Short rows of the wave tier are counted up to 64 at a time over one
//    shared table (packs); vertices of long walks in parts (tc_kernels.h).
//  * The count is reduced per wave in registers, per workgroup in LDS, and
//    added once per workgroup to one of 16 lines in device memory
//    (TC.cu:586-596).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "tc_kernels.h"
#include "wave_ops.h"

namespace trust {

constexpr int kEmpty = -1;
constexpr int kNoProbe = -2;  // a window position past the end: matches no slot

// The kernel's arguments, read through the kernel argument segment.  The
// fields are wave-uniform and loaded with scalar loads; held by value they
// stay in scalar registers across the whole probe walk, and the count kernel
// spilled 80-124 of them (into vector registers, which then spilled too).
// A pointer from args_again() hides that it is the same one, so a workgroup
// vertex loads the fields it needs afresh (from the scalar cache).  The wave
// tier's vertices are too short for that: their loads would wait for these.
template <typename OffT>
using ArgP = const __attribute__((address_space(4))) TcArgs<OffT> *;

template <typename OffT>
__device__ __forceinline__ ArgP<OffT> args_again()
{
    auto p = (ArgP<OffT>)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return p;
}

__device__ __forceinline__ unsigned long long uniform(unsigned long long x)
{
    const int lo = __builtin_amdgcn_readfirstlane((int)(x & 0xffffffffu));
    const int hi = __builtin_amdgcn_readfirstlane((int)(x >> 32));
    return ((unsigned long long)(unsigned int)hi << 32) | (unsigned int)lo;
}

// Per-wave attribution of triangles to the graphs of a batch.  The state
// sits in LDS, in the kMarkStride - kWave words after the wave's mark array,
// not in registers, where it would stay live across the whole probe walk and
// push other values out: (gs[0], gs[1]) = the vertex range of the graph being
// counted, gs[2] = that graph (-1: none), gs[4..5] = its triangles so far.
// Entering a vertex of another graph adds those to the previous graph, with
// a completion time stamp, and clears them.  Called with the whole wave
// active, u wave-uniform, before the vertex's hits are added.
__device__ __forceinline__ void graph_init(int *gs)
{
    if (lane_id() < kMarkStride - kWave)
        gs[lane_id()] = lane_id() == 2 ? -1 : 0;  // an empty range: the first vertex enters its graph
    wave_sync();
}

template <typename Args>
__device__ __forceinline__ void graph_flush(Args a, int *gs)
{
    const int g = __builtin_amdgcn_readfirstlane(gs[2]);
    if (g >= 0 && lane_id() == 0) {
        unsigned long long *total = (unsigned long long *)(gs + 4);
        if (*total)
            atomicAdd(a->graph_counts + g, *total);
        atomicMax(a->graph_done + g, (unsigned long long)wall_clock64());
        *total = 0;
    }
    wave_sync();
}

template <typename Args>
__device__ __forceinline__ void graph_enter(Args a, int *gs, int u)
{
    const int2 range = *(const int2 *)gs;
    if (u >= __builtin_amdgcn_readfirstlane(range.x) && u < __builtin_amdgcn_readfirstlane(range.y))
        return;
    graph_flush(a, gs);
    // the page of u bounds the search: vbase[lo] <= u < vbase[hi]
    const int pg = u >> a->graph_page_shift;
    int lo = a->graph_page[pg], hi = a->graph_page[pg + 1] + 1;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (a->graph_vbase[mid] <= u)
            lo = mid;
        else
            hi = mid;
    }
    const int g = __builtin_amdgcn_readfirstlane(lo);
    gs[0] = (int)a->graph_vbase[g];  // every lane stores the same values
    gs[1] = (int)a->graph_vbase[g + 1];
    gs[2] = g;
    wave_sync();
}

// Adds a wave's hits and probes of one vertex (wave-uniform) to the sums in
// LDS: the workgroup's {triangles, probes}, in batch mode the triangles to
// the wave's current graph.
template <int kMode>
__device__ __forceinline__ void add_result(unsigned long long *sum, int *mark,
                                           unsigned long long hits, unsigned long long probes)
{
    const int lane = lane_id();
    if constexpr (kMode == kModeBatch) {
        if (lane == 0)
            *(unsigned long long *)(mark + kWave + 4) += hits;
        if (lane == 1)
            atomicAdd(sum + 1, probes);
    } else {
        if (lane < 2)
            atomicAdd(sum + lane, lane == 0 ? hits : probes);
    }
}

// ---------------------------------------------------------- hash tables
__device__ __forceinline__ int ceil_lg(int x)  // smallest lg with 2^lg >= x (x >= 1)
{
    return x > 1 ? 32 - __clz(x - 1) : 0;
}

// Table size for a hash source of degree d in a tier whose capacity is
// 2^cap_lg: >= 2d slots (the planner only sends vertices whose 2d fits).
__device__ __forceinline__ int table_lg(int d, int cap_lg)
{
    int lg = ceil_lg(2 * d);
    lg = lg < kMinTableLg ? kMinTableLg : lg;
    return lg > cap_lg ? cap_lg : lg;
}

// ---- bucketed two-choice cuckoo table (the lookup path) ----
// 2^lg int slots = 2^(lg-1) buckets of two slots.  A key lives in bucket
// b1 = key & mask or b2 = a multiplicative hash of key, so a lookup is
// exactly two 8-byte reads and branch-free compares: no probe chain whose
// longest lane would stall the whole wave.  Load factor <= 1/2, far below
// the ~0.89 limit of 2-way, 2-slot cuckoo hashing.  b2 multiplies the low
// 24 bits (a full-rate v_mul_u32_u24; the 32-bit multiply is quarter rate
// and the walk is instruction-bound) and takes the top bits of the low word;
// keys equal in their low 24 bits share both buckets, which a bucket pair's
// four slots absorb, and a failed insertion falls back to linear probing.
__device__ __forceinline__ unsigned int bucket1(int key, int lgb)
{
    return (unsigned int)key & ((1u << lgb) - 1u);
}
__device__ __forceinline__ unsigned int bucket2(int key, int lgb)
{
    // __umul24 returns int: shift the unsigned value (a logical shift)
    return (unsigned int)__umul24((unsigned int)key, 0x9E3779u) >> (32 - lgb);
}

template <bool kGlobal>
__device__ __forceinline__ int2 bucket_load(const int *tab, unsigned int b)
{
    if constexpr (kGlobal) {
        unsigned long long v = __hip_atomic_load((const unsigned long long *)tab + b,
                                                 __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return make_int2((int)(v & 0xffffffffu), (int)(v >> 32));
    } else {
        return *((const int2 *)tab + b);
    }
}

// Concurrent insertion: claim an empty slot in either bucket, else evict
// an occupant with an atomic exchange and carry it to its other bucket.
// Returns true when `kMaxKicks` evictions did not place every key (the
// caller then rebuilds the table with linear probing).
constexpr int kMaxKicks = 48;
__device__ __forceinline__ bool cuckoo_insert(int *tab, int lgb, int key)
{
    for (int it = 0; it < kMaxKicks; it++) {
        const unsigned int c1 = bucket1(key, lgb), c2 = bucket2(key, lgb);
        int prev = atomicCAS(tab + 2 * c1, kEmpty, key);
        if (prev == kEmpty || prev == key)
            return false;
        prev = atomicCAS(tab + 2 * c1 + 1, kEmpty, key);
        if (prev == kEmpty || prev == key)
            return false;
        prev = atomicCAS(tab + 2 * c2, kEmpty, key);
        if (prev == kEmpty || prev == key)
            return false;
        prev = atomicCAS(tab + 2 * c2 + 1, kEmpty, key);
        if (prev == kEmpty || prev == key)
            return false;
        const unsigned int slot = 2 * ((it & 1) ? c2 : c1) + (((unsigned int)it >> 1) & 1u);
        key = atomicExch(tab + slot, key);
        if (key == kEmpty)
            return false;
    }
    return true;
}

// Membership count of N keys (kNoProbe matches no slot), summed over
// the wave: the per-key hit masks are counted with scalar popcounts, which
// keeps vector instructions (the walk's bound) for the lookup itself.  All
// 64 lanes must call it.  Both buckets of every key are read at once:
// reading the second bucket only when the first is full (sound, as slots
// are never vacated) saves LDS reads but serialises two LDS round trips, and
// measured 12% slower at R-MAT 24.
template <bool kGlobal, int N>
__device__ __forceinline__ unsigned int cuckoo_count(const int *tab, int lg, const int (&w)[N])
{
    const int lgb = lg - 1;
    int2 x1[N], x2[N];
#pragma unroll
    for (int k = 0; k < N; k++) {
        x1[k] = bucket_load<kGlobal>(tab, bucket1(w[k], lgb));
        x2[k] = bucket_load<kGlobal>(tab, bucket2(w[k], lgb));
    }
    unsigned int hits = 0;
#pragma unroll
    for (int k = 0; k < N; k++) {
        // each compare's lane mask feeds a scalar OR and popcount directly
        const unsigned long long m = __builtin_amdgcn_ballot_w64(x1[k].x == w[k]) |
                                     __builtin_amdgcn_ballot_w64(x1[k].y == w[k]) |
                                     __builtin_amdgcn_ballot_w64(x2[k].x == w[k]) |
                                     __builtin_amdgcn_ballot_w64(x2[k].y == w[k]);
        hits += (unsigned int)__popcll(m);
    }
    return hits;
}

// ---- linear probing (fallback when a cuckoo insertion fails) ----

__device__ __forceinline__ unsigned int hash_slot(int key, int lg)
{
    return ((unsigned int)key * 0x9E3779B1u) >> (32 - lg);
}

template <bool kGlobal>
__device__ __forceinline__ int slot_load(const int *p)
{
    if constexpr (kGlobal)
        return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else
        return *p;
}

template <bool kGlobal>
__device__ __forceinline__ void slot_clear(int *p)
{
    if constexpr (kGlobal)
        __hip_atomic_store(p, kEmpty, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else
        *p = kEmpty;
}

__device__ __forceinline__ void table_insert(int *tab, int lg, int key)
{
    const unsigned int mask = (1u << lg) - 1u;
    unsigned int h = hash_slot(key, lg);
    for (;;) {
        int prev = atomicCAS(tab + h, kEmpty, key);
        if (prev == kEmpty || prev == key)
            return;
        h = (h + 1u) & mask;
    }
}

// Membership of up to N keys (key < 0: skip), summed over the wave.
// First slots of all keys are read together, then each key finishes its
// probe sequence.  All 64 lanes must call it.
template <bool kGlobal, int N>
__device__ __forceinline__ unsigned int linear_count(const int *tab, int lg, const int (&w)[N])
{
    const unsigned int mask = (1u << lg) - 1u;
    unsigned int h[N];
    int s[N];
#pragma unroll
    for (int k = 0; k < N; k++) {
        h[k] = hash_slot(w[k], lg);
        s[k] = w[k] >= 0 ? slot_load<kGlobal>(tab + h[k]) : kEmpty;
    }
    unsigned int hits = 0;
#pragma unroll
    for (int k = 0; k < N; k++) {
        if (w[k] < 0)
            continue;
        for (;;) {
            if (s[k] == w[k]) {
                hits++;
                break;
            }
            if (s[k] == kEmpty)
                break;
            h[k] = (h[k] + 1u) & mask;
            s[k] = slot_load<kGlobal>(tab + h[k]);
        }
    }
    return (unsigned int)wave_sum((unsigned long long)hits);
}

// ---------------------------------------------------------- probe walk
// Lane state for a group of up to 64 neighbours v (one per lane): this
// lane's list is positions [excl, incl) of the concatenation, whose element
// at position t is adjP[base + t].
template <typename OffT>
struct Group {
    int incl, excl, deg;
    OffT base;
    int total;  // uniform: sum of the 64 degrees
};

template <typename OffT>
__device__ __forceinline__ Group<OffT> make_group(OffT s, int deg)
{
    Group<OffT> g;
    g.deg = deg;
    g.incl = wave_scan_add(deg);
    g.excl = g.incl - deg;
    g.total = readlane(g.incl, 63);
    g.base = s - (OffT)g.excl;
    return g;
}

template <typename OffT>
__device__ __forceinline__ Group<OffT> load_group(int v, bool valid, const OffT *__restrict__ begP)
{
    OffT s = 0;
    int deg = 0;
    if (valid) {
        s = begP[v];
        deg = (int)(begP[v + 1] - s);
    }
    return make_group(s, deg);
}

// Group of 64 walk entries starting at entry `at` of the walk view.  A walk
// index that stores each entry's list start and length (entW) is read in
// place, coalesced, one load per entry; otherwise the entry is a vertex id whose offsets
// are looked up.
template <typename OffT>
__device__ __forceinline__ Group<OffT> walk_group(ArgP<OffT> a, OffT at, bool valid)
{
    if (a->entW) {
        OffT s = 0;
        int deg = 0;
        if (valid) {
            const WalkEntry<OffT> x = a->entW[at];
            s = x.start;
            deg = x.deg;
        }
        return make_group(s, deg);
    }
    return load_group(valid ? a->adjW[at] : 0, valid, a->begP);
}

// Probes windows [wbeg, wend) (64 positions each) of a group's
// concatenation against the table and returns the hits of the whole wave
// (wave-uniform; gather mode: the wave's checksum).  All 64 lanes must call
// it.  `mark` is this wave's 64-int LDS scratch: all-zero on entry and exit.
template <typename OffT, bool kGlobal, int kMode, int kU>
__device__ __forceinline__ unsigned long long probe_windows(const Group<OffT> &g, int wbeg, int wend,
                                                      const int32_t *__restrict__ adjP,
                                                      const int *tab, int lg, bool linear,
                                                      int *mark)
{
    const int lane = lane_id();
    const int bend = min(wend * kWave, g.total);
    const int b = wbeg * kWave;
    if (b >= bend)
        return 0;
    // segment holding position b = number of lists ending at or before b
    int carry = (int)__popcll(__ballot(g.incl <= b));
    // end and base of list `carry`, kept in scalar registers until it changes
    int carry_incl = readlane(g.incl, carry);
    OffT carry_base = readlane(g.base, carry);
    // Base of the window starting at position bk (< bend): adjP[base + t] is
    // position t.  A window inside one list takes the cached base; otherwise
    // each position's list comes from the mark array and a max-scan.
    auto window_base = [&](int bk) -> OffT {
        if (carry_incl >= bk + kWave)
            return carry_base;
        const unsigned int off = (unsigned int)(g.excl - bk);
        if (g.deg > 0 && off < (unsigned int)kWave)
            mark[off] = lane;
        wave_sync();
        const int m = mark[lane];
        mark[lane] = 0;
        wave_sync();
        const int j = max(wave_scan_max(m), carry);
        carry = readlane(j, 63);
        carry_incl = readlane(g.incl, carry);
        carry_base = readlane(g.base, carry);
        return shfl_idx(g.base, j);
    };
    unsigned long long total = 0;  // wave-uniform hits
    unsigned int checksum = 0;     // gather mode, per lane
    auto lookup = [&](const auto &w) {
        constexpr int N = (int)(sizeof(w) / sizeof(int));
        if constexpr (kMode == kModeGather) {
#pragma unroll
            for (int k = 0; k < N; k++)
                checksum += w[k] >= 0 ? (unsigned int)w[k] : 0u;
        } else if constexpr (N > 4 && N % 2 == 0) {
            // two halves, so that the table reads of one half and their
            // compares need only half the registers
            int lo[N / 2], hi[N / 2];
#pragma unroll
            for (int k = 0; k < N / 2; k++) {
                lo[k] = w[k];
                hi[k] = w[N / 2 + k];
            }
            total += linear ? linear_count<kGlobal, N / 2>(tab, lg, lo)
                            : cuckoo_count<kGlobal, N / 2>(tab, lg, lo);
            total += linear ? linear_count<kGlobal, N / 2>(tab, lg, hi)
                            : cuckoo_count<kGlobal, N / 2>(tab, lg, hi);
        } else {
            total += linear ? linear_count<kGlobal, N>(tab, lg, w)
                            : cuckoo_count<kGlobal, N>(tab, lg, w);
        }
    };
    if (bend - b <= kWave) {
        // a single window (most small vertices): one load, one lookup
        const OffT bj = window_base(b);
        const int t = b + lane;
        const int w1[1] = {t < bend ? adjP[bj + (OffT)t] : kNoProbe};
        lookup(w1);
    } else {
        // Element idx of adjP.  With int32 offsets adj holds fewer than 2^30
        // ids (the engine's rule), so the byte offset fits 32 bits and the
        // load takes a 32-bit offset from the scalar base: no sign extension
        // and no 64-bit address arithmetic per lane.
        auto load = [&](OffT idx) -> int {
            if constexpr (sizeof(OffT) == 4)
                return *(const int *)((const char *)adjP + ((uint32_t)idx << 2));
            else
                return adjP[idx];
        };
        auto bases = [&](int at, OffT (&bj)[kU]) {
#pragma unroll
            for (int k = 0; k < kU; k++)
                bj[k] = at + k * kWave < bend ? window_base(at + k * kWave) : (OffT)0;
        };
        // The loads of a batch lying entirely before bend.  Every lane loads
        // and nothing reads the results here: with no branch around the
        // loads the compiler knows exactly kU loads are younger than the
        // previous batch and waits for that batch alone.
        auto fetch_full = [&](int at, int (&w)[kU]) {
            OffT bj[kU];
            bases(at, bj);
#pragma unroll
            for (int k = 0; k < kU; k++)
                w[k] = load(bj[k] + (OffT)(at + k * kWave + lane));
        };
        // The last batch: positions past bend read adjP[0] (which exists,
        // since bend > 0) and are masked before the lookup.
        auto fetch_tail = [&](int at, int (&w)[kU]) {
            OffT bj[kU];
            bases(at, bj);
#pragma unroll
            for (int k = 0; k < kU; k++) {
                const int t = at + k * kWave + lane;
                w[k] = load(t < bend ? bj[k] + (OffT)t : (OffT)0);
            }
        };
        // Software pipeline over batches of kU windows: the next
        // batch's loads are in flight while the current one is looked up.
        constexpr int kBatch = kWave * kU;
        const int last = b + (bend - b - 1) / kBatch * kBatch;  // start of the last batch
        int wcur[kU];
        if (last == b) {
            fetch_tail(b, wcur);
        } else {
            fetch_full(b, wcur);
            for (int bn = b + kBatch; bn < last; bn += kBatch) {
                int wnext[kU];
                fetch_full(bn, wnext);
                lookup(wcur);
#pragma unroll
                for (int k = 0; k < kU; k++)
                    wcur[k] = wnext[k];
            }
            int wtail[kU];
            fetch_tail(last, wtail);
            lookup(wcur);
#pragma unroll
            for (int k = 0; k < kU; k++)
                wcur[k] = wtail[k];
        }
#pragma unroll
        for (int k = 0; k < kU; k++)
            wcur[k] = last + k * kWave + lane < bend ? wcur[k] : kNoProbe;
        lookup(wcur);
    }
    if constexpr (kMode == kModeGather)
        total += wave_sum((unsigned long long)checksum);
    return total;
}

// ------------------------------------------------------- per-vertex work
// Whole workgroup counts vertex u with a table at `tab` (LDS or HBM) of
// capacity 2^cap_lg.  misc[0]: unit cursor, misc[2]: window total;
// ctot: kMaxChunks+1 ints of LDS.
template <typename OffT, bool kGlobal, int kMode, int kU>
__device__ __forceinline__ void group_vertex(int u, int tier, long long at, int *tab, int cap_lg,
                                             int *mark, int *misc, int *ctot)
{
    constexpr bool kInstr = kMode == kModeInstr;
    constexpr bool kTable = kMode != kModeGather;
    ArgP<OffT> a = args_again<OffT>();
    if constexpr (kMode == kModeBatch)
        graph_enter(a, mark + kWave, u);
    unsigned long long t0 = 0;
    if (kInstr && threadIdx.x == 0)
        t0 = clock64();
    const int lane = lane_id();
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave);  // uniform
    const int tid = wave * kWave + lane;
    const int nwaves = blockDim.x / kWave;
    const OffT sH = a->begH[u];
    const int dH = (int)(a->begH[u + 1] - sH);
    OffT sW = a->begW[u];
    int dW = (int)(a->endW[u] - sW);
    int part = 0;
    if constexpr (!kGlobal) {
        const int parts = group_parts(dW, a->part_entries, tier);
        if (parts > 1) {
            // the vertex fills `parts` list positions in a row: this one's
            // number is the count of those before it
            const int32_t *list = a->list + at;
            for (int back = 1; back < parts; back += kWave) {
                const bool mine = back + lane < parts && back + lane <= at &&
                                  list[-(back + lane)] == u;
                const unsigned long long m = __ballot(mine);
                part += __popcll(m);
                if (~m)
                    break;
            }
            const int entries = a->part_entries << (tier == kTierBig ? kBigPartLg : 0);
            sW += (OffT)((long long)part * entries);
            dW = min(entries, dW - part * entries);
        }
    }
    const int lg = table_lg(dH, cap_lg);
    const int size = 1 << lg;
    if constexpr (kTable)
        for (int i = tid; i < size; i += blockDim.x)
            slot_clear<kGlobal>(tab + i);
    if (tid == 0) {
        misc[0] = 0;                       // window-unit cursor
        misc[3] = a->force_linear == 1;     // linear-probing table for this vertex
    }
    if constexpr (kGlobal)
        __threadfence();  // HBM slots: cleared values visible in L2 before any insert/lookup
    __syncthreads();
    bool linear = false;
    if constexpr (kTable) {
        bool failed = a->force_linear == 2;  // forced: rebuild after the cuckoo attempt
        if (a->force_linear != 1)
            for (int i = tid; i < dH; i += blockDim.x)
                failed |= cuckoo_insert(tab, lg - 1, a->adjH[sH + (OffT)i]);
        if (failed)
            misc[3] = 1;  // benign race: every writer stores 1
        if constexpr (kGlobal)
            __threadfence();
        __syncthreads();
        linear = misc[3] != 0;
        if (linear) {  // rebuild this vertex's table with linear probing
            if (tid == 0 && a->force_linear != 1 && part == 0)
                atomicAdd(&a->ctl->rebuilds, 1ull);
            __syncthreads();
            for (int i = tid; i < size; i += blockDim.x)
                slot_clear<kGlobal>(tab + i);
            if constexpr (kGlobal)
                __threadfence();
            __syncthreads();
            for (int i = tid; i < dH; i += blockDim.x)
                table_insert(tab, lg, a->adjH[sH + (OffT)i]);
        }
    }
    if constexpr (kGlobal)
        __threadfence();
    __syncthreads();
    a = args_again<OffT>();
    const int nchunks = (dW + kWave - 1) / kWave;
    unsigned long long hits = 0;  // wave-uniform
    unsigned long long wave_probes = 0;
    if (nchunks <= kMaxChunks) {
        // window count of every 64-neighbour chunk, then an exclusive prefix
        for (int c = wave; c < nchunks; c += nwaves) {
            const int idx = c * kWave + lane;
            const Group<OffT> g = walk_group(a, sW + (OffT)idx, idx < dW);
            if (lane == 0)
                ctot[c] = (g.total + kWave - 1) / kWave;
            wave_probes += (unsigned long long)g.total;
        }
        __syncthreads();
        if (wave == 0) {
            int run = 0;
            for (int c0 = 0; c0 < nchunks; c0 += kWave) {
                const int x = c0 + lane < nchunks ? ctot[c0 + lane] : 0;
                const int inc = wave_scan_add(x);
                if (c0 + lane < nchunks)
                    ctot[c0 + lane] = run + inc - x;
                run += readlane(inc, 63);
            }
            if (lane == 0) {
                ctot[nchunks] = run;
                misc[2] = run;
            }
        }
        __syncthreads();
        const int TW = misc[2];
        // units of K windows, K a multiple of kU
        int K = TW / (nwaves * 4);
        K = K < kU ? kU : (K > 64 ? 64 : K);
        K = (K + kU - 1) / kU * kU;
        int cur = -1;
        Group<OffT> g = {0, 0, 0, 0, 0};
        for (;;) {
            int k = 0;
            if (lane == 0)
                k = atomicAdd(&misc[0], 1);
            k = __builtin_amdgcn_readfirstlane(k);
            int w0 = k * K;
            if (w0 >= TW)
                break;
            const int w1 = min(w0 + K, TW);
            while (w0 < w1) {
                int lo = 0, hi = nchunks;  // ctot[lo] <= w0 < ctot[hi]
                while (hi - lo > 1) {
                    const int mid = (lo + hi) >> 1;
                    if (ctot[mid] <= w0)
                        lo = mid;
                    else
                        hi = mid;
                }
                if (lo != cur) {
                    const int idx = lo * kWave + lane;
                    g = walk_group(a, sW + (OffT)idx, idx < dW);
                    cur = lo;
                }
                const int cend = min(w1, ctot[lo + 1]);
                hits += probe_windows<OffT, kGlobal, kMode, kU>(g, w0 - ctot[lo], cend - ctot[lo], a->adjP,
                                                     tab, lg, linear, mark);
                w0 = cend;
            }
        }
    } else {
        // very long walk lists: whole chunks pulled from the cursor
        for (;;) {
            int c = 0;
            if (lane == 0)
                c = atomicAdd(&misc[0], 1);
            c = __builtin_amdgcn_readfirstlane(c);
            if (c >= nchunks)
                break;
            const int idx = c * kWave + lane;
            const Group<OffT> g = walk_group(a, sW + (OffT)idx, idx < dW);
            wave_probes += (unsigned long long)g.total;
            hits += probe_windows<OffT, kGlobal, kMode, kU>(g, 0, (g.total + kWave - 1) / kWave, a->adjP, tab,
                                                 lg, linear, mark);
        }
    }
    add_result<kMode>((unsigned long long *)(misc + 4), mark, hits, wave_probes);
    __syncthreads();
    if constexpr (kInstr) {
        if (lane == 0 && wave_probes)
            atomicAdd(a->instr_probes + u, wave_probes);
        if (tid == 0)
            a->instr_cycles[u] = clock64() - t0;
    }
}

// One wavefront counts vertex u with its own LDS table slice.
template <typename OffT, int kMode, int kU>
__device__ __forceinline__ void wave_vertex(ArgP<OffT> a, int u, bool first, OffT sH, int dH,
                                            OffT sW, int dW, int *tab, int *mark,
                                            unsigned long long *sum)
{
    constexpr bool kInstr = kMode == kModeInstr;
    constexpr bool kTable = kMode != kModeGather;
    unsigned long long t0 = 0;
    if (kInstr)
        t0 = clock64();
    const int lane = lane_id();
    const int lg = table_lg(dH, a->wave_lg);
    const int size = 1 << lg;
    // On an unpartitioned graph the hashed row and the walked row are one
    // row: its first 64 ids, loaded for the table, also start the walk
    // (one dependent load less per vertex).
    const bool same_row = kTable && a->adjH == a->adjW && sH == sW && dH == dW;
    int head = 0;
    if constexpr (kTable)
        head = lane < dH ? a->adjH[sH + (OffT)lane] : 0;
    bool linear = false;
    if constexpr (kTable) {
        for (int i = lane; i < size; i += kWave)
            tab[i] = kEmpty;
        wave_sync();
        // force_linear 1: linear probing only; 2: rebuild after the cuckoo attempt
        bool failed = a->force_linear != 0;
        if (a->force_linear != 1) {
            if (lane < dH)
                failed |= cuckoo_insert(tab, lg - 1, head);
            for (int i = lane + kWave; i < dH; i += kWave)
                failed |= cuckoo_insert(tab, lg - 1, a->adjH[sH + (OffT)i]);
        }
        wave_sync();
        linear = __ballot(failed) != 0;
        if (linear) {  // rebuild this vertex's table with linear probing
            if (lane == 0 && a->force_linear != 1 && first)
                atomicAdd(&a->ctl->rebuilds, 1ull);
            for (int i = lane; i < size; i += kWave)
                tab[i] = kEmpty;
            wave_sync();
            for (int i = lane; i < dH; i += kWave)
                table_insert(tab, lg, a->adjH[sH + (OffT)i]);
            wave_sync();
        }
    }
    unsigned long long hits = 0;  // wave-uniform
    unsigned long long wave_probes = 0;
    for (int c = 0; c < dW; c += kWave) {
        const bool valid = c + lane < dW;
        Group<OffT> g;
        if (a->entW) {
            g = walk_group(a, sW + (OffT)(c + lane), valid);
        } else {
            const int v = c == 0 && same_row ? head : (valid ? a->adjW[sW + (OffT)(c + lane)] : 0);
            g = load_group(v, valid, a->begP);
        }
        wave_probes += (unsigned long long)g.total;
        hits += probe_windows<OffT, false, kMode, kU>(g, 0, (g.total + kWave - 1) / kWave, a->adjP, tab, lg,
                                           linear, mark);
    }
    wave_sync();
    add_result<kMode>(sum, mark, hits, wave_probes);
    if constexpr (kInstr) {
        if (lane == 0) {
            a->instr_probes[u] = wave_probes;
            a->instr_cycles[u] = clock64() - t0;
        }
    }
}

// ------------------------------------------------------------------ packs
// Vertices with short rows are counted several to a wave.  One at a time, a
// vertex of five neighbours costs the wave its table, its scans, a partly
// filled window or two and a chain of dependent loads, about 250
// instructions: on Chung-Lu (4.4 neighbours, 37 probes per vertex) the count
// was bound by issuing them.  Packs took it from 1.20 to 0.44 ms, and a batch
// of 400 ER/BA graphs (18 neighbours, 306 probes) from 8.4 to 7.3 ms.  A pack is a run of list positions whose rows
// hold at most 64 entries together: a lane per entry loads the ids, one
// table holds the keys of every row, tagged with the row's number in the
// pack, and the 64 probed lists are laid end to end as for one vertex, each
// position looked up with the tag of its entry's row.
//
// Ids take tag_shift bits, so id | row << tag_shift is exact; rows stay
// below pack_rows, which keeps every key off kEmpty and kNoProbe.  One id is
// often in many rows of a pack (hubs are), so the buckets depend on the row
// too.  A pack whose insertion fails is counted vertex by vertex.
constexpr int kPackLg = 8;  // table of 2^kPackLg slots (>= 4 per key), at most the wave's slice

__device__ __forceinline__ unsigned int pack_fold(unsigned int id, unsigned int row)
{
    return id + __umul24(row, 0x9E5u);
}

// Inserts key = id | row << shift; true: not placed within kMaxKicks.
__device__ __forceinline__ bool pack_insert(int *tab, int lgb, int key, int shift)
{
    for (int it = 0; it < kMaxKicks; it++) {
        const unsigned int f = pack_fold((unsigned int)key & ((1u << shift) - 1u),
                                         (unsigned int)key >> shift);
        const unsigned int c1 = bucket1((int)f, lgb), c2 = bucket2((int)f, lgb);
        for (unsigned int q = 0; q < 4; q++) {
            const int prev = atomicCAS(tab + 2 * (q < 2 ? c1 : c2) + (q & 1u), kEmpty, key);
            if (prev == kEmpty || prev == key)
                return false;
        }
        const unsigned int slot = 2 * ((it & 1) ? c2 : c1) + (((unsigned int)it >> 1) & 1u);
        key = atomicExch(tab + slot, key);
        if (key == kEmpty)
            return false;
    }
    return true;
}

// The row (lane index of the pack's rows) that holds each of the first
// `total` <= 64 entries; incl / d: a row's inclusive entry count and length.
__device__ __forceinline__ int pack_rows_of(int incl, int d, int n, int *mark)
{
    const int lane = lane_id();
    if (lane < n && d > 0)
        mark[incl - d] = lane;
    wave_sync();
    const int m = mark[lane];
    mark[lane] = 0;
    wave_sync();
    return wave_scan_max(m);
}

// Probes a pack's lists; `row`: this lane's entry's row.  Returns the
// wave's hits (gather mode: its checksum).
template <typename OffT, int kMode>
__device__ __forceinline__ unsigned long long probe_pack(const Group<OffT> &g, int row,
                                                         const int32_t *__restrict__ adjP,
                                                         const int *tab, int lg, int shift, int *mark)
{
    constexpr int kU = kUnroll;
    const int lane = lane_id();
    const int lgb = lg - 1;
    int carry = 0;  // list of the last position before the window
    unsigned long long total = 0;
    unsigned int checksum = 0;
    // ids of the windows at [at, at + kU * 64) and the rows they are probed for
    auto fetch = [&](int at, int (&w)[kU], int (&r)[kU]) {
        OffT idx[kU];
#pragma unroll
        for (int k = 0; k < kU; k++) {
            const int bk = at + k * kWave;
            idx[k] = 0;
            r[k] = 0;
            if (bk < g.total) {
                const unsigned int off = (unsigned int)(g.excl - bk);
                if (g.deg > 0 && off < (unsigned int)kWave)
                    mark[off] = lane;
                wave_sync();
                const int m = mark[lane];
                mark[lane] = 0;
                wave_sync();
                const int j = max(wave_scan_max(m), carry);
                carry = readlane(j, 63);
                const OffT b = shfl_idx(g.base, j);  // with every lane active
                r[k] = shfl_idx(row, j);
                // positions past the end read adjP[0], which exists
                idx[k] = bk + lane < g.total ? b + (OffT)(bk + lane) : (OffT)0;
            }
        }
#pragma unroll
        for (int k = 0; k < kU; k++)
            w[k] = adjP[idx[k]];
    };
    auto lookup = [&](int at, const int (&w)[kU], const int (&r)[kU]) {
        if constexpr (kMode == kModeGather) {
#pragma unroll
            for (int k = 0; k < kU; k++)
                checksum += at + k * kWave + lane < g.total ? (unsigned int)w[k] : 0u;
        } else {
            int2 x1[kU], x2[kU];
            int key[kU];
#pragma unroll
            for (int k = 0; k < kU; k++) {
                const unsigned int f = pack_fold((unsigned int)w[k], (unsigned int)r[k]);
                key[k] = at + k * kWave + lane < g.total ? w[k] | r[k] << shift : kNoProbe;
                x1[k] = bucket_load<false>(tab, bucket1((int)f, lgb));
                x2[k] = bucket_load<false>(tab, bucket2((int)f, lgb));
            }
#pragma unroll
            for (int k = 0; k < kU; k++) {
                const unsigned long long m = __builtin_amdgcn_ballot_w64(x1[k].x == key[k]) |
                                             __builtin_amdgcn_ballot_w64(x1[k].y == key[k]) |
                                             __builtin_amdgcn_ballot_w64(x2[k].x == key[k]) |
                                             __builtin_amdgcn_ballot_w64(x2[k].y == key[k]);
                total += (unsigned int)__popcll(m);
            }
        }
    };
    int w[kU], r[kU];
    fetch(0, w, r);
    for (int at = 0;;) {
        const int next = at + kU * kWave;
        if (next >= g.total) {
            lookup(at, w, r);
            break;
        }
        int wn[kU], rn[kU];
        fetch(next, wn, rn);
        lookup(at, w, r);
#pragma unroll
        for (int k = 0; k < kU; k++) {
            w[k] = wn[k];
            r[k] = rn[k];
        }
        at = next;
    }
    if constexpr (kMode == kModeGather)
        total += wave_sum((unsigned long long)checksum);
    return total;
}

// Counts the vertices at list positions [i, ...) that fit one pack, at least
// one and none at or past `last`; returns how many.
template <typename OffT, int kMode, int kU>
__device__ __forceinline__ int wave_next(ArgP<OffT> a, long long i, long long last, int *tab,
                                         int *mark, unsigned long long *sum)
{
    constexpr bool kTable = kMode != kModeGather;
    const int lane = lane_id();
    const bool in = i + lane < last;
    int u = in ? a->list[i + lane] : 0;
    OffT sH = 0, sW = 0;
    int dH = 0, dW = 0, part = 0;
    const bool split = a->wave_part != 0;
    const bool same = !split && a->begH == a->begW && a->adjH == a->adjW;
    if (split) {
        part = (int)((unsigned int)u >> kPartShift);
        u &= (1 << kPartShift) - 1;
    }
    if (in) {
        sH = a->begH[u];
        dH = (int)(a->begH[u + 1] - sH);
        if (same) {
            sW = sH;
            dW = dH;
        } else {
            sW = a->begW[u];
            dW = (int)(a->endW[u] - sW);
        }
        if (split) {  // this part's share of the walk
            const int parts = wave_parts(dW, a->wave_part);
            const int each = (dW + parts - 1) / parts;
            sW += (OffT)(part * each);
            dW = max(0, min(each, dW - part * each));
        }
    }
    const int u0 = readlane(u, 0);
    if constexpr (kMode == kModeBatch)
        graph_enter(a, mark + kWave, u0);
    if constexpr (kMode != kModeInstr) {
        const int iH = wave_scan_add(min(dH, kWave + 1));
        const int iW = same ? iH : wave_scan_add(min(dW, kWave + 1));
        bool fits = in && lane < a->pack_rows && iH <= kWave && iW <= kWave;
        if constexpr (kMode == kModeBatch) {  // one graph
            const int2 range = *(const int2 *)(mark + kWave);
            fits = fits && u >= range.x && u < range.y;
        }
        const unsigned long long out = ~__ballot(fits);
        const int n = out ? __builtin_ctzll(out) : kWave;
        if (n > 1) {
            const int shift = a->tag_shift;
            const int lg = min(kPackLg, a->wave_lg);
            int row = pack_rows_of(iH, dH, n, mark);
            const int keys = readlane(iH, n - 1);
            int id = 0;
            bool failed = false;
            if (kTable || same) {
                const OffT at = shfl_idx((OffT)(sH - (OffT)(iH - dH)), row) + (OffT)lane;
                id = lane < keys ? a->adjH[at] : 0;
            }
            if constexpr (kTable) {
                for (int k = lane; k < 1 << lg; k += kWave)
                    tab[k] = kEmpty;
                wave_sync();
                if (lane < keys)
                    failed = pack_insert(tab, lg - 1, id | row << shift, shift);
                wave_sync();
            }
            if (__ballot(failed) == 0) {
                int entries = keys;
                OffT at = 0;
                if (!same || a->entW) {
                    if (!same) {
                        row = pack_rows_of(iW, dW, n, mark);
                        entries = readlane(iW, n - 1);
                    }
                    at = shfl_idx((OffT)(sW - (OffT)(iW - dW)), row) + (OffT)lane;
                }
                const bool valid = lane < entries;
                const Group<OffT> g = !same || a->entW ? walk_group(a, at, valid)
                                                       : load_group(id, valid, a->begP);
                unsigned long long hits = 0;
                if (g.total > 0)
                    hits = probe_pack<OffT, kMode>(g, row, a->adjP, tab, lg, shift, mark);
                wave_sync();
                add_result<kMode>(sum, mark, hits, (unsigned long long)g.total);
                return n;
            }
        }
    }
    wave_vertex<OffT, kMode, kU>(a, u0, readlane(part, 0) == 0, readlane(sH, 0), readlane(dH, 0),
                                 readlane(sW, 0), readlane(dW, 0), tab, mark, sum);
    return 1;
}

// ------------------------------------------------------------ the kernel
// Chunks of `chunk` list positions that belong to this rank (chunk c is rank
// c % nranks's), out of a tier of `items` (< 2^31) positions.
__device__ __forceinline__ unsigned int rank_chunks(long long items, int chunk, int rank, int nranks)
{
    const unsigned int n = ((unsigned int)items + (unsigned int)chunk - 1u) / (unsigned int)chunk;
    if (nranks == 1)
        return n;
    return n > (unsigned int)rank
               ? (n - (unsigned int)rank + (unsigned int)nranks - 1u) / (unsigned int)nranks
               : 0u;
}

// A queue of n chunks over S counters (kShardStride apart).  Shard s hands
// out chunks s, s + S, ... (the list order is kept across shards), or with
// kContig the s-th contiguous part.  From S workgroups on every shard is the
// home of some of them (blockIdx % S).  A wave leaves its home only when that
// is empty, so a shard's last chunks are always taken; it then helps the next
// three shards, which level interleaved ones, and no more: looking for
// leftovers in all of them, 8192 waves took 94 us to find them empty at the
// end of every count.  Parts of unequal work, and shards that may have no
// home, are all tried.  All 64 lanes call; returns n when nothing is left.
constexpr unsigned int kShardTries = 4;
template <int S, bool kContig>
__device__ __forceinline__ unsigned int queue_take(unsigned int *next, unsigned int n,
                                                   unsigned int &shard, unsigned int groups)
{
    static_assert((S & (S - 1)) == 0, "a power of two");
    const unsigned int per = (n + S - 1) / S;
    auto share = [&](unsigned int s) -> unsigned int {  // chunks of shard s
        if constexpr (kContig)
            return s * per < n ? min(per, n - s * per) : 0u;
        else
            return (n + S - 1u - s) / S;
    };
    const unsigned int tries = kContig || groups < S ? S : kShardTries;
    for (unsigned int dry = 0;;) {
        unsigned int k = 0;
        if (lane_id() == 0)
            k = atomicAdd(next + shard * kShardStride, 1u);
        k = __builtin_amdgcn_readfirstlane(k);
        if (k < share(shard))
            return kContig ? shard * per + k : k * S + shard;
        if (++dry >= tries)
            return n;
        shard = (shard + 1) & (S - 1);
    }
}

// No more chunks than workgroups: workgroup b counts chunk b, no counter is
// touched.  The queue's bounds are read again for each chunk: held in scalar
// registers they would be live across the probe walk.
constexpr unsigned int kFixed = ~0u;
template <typename OffT, int kMode, bool kGlobal, int kU>
__device__ __forceinline__ void group_phase(int tier, unsigned int groups,
                                            int *tab, int cap_lg, int *mark, int *misc, int *ctot)
{
    unsigned int shard = blockIdx.x % kGroupShards;
    do {
        ArgP<OffT> a = args_again<OffT>();
        const long long lb = a->ctl->list_begin[tier], le = a->ctl->list_begin[tier + 1];
        const unsigned int n = rank_chunks(le - lb, a->chunk_group, a->rank, a->nranks);
        unsigned int k = blockIdx.x;
        if (n <= groups) {
            shard = kFixed;
        } else {
            __syncthreads();
            if (__builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave) == 0)
                misc[1] = (int)queue_take<kGroupShards, false>(a->ctl->group_next[tier], n, shard,
                                                               groups);
            __syncthreads();
            k = (unsigned int)__builtin_amdgcn_readfirstlane(misc[1]);
        }
        if (k >= n)
            break;
        const long long first = lb + ((long long)k * a->nranks + a->rank) * a->chunk_group;
        const long long last = min(first + (long long)a->chunk_group, le);
        for (long long i = first; i < last; i++)
            group_vertex<OffT, kGlobal, kMode, kU>(args_again<OffT>()->list[i], tier, i, tab, cap_lg,
                                                   mark, misc, ctot);
    } while (shard != kFixed);
}

// Waves per SIMD: with int32 offsets eight, and the compiler fits the
// kernel in 64 VGPRs (a few spills outside the probe loop).  The walk is
// latency-bound, and the eighth wave measured 15% faster at R-MAT 24 than
// seven waves without spills (1.6x at 1024-thread workgroups).  With int64
// offsets (64-bit window bases and list starts) 64 VGPRs spill inside the
// probe loop: seven waves (72 VGPRs) measured 25.4 ms on a 1000-graph batch
// against 33.4 ms at eight, 26.3 at six.  kBig: the large-LDS launch
// (HBM-table spill tier + big tier); otherwise the main launch (hub + wave
// tiers).  Each is compiled with only its own phases, so the registers of
// one do not constrain the other.
template <typename OffT>
constexpr int kMinWavesPerEU = sizeof(OffT) == 4 ? 8 : 7;

template <typename OffT, int kMode, bool kBig, int kU = kUnroll>
__global__ void __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(kMinWavesPerEU<OffT>, 8)))
tc_count_kernel(TcArgs<OffT>)
{
    ArgP<OffT> a = args_again<OffT>();
    extern __shared__ int lds[];
    const int nwaves = blockDim.x / kWave;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave);  // uniform
    const int lane = lane_id();
    int *mark = lds + a->table_words + wave * kMarkStride;  // + the graph state (batch mode)
    int *misc = lds + a->table_words + nwaves * kMarkStride;  // 8 words, the last four: sums
    int *ctot = misc + 8;                                     // kMaxChunks + 1 words
    unsigned long long *sum = (unsigned long long *)(misc + 4);  // triangles, probes
    mark[lane] = 0;
    if (wave == 0 && lane < 2)
        sum[lane] = 0;
    __syncthreads();
    if constexpr (kMode == kModeBatch) {
        graph_init(mark + kWave);
        if (wave == 0 && lane == 0)
            atomicMin(a->graph_t0, (unsigned long long)wall_clock64());
    }

    if (kBig && a->spill_tier >= 0 && (int)blockIdx.x < a->spill_groups) {
        int *tab = a->spill_mem + (long long)blockIdx.x * a->spill_slots;
        int cap_lg = 0;
        while ((2ll << cap_lg) <= a->spill_slots)
            cap_lg++;
        group_phase<OffT, kMode, true, kU>(a->spill_tier, (unsigned int)a->spill_groups, tab, cap_lg,
                                           mark, misc, ctot);
    }
    if (a->group_tier >= 0)
        group_phase<OffT, kMode, false, kU>(a->group_tier, gridDim.x, lds, a->group_lg, mark, misc,
                                            ctot);
    __syncthreads();  // the wave tables reuse the group table's LDS
    if (!kBig && a->wave_tier >= 0) {
        int *wtab = lds + wave * a->wave_slots;
        // Chunk j of the rank is chunk j * nranks + rank of the list, the
        // reference's interleave.  A single large graph interleaves the
        // shards, which spreads each vertex range over all eight L2s (R-MAT
        // 26: contiguous shards measured up to 3% slower).  A batch's list
        // is in graph order (the further parts of all graphs, if any, then
        // the vertices of all): its shards are contiguous eighths, one for the
        // workgroups of each XCD (dealt round-robin), so the graphs that an
        // XCD counts at a time stay in its L2 (10k-graph ER/BA batch: 4.8%
        // faster; four parts per XCD measured 17% slower than one).
        //
        // With no more chunks than waves, wave w takes chunk w and no
        // counter is touched; consecutive chunks go to different workgroups
        // (the list's first chunks are its heaviest).
        // The tier's list holds the parts beyond a vertex's first (wave_parts),
        // each a chunk of its own, then every vertex (its first part).
        const long long items = a->ctl->list_begin[kTierWave + 1] - a->ctl->list_begin[kTierWave];
        // (a batch's further parts are positions like the others)
        constexpr bool kBatch = kMode == kModeBatch;
        const unsigned int extra = kBatch ? 0u : (unsigned int)a->ctl->extra[kTierWave];
        const unsigned int whole = (unsigned int)items - extra;
        const unsigned int waves = gridDim.x * (unsigned int)nwaves;
        // chosen here: two grabs per wave at least, of at most 64 vertices; but
        // four per wave from the first quarter, since lists come in descending
        // length.  With a quarter's chunks as large as the others', the waves
        // that took 10 to 64 of the longest at once ended last: R-MAT 18
        // 775 us, now 570; R-MAT 22 with int64 offsets 2.65 ms, now 2.22.
        // Single vertices all along cost what packs give (Chung-Lu, 3.8 M
        // vertices: 450 us, 1040).  A batch's vertices come graph by graph.
        unsigned int chunk = a->chunk_wave, fchunk = 1, fronts = 0;
        if (a->chunk_wave <= 0) {
            const bool even = kBatch || a->chunk_wave < 0;
            chunk = even ? whole : whole - whole / 4;
            // a small batch, in the L2s as a whole, is dealt out without a
            // queue: emptying its eight shards cost more than the imbalance
            // (13 graphs of 900 to 2200 vertices 390 us, now 190; 200 of 100
            // to 200 246, 136; to 8 chunks' worth where lists may be long)
            if (kBatch && whole < (a->chunk_wave < 0 ? 32u : 8u) * waves)
                chunk = max(2u, (whole + waves - 1u) / waves);
            else
                chunk = max(1u, min((unsigned int)kWave, chunk / (2u * waves)));
            fchunk = max(1u, min(chunk, whole / (16u * waves)));
            fronts = even ? 0 : whole / (4u * fchunk);
        }
        const unsigned int front = extra + fronts * fchunk;  // where the others begin
        const unsigned int n = rank_chunks(
            extra + fronts + ((unsigned int)items - front + chunk - 1u) / chunk, 1, a->rank, a->nranks);
        constexpr int kShards = kBatch ? kXcds : kWaveShards;
        const bool fixed = n <= waves;
        unsigned int shard = kBatch ? (unsigned int)xcc_id() : blockIdx.x % kShards;
        do {
            const unsigned int j = fixed ? (unsigned int)wave * gridDim.x + blockIdx.x
                                         : queue_take<kShards, kBatch>(a->ctl->wave_next, n, shard,
                                                                       gridDim.x);
            if (j >= n)
                break;
            const long long lb = a->ctl->list_begin[kTierWave], le = a->ctl->list_begin[kTierWave + 1];
            const unsigned int c = j * (unsigned int)a->nranks + (unsigned int)a->rank;
            unsigned int at = c, step = 1;
            if (kBatch || c >= extra + fronts) {
                at = front + (c - extra - fronts) * chunk;
                step = chunk;
            } else if (c >= extra) {
                at = extra + (c - extra) * fchunk;
                step = fchunk;
            }
            const long long first = lb + at;
            const long long last = min(first + (long long)step, le);
            for (long long i = first; i < last;)
                i += wave_next<OffT, kMode, kU>(a, i, last, wtab, mark, sum);
        } while (!fixed);
    }
    if constexpr (kMode == kModeBatch)
        graph_flush(a, mark + kWave);  // the batch total is the graphs' sum
    // one pair of atomics per workgroup
    __syncthreads();
    if (wave == 0 && lane < 2 && sum[lane] && (kMode != kModeBatch || lane == 1))
        atomicAdd(&a->ctl->sums[blockIdx.x % kSumLines].count + lane, sum[lane]);
}

// ------------------------------------------------------------- planning
// The degree split in two launches: each workgroup counts the tiers of its
// per_block vertices, then every workgroup sums the counts of those before it
// (at most kPlanBlocks, 32 bytes each) and writes its vertices' list
// positions in order.  The first launch also clears the control block.  With
// a fill, a count, a one-workgroup scan and a scatter a plan took 45-60 us
// however small the graph; this takes 10-15.
template <typename OffT>
__device__ __forceinline__ int plan_tier(const PlanArgs<OffT> &p, long long u, int &parts)
{
    const long long dH = (long long)(p.begH[u + 1] - p.begH[u]);
    const long long dW = (long long)(p.endW[u] - p.begW[u]);
    parts = 1;
    if (dH == 0 || dW == 0 || (p.same_csr && dH < 2))
        return kTierNone;  // contributes nothing (reference skips d+ < 2, TC.cu:440-441)
    int lg = kMinTableLg;
    while ((1ll << lg) < 2 * dH)
        lg++;
    if (p.force_spill || lg > max(p.hub_lg, p.big_lg))
        return kTierSpill;
    if (lg > p.hub_lg) {
        parts = group_parts((int)dW, p.part_entries, kTierBig);
        return kTierBig;
    }
    if ((!p.wave_only && dW > p.hub_threshold) || lg > p.wave_lg) {
        parts = group_parts((int)dW, p.part_entries, kTierHub);
        return kTierHub;
    }
    if (p.wave_part)
        parts = wave_parts((int)dW, p.wave_part);
    return kTierWave;
}

__device__ __forceinline__ int wave_total(int x) { return readlane(wave_scan_add(x), kWave - 1); }

template <typename OffT>
__global__ void __launch_bounds__(1024) plan_count_kernel(PlanArgs<OffT> p)
{
    __shared__ int cnt[2 * kNumTiers];  // list positions, then those beyond one per vertex
    if (threadIdx.x < 2 * kNumTiers)
        cnt[threadIdx.x] = 0;
    if (blockIdx.x == 0)
        for (int i = threadIdx.x; i < (int)(sizeof(TcCtl) / 4); i += blockDim.x)
            ((uint32_t *)p.ctl)[i] = 0;
    __syncthreads();
    const long long lo = (long long)blockIdx.x * p.per_block;
    const long long hi = min(lo + p.per_block, p.V);
    int n[kNumTiers] = {0, 0, 0, 0}, more[kNumTiers] = {0, 0, 0, 0};
    for (long long u0 = lo; u0 < hi; u0 += blockDim.x) {
        const long long u = u0 + threadIdx.x;
        int parts = 1;
        const int t = u < hi ? plan_tier(p, u, parts) : kTierNone;
        const bool split = __ballot(parts > 1) != 0;
#pragma unroll
        for (int q = 0; q < kNumTiers; q++) {
            n[q] += __popcll(__ballot(t == q));
            if (split)
                more[q] += wave_total(t == q ? parts - 1 : 0);
        }
    }
    if (lane_id() == 0)
        for (int q = 0; q < kNumTiers; q++) {
            if (n[q])
                atomicAdd(&cnt[q], n[q] + more[q]);
            if (more[q])
                atomicAdd(&cnt[kNumTiers + q], more[q]);
        }
    __syncthreads();
    if (threadIdx.x < 2 * kNumTiers)
        p.block_counts[(long long)blockIdx.x * 2 * kNumTiers + threadIdx.x] = cnt[threadIdx.x];
}

template <typename OffT>
// Above 80 SGPRs a CU holds one workgroup of 1024 threads instead of two
// (3.8 M vertices: 48 us, 30).
__global__ void __launch_bounds__(1024) __attribute__((amdgpu_num_sgpr(80)))
plan_scatter_kernel(PlanArgs<OffT> p, int nblocks)
{
    // index kNumTiers: the wave tier's parts beyond a vertex's first, which
    // come before its vertices
    constexpr int kRuns = kNumTiers + 1;
    __shared__ int all[2 * kNumTiers], before[kRuns];
    constexpr int kRow = 1024 / kWave;  // most waves in the workgroup
    __shared__ int wcount[kRuns][kRow];
    __shared__ int run[kRuns];
    const int wave = threadIdx.x / kWave, nwaves = blockDim.x / kWave;
    if (threadIdx.x < 2 * kNumTiers)
        all[threadIdx.x] = 0;
    if (threadIdx.x < kRuns)
        before[threadIdx.x] = 0;
    __syncthreads();
    {
        int sum[2 * kNumTiers] = {0}, mine[kRuns] = {0};
        for (int b = threadIdx.x; b < nblocks; b += blockDim.x) {
            const int4 c = ((const int4 *)p.block_counts)[2 * b];
            const int4 e = ((const int4 *)p.block_counts)[2 * b + 1];
            const int v[2 * kNumTiers] = {c.x, c.y, c.z, c.w, e.x, e.y, e.z, e.w};
#pragma unroll
            for (int q = 0; q < 2 * kNumTiers; q++) {
                sum[q] += v[q];
                if (q < kNumTiers && b < (int)blockIdx.x)
                    mine[q] += q == kTierWave ? v[q] - v[kNumTiers + q] : v[q];
            }
            if (b < (int)blockIdx.x)
                mine[kNumTiers] += v[kNumTiers + kTierWave];
        }
#pragma unroll
        for (int q = 0; q < 2 * kNumTiers; q++) {
            const int x = wave_total(sum[q]);
            if (lane_id() == 0 && x)
                atomicAdd(&all[q], x);
            if (q < kRuns) {
                const int y = wave_total(mine[q]);
                if (lane_id() == 0 && y)
                    atomicAdd(&before[q], y);
            }
        }
    }
    __syncthreads();
    if (threadIdx.x < kNumTiers) {
        int base = 0;
        for (int q = 0; q < (int)threadIdx.x; q++)
            base += all[q];
        if (threadIdx.x == kTierWave) {
            run[kNumTiers] = base + before[kNumTiers];
            run[kTierWave] = base + all[kNumTiers + kTierWave] + before[kTierWave];
        } else {
            run[threadIdx.x] = base + before[threadIdx.x];
        }
        if (blockIdx.x == 0) {
            p.ctl->list_begin[threadIdx.x] = base;
            p.ctl->extra[threadIdx.x] = all[kNumTiers + threadIdx.x];
            if (threadIdx.x == kNumTiers - 1)
                p.ctl->list_begin[kNumTiers] = base + all[threadIdx.x];
        }
    }
    __syncthreads();
    const long long lo = (long long)blockIdx.x * p.per_block;
    const long long hi = min(lo + p.per_block, p.V);
    for (long long u0 = lo; u0 < hi; u0 += blockDim.x) {
        const long long u = u0 + threadIdx.x;
        int parts = 1;
        const int tier = u < hi ? plan_tier(p, u, parts) : kTierNone;
        const bool split = __ballot(parts > 1) != 0;
        int pos = 0, more = 0;  // in the wave, within the tier (more: of the extra parts)
        // a vertex's positions lie side by side, but in the wave tier its
        // first stands among the vertices and the rest among the extras
        const int put = tier == kTierWave ? 1 : parts;
#pragma unroll
        for (int t = 0; t < kNumTiers; t++) {
            int total, at;
            if (!split || t == kTierWave) {
                const unsigned long long m = __ballot(tier == t);
                total = __popcll(m);
                at = __builtin_amdgcn_mbcnt_hi((unsigned int)(m >> 32),
                                               __builtin_amdgcn_mbcnt_lo((unsigned int)m, 0));
            } else {
                const int x = tier == t ? put : 0;
                const int incl = wave_scan_add(x);
                total = readlane(incl, kWave - 1);
                at = incl - x;
            }
            pos = tier == t ? at : pos;
            if (lane_id() == 0)
                wcount[t][wave] = total;
        }
        if (p.wave_part) {
            const int x = tier == kTierWave ? parts - 1 : 0;
            const int incl = split ? wave_scan_add(x) : 0;
            more = incl - x;
            if (lane_id() == kWave - 1)
                wcount[kNumTiers][wave] = incl;
        }
        __syncthreads();
        if (threadIdx.x < kRuns * kRow) {  // a wave's first position, per tier
            const int t = threadIdx.x / kRow, w = threadIdx.x % kRow;
            const int x = w < nwaves && (t < kNumTiers || p.wave_part) ? wcount[t][w] : 0;
            int incl = x;
#pragma unroll
            for (int d = 1; d < kRow; d *= 2) {
                const int y = __shfl_up(incl, d, kRow);
                incl += w >= d ? y : 0;
            }
            const int at = run[t] + incl;
            wcount[t][w] = at - x;
            if (w == kRow - 1)
                run[t] = at;
        }
        __syncthreads();
        if (tier < kNumTiers) {
            pos += wcount[tier][wave];
            for (int q = 0; q < put; q++)
                p.list[pos + q] = (int32_t)u;
            if (put < parts) {
                more += wcount[kNumTiers][wave];
                for (int q = 1; q < parts; q++)
                    p.list[more + q - 1] = (int32_t)u | q << kPartShift;
            }
        }
        __syncthreads();
    }
}

__global__ void offsets_to_i32_kernel(const int64_t *src, int32_t *dst, long long n)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x)
        dst[i] = (int32_t)src[i];
}

// ------------------------------------------------------ short-side walk
// The walk rows of the short-side walk.  Row x lists first the v in N+(x)
// with d+(v) <= d+(x) (N+(v) is probed against x's table), then the u with
// u -> x and d+(u) < d+(x) (N+(u) is probed against x's table); an edge from
// a vertex with d+ < 2 closes no triangle at that edge and is left out.
// Every oriented edge that can close a triangle lands in exactly one row.
//
// A wave takes 64 consecutive rows u, whose lists are contiguous in adj, and
// walks them in coalesced 64-wide windows; the row of each position comes
// from a mark array and a max-scan.
//   kPass 0: sums the probes of the reference walk and of the short-side
//            walk into stats[0], stats[1];
//   kPass 1: kept[u] = number of kept out-entries of row u (counted in LDS,
//            each row belongs to one wave), incnt[v] += 1 per in-entry;
//   kPass 2: writes the rows: out-entries at begX[u] + (LDS slot), in-entries
//            from the row's end down (incnt counts back to zero).  An entry x
//            is stored as its list's start and length (entX = {beg[x],
//            d+(x)}, one store), which the count reads in place of x.
// The entries' rows (rowX, the learned plan's features) follow from begX
// alone and are written afterwards, in order, by side_rows_kernel: in the
// scatter pass they were a third of the in-entries' random writes.
constexpr int kSideWin = 4;

template <typename OffT, int kPass>
__global__ void __launch_bounds__(256) side_pass_kernel(const OffT *__restrict__ beg,
                                                        const int32_t *__restrict__ adj,
                                                        long long V, int *__restrict__ incnt,
                                                        int *__restrict__ kept,
                                                        const OffT *__restrict__ begX,
                                                        WalkEntry<OffT> *__restrict__ entX,
                                                        unsigned long long *__restrict__ stats)
{
    unsigned long long w_ref = 0, w_short = 0;
    __shared__ int mark_s[4][kWave * kSideWin];
    __shared__ int rowcnt_s[4][kWave];
    const int wave = threadIdx.x / kWave, lane = lane_id();
    int *mark = mark_s[wave];
    int *rowcnt = rowcnt_s[wave];
    for (int k = 0; k < kSideWin; k++)
        mark[k * kWave + lane] = 0;
    const long long step = (long long)gridDim.x * (blockDim.x / kWave) * kWave;
    for (long long u0 = ((long long)blockIdx.x * (blockDim.x / kWave) + wave) * kWave; u0 < V;
         u0 += step) {
        const int n = (int)min((long long)kWave, V - u0);
        // lane i < n holds row u0 + i; lane n (if any) the end of the range
        const OffT s = beg[u0 + min(lane, n)];
        const int d = lane < n ? (int)(beg[u0 + lane + 1] - s) : 0;
        const long long e0 = (long long)readlane(s, 0);
        const long long e1 = n == kWave ? (long long)readlane(s, 63) + readlane(d, 63)
                                        : (long long)readlane(s, n);
        rowcnt[lane] = 0;
        wave_sync();
        int carry = 0;
        for (long long p = e0; p < e1; p += kWave * kSideWin) {
            // a non-empty row starting inside this span marks its position
            if (d > 0 && (long long)s >= p && (long long)s < p + kWave * kSideWin)
                mark[(int)((long long)s - p)] = lane;
            wave_sync();
            int own[kSideWin], v[kSideWin];
#pragma unroll
            for (int k = 0; k < kSideWin; k++) {
                own[k] = max(wave_scan_max(mark[k * kWave + lane]), carry);
                carry = readlane(own[k], 63);
                const long long pos = p + k * kWave + lane;
                v[k] = pos < e1 ? adj[pos] : -1;
            }
            wave_sync();
#pragma unroll
            for (int k = 0; k < kSideWin; k++)
                mark[k * kWave + lane] = 0;
#pragma unroll
            for (int k = 0; k < kSideWin; k++) {
                const int du = shfl_idx(d, own[k]);
                OffT su = 0;  // beg[u], shuffled while every lane is active
                if constexpr (kPass == 2)
                    su = shfl_idx(s, own[k]);
                if (v[k] >= 0 && du >= 2) {
                    const OffT bv = beg[v[k]];
                    const int dv = (int)(beg[v[k] + 1] - bv);
                    if constexpr (kPass == 0) {
                        w_ref += (unsigned long long)dv;
                        w_short += (unsigned long long)min(du, dv);
                    } else if constexpr (kPass == 1) {
                        if (dv <= du)
                            atomicAdd(rowcnt + own[k], 1);
                        else
                            atomicAdd(incnt + v[k], 1);
                    } else {
                        const long long u = u0 + own[k];
                        if (dv <= du) {
                            const int slot = atomicAdd(rowcnt + own[k], 1);
                            const OffT at = begX[u] + (OffT)slot;
                            entX[at] = WalkEntry<OffT>{bv, dv};
                        } else {
                            const int k2 = atomicSub(incnt + v[k], 1);
                            const OffT at = begX[v[k] + 1] - (OffT)k2;
                            entX[at] = WalkEntry<OffT>{su, du};
                        }
                    }
                }
            }
            wave_sync();
        }
        if constexpr (kPass == 1) {
            if (lane < n)
                kept[u0 + lane] = rowcnt[lane];
        }
        wave_sync();
    }
    if constexpr (kPass == 0) {
        w_ref = wave_sum(w_ref);
        w_short = wave_sum(w_short);
        if (lane == 0 && w_ref) {
            atomicAdd(stats, w_ref);
            atomicAdd(stats + 1, w_short);
        }
    }
}

// rowX[at] = the row whose entries [begX[u], begX[u+1]) hold position at.
// A wave takes 64 consecutive rows, whose entries are contiguous, and
// writes them in 64-wide windows: each non-empty row marks its first
// position in LDS, and a max-scan carries the owner across the window.
template <typename OffT>
__global__ void __launch_bounds__(256) side_rows_kernel(const OffT *__restrict__ begX, long long V,
                                                        int32_t *__restrict__ rowX)
{
    __shared__ int mark_s[4][kWave];
    const int wave = threadIdx.x / kWave, lane = lane_id();
    int *mark = mark_s[wave];
    mark[lane] = 0;
    const long long step = (long long)gridDim.x * (blockDim.x / kWave) * kWave;
    for (long long u0 = ((long long)blockIdx.x * (blockDim.x / kWave) + wave) * kWave; u0 < V;
         u0 += step) {
        const int n = (int)min((long long)kWave, V - u0);
        // lane i < n: row u0 + i is [s, e); lane n (if any) holds the range's end in s
        const OffT s = begX[u0 + min(lane, n)];
        const OffT e = lane < n ? begX[u0 + lane + 1] : s;
        const long long p0 = (long long)readlane(s, 0);
        const long long p1 = n == kWave ? (long long)readlane(e, 63) : (long long)readlane(s, n);
        wave_sync();
        int carry = 0;
        for (long long w = p0; w < p1; w += kWave) {
            if (lane < n && e > s && (long long)s >= w && (long long)s < w + kWave)
                mark[(int)((long long)s - w)] = lane;
            wave_sync();
            const int own = max(wave_scan_max(mark[lane]), carry);
            carry = readlane(own, 63);
            wave_sync();
            mark[lane] = 0;
            if (w + lane < p1)
                rowX[w + lane] = (int32_t)(u0 + own);
            wave_sync();
        }
    }
}

template <typename OffT>
hipError_t launch_side_build(const OffT *beg, const int32_t *adj, long long V, int *cnt,
                             long long *bsum, OffT *begX, WalkEntry<OffT> *entX,
                             hipStream_t stream)
{
    if (V <= 0)
        return hipSuccess;
    int *incnt = cnt, *kept = cnt + V;
    const int pass_blocks = (int)min((V + 4 * kWave - 1) / (4 * kWave), 16384ll);
    hipError_t e = launch_fill_u32((uint32_t *)incnt, 0u, V, stream);
    if (e != hipSuccess)
        return e;
    hipLaunchKernelGGL((side_pass_kernel<OffT, 1>), dim3(pass_blocks), dim3(256), 0, stream,
                       beg, adj, V, incnt, kept, (const OffT *)nullptr,
                       (WalkEntry<OffT> *)nullptr, (unsigned long long *)nullptr);
    if ((e = launch_scan<OffT>(incnt, kept, V, bsum, begX, stream)) != hipSuccess)
        return e;
    hipLaunchKernelGGL((side_pass_kernel<OffT, 2>), dim3(pass_blocks), dim3(256), 0, stream,
                       beg, adj, V, incnt, (int *)nullptr, (const OffT *)begX, entX,
                       (unsigned long long *)nullptr);
    return hipGetLastError();
}

template <typename OffT>
hipError_t launch_side_rows(const OffT *begX, long long V, int32_t *rowX, hipStream_t stream)
{
    if (V <= 0)
        return hipSuccess;
    const int row_blocks = (int)min((V + 4 * kWave - 1) / (4 * kWave), 16384ll);
    hipLaunchKernelGGL((side_rows_kernel<OffT>), dim3(row_blocks), dim3(256), 0, stream, begX, V,
                       rowX);
    return hipGetLastError();
}

template hipError_t launch_side_build<int32_t>(const int32_t *, const int32_t *, long long, int *,
                                               long long *, int32_t *, WalkEntry<int32_t> *,
                                               hipStream_t);
template hipError_t launch_side_build<int64_t>(const int64_t *, const int32_t *, long long, int *,
                                               long long *, int64_t *, WalkEntry<int64_t> *,
                                               hipStream_t);
template hipError_t launch_side_rows<int32_t>(const int32_t *, long long, int32_t *, hipStream_t);
template hipError_t launch_side_rows<int64_t>(const int64_t *, long long, int32_t *, hipStream_t);

template <typename OffT>
hipError_t launch_side_stats(const OffT *beg, const int32_t *adj, long long V,
                             unsigned long long *stats, hipStream_t stream)
{
    hipError_t e = launch_fill_u32((uint32_t *)stats, 0u, 4, stream);
    if (e != hipSuccess || V <= 0)
        return e;
    const int pass_blocks = (int)min((V + 4 * kWave - 1) / (4 * kWave), 16384ll);
    hipLaunchKernelGGL((side_pass_kernel<OffT, 0>), dim3(pass_blocks), dim3(256), 0, stream,
                       beg, adj, V, (int *)nullptr, (int *)nullptr, (const OffT *)nullptr,
                       (WalkEntry<OffT> *)nullptr, stats);
    return hipGetLastError();
}

template <typename OffT>
__global__ void __launch_bounds__(256) start_index_kernel(const OffT *__restrict__ begP,
                                                          const int32_t *__restrict__ adj,
                                                          long long E,
                                                          WalkEntry<OffT> *__restrict__ entR)
{
    const long long stride = (long long)gridDim.x * blockDim.x;
    for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < E; e += stride) {
        const int v = adj[e];
        const OffT s = begP[v];
        entR[e] = WalkEntry<OffT>{s, (int32_t)(begP[v + 1] - s)};
    }
}

template <typename OffT>
hipError_t launch_start_index(const OffT *begP, const int32_t *adj, long long E,
                              WalkEntry<OffT> *entR, hipStream_t stream)
{
    if (E <= 0)
        return hipSuccess;
    const int blocks = (int)min((E + 255) / 256, 32768ll);
    hipLaunchKernelGGL((start_index_kernel<OffT>), dim3(blocks), dim3(256), 0, stream, begP, adj, E,
                       entR);
    return hipGetLastError();
}

template hipError_t launch_start_index<int32_t>(const int32_t *, const int32_t *, long long,
                                                WalkEntry<int32_t> *, hipStream_t);
template hipError_t launch_start_index<int64_t>(const int64_t *, const int32_t *, long long,
                                                WalkEntry<int64_t> *, hipStream_t);

template hipError_t launch_side_stats<int32_t>(const int32_t *, const int32_t *, long long,
                                               unsigned long long *, hipStream_t);
template hipError_t launch_side_stats<int64_t>(const int64_t *, const int32_t *, long long,
                                               unsigned long long *, hipStream_t);

// Plain streaming copy: the known-traffic kernel that calibrates HBM byte
// counters and gives the sequential-bandwidth reference.
__global__ void __launch_bounds__(256) copy_kernel(const int4 *__restrict__ src,
                                                   int4 *__restrict__ dst, long long n)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x)
        dst[i] = src[i];
}

hipError_t launch_copy(const int4 *src, int4 *dst, long long n, int blocks, hipStream_t stream)
{
    hipLaunchKernelGGL(copy_kernel, dim3(blocks), dim3(256), 0, stream, src, dst, n);
    return hipGetLastError();
}

// Every workgroup reads the whole buffer `reps` times from its own starting
// point: a buffer that fits the L2 measures the L2s' read rate (the dense
// core's bit rows are read from there).
__global__ void __launch_bounds__(256) read_kernel(const int4 *__restrict__ src, long long n,
                                                   int reps, unsigned *__restrict__ sink)
{
    unsigned acc = 0;
    const long long start = ((long long)blockIdx.x * 977) % n;
    for (int r = 0; r < reps; r++)
        for (long long i = threadIdx.x; i < n; i += blockDim.x) {
            long long j = i + start;
            if (j >= n)
                j -= n;
            const int4 x = src[j];
            acc += (unsigned)(x.x ^ x.y ^ x.z ^ x.w);
        }
    if (acc == 0x9e3779b9u)  // keeps the loads; practically never stores
        sink[blockIdx.x] = acc;
}

hipError_t launch_read(const int4 *src, long long n, int reps, int blocks, unsigned *sink,
                       hipStream_t stream)
{
    hipLaunchKernelGGL(read_kernel, dim3(blocks), dim3(256), 0, stream, src, n, reps, sink);
    return hipGetLastError();
}

__global__ void fill_u32_kernel(uint32_t *dst, uint32_t value, long long n)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x)
        dst[i] = value;
}

__global__ void totals_kernel(const TcCtl *__restrict__ ctl, int n, TcTotals *__restrict__ totals)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n)
        return;
    TcTotals t = {ctl[i].count, ctl[i].probes, ctl[i].rebuilds};
    for (int k = 0; k < kSumLines; k++) {
        t.count += ctl[i].sums[k].count;
        t.probes += ctl[i].sums[k].probes;
    }
    totals[i] = t;
}

// ------------------------------------------------------------- wrappers
hipError_t launch_totals(const TcCtl *ctl, int n, TcTotals *totals, hipStream_t stream)
{
    if (n <= 0)
        return hipSuccess;
    hipLaunchKernelGGL(totals_kernel, dim3((unsigned)(n + 63) / 64), dim3(64), 0, stream, ctl, n,
                       totals);
    return hipGetLastError();
}

template <typename OffT>
hipError_t launch_plan(PlanArgs<OffT> p, hipStream_t stream)
{
    // small graphs: many small workgroups; large ones: at most kPlanBlocks
    const int threads = p.V < (1 << 20) ? 256 : 1024;
    const long long per = std::max<long long>(1, (p.V + (long long)threads * kPlanBlocks - 1) /
                                                     ((long long)threads * kPlanBlocks));
    p.per_block = (int)(per * threads);
    const int nblocks = (int)std::max<long long>(1, (p.V + p.per_block - 1) / p.per_block);
    hipLaunchKernelGGL(plan_count_kernel<OffT>, dim3(nblocks), dim3(threads), 0, stream, p);
    hipLaunchKernelGGL(plan_scatter_kernel<OffT>, dim3(nblocks), dim3(threads), 0, stream, p, nblocks);
    return hipGetLastError();
}

template <typename OffT, bool kBig>
static void launch_count_t(const TcArgs<OffT> &a, int blocks, int threads, size_t lds_bytes,
                           int mode, hipStream_t stream)
{
    const bool deep = (mode & kProbeDeep) != 0;
    mode &= ~kProbeDeep;
    if (mode == kModeInstr)
        hipLaunchKernelGGL((tc_count_kernel<OffT, kModeInstr, kBig>), dim3(blocks), dim3(threads),
                           lds_bytes, stream, a);
    else if (mode == kModeGather && deep)
        hipLaunchKernelGGL((tc_count_kernel<OffT, kModeGather, kBig, kUnrollDeep>), dim3(blocks),
                           dim3(threads), lds_bytes, stream, a);
    else if (mode == kModeGather)
        hipLaunchKernelGGL((tc_count_kernel<OffT, kModeGather, kBig>), dim3(blocks), dim3(threads),
                           lds_bytes, stream, a);
    else if (mode == kModeBatch)
        hipLaunchKernelGGL((tc_count_kernel<OffT, kModeBatch, kBig>), dim3(blocks), dim3(threads),
                           lds_bytes, stream, a);
    else if (deep)
        hipLaunchKernelGGL((tc_count_kernel<OffT, kModeCount, kBig, kUnrollDeep>), dim3(blocks),
                           dim3(threads), lds_bytes, stream, a);
    else
        hipLaunchKernelGGL((tc_count_kernel<OffT, kModeCount, kBig>), dim3(blocks), dim3(threads),
                           lds_bytes, stream, a);
}

template <typename OffT>
hipError_t launch_count(const TcArgs<OffT> &a, int blocks, int threads, size_t lds_bytes,
                        int mode, bool big, hipStream_t stream)
{
    if (big)
        launch_count_t<OffT, true>(a, blocks, threads, lds_bytes, mode, stream);
    else
        launch_count_t<OffT, false>(a, blocks, threads, lds_bytes, mode, stream);
    return hipGetLastError();
}

template <typename OffT, bool kBig>
static hipError_t count_occupancy_t(int threads, size_t lds_bytes, int mode, int *blocks_per_cu)
{
    const bool deep = (mode & kProbeDeep) != 0;
    mode &= ~kProbeDeep;
    if (mode == kModeInstr)
        return hipOccupancyMaxActiveBlocksPerMultiprocessor(
            blocks_per_cu, tc_count_kernel<OffT, kModeInstr, kBig>, threads, lds_bytes);
    if (mode == kModeGather)
        return deep ? hipOccupancyMaxActiveBlocksPerMultiprocessor(
                          blocks_per_cu, tc_count_kernel<OffT, kModeGather, kBig, kUnrollDeep>,
                          threads, lds_bytes)
                    : hipOccupancyMaxActiveBlocksPerMultiprocessor(
                          blocks_per_cu, tc_count_kernel<OffT, kModeGather, kBig>, threads,
                          lds_bytes);
    if (mode == kModeBatch)
        return hipOccupancyMaxActiveBlocksPerMultiprocessor(
            blocks_per_cu, tc_count_kernel<OffT, kModeBatch, kBig>, threads, lds_bytes);
    return deep ? hipOccupancyMaxActiveBlocksPerMultiprocessor(
                      blocks_per_cu, tc_count_kernel<OffT, kModeCount, kBig, kUnrollDeep>, threads,
                      lds_bytes)
                : hipOccupancyMaxActiveBlocksPerMultiprocessor(
                      blocks_per_cu, tc_count_kernel<OffT, kModeCount, kBig>, threads, lds_bytes);
}

template <typename OffT>
hipError_t count_occupancy(int threads, size_t lds_bytes, int mode, bool big, int *blocks_per_cu)
{
    return big ? count_occupancy_t<OffT, true>(threads, lds_bytes, mode, blocks_per_cu)
               : count_occupancy_t<OffT, false>(threads, lds_bytes, mode, blocks_per_cu);
}

hipError_t launch_offsets_to_i32(const int64_t *src, int32_t *dst, long long n, hipStream_t stream)
{
    if (n <= 0)
        return hipSuccess;
    long long g = min((n + 255) / 256, 65536ll);
    hipLaunchKernelGGL(offsets_to_i32_kernel, dim3((unsigned)g), dim3(256), 0, stream, src, dst, n);
    return hipGetLastError();
}

hipError_t launch_fill_u32(uint32_t *dst, uint32_t value, long long n, hipStream_t stream)
{
    if (n <= 0)
        return hipSuccess;
    long long g = min((n + 255) / 256, 65536ll);
    hipLaunchKernelGGL(fill_u32_kernel, dim3((unsigned)g), dim3(256), 0, stream, dst, value, n);
    return hipGetLastError();
}

template hipError_t launch_plan<int32_t>(PlanArgs<int32_t>, hipStream_t);
template hipError_t launch_plan<int64_t>(PlanArgs<int64_t>, hipStream_t);
template hipError_t launch_count<int32_t>(const TcArgs<int32_t> &, int, int, size_t, int, bool,
                                          hipStream_t);
template hipError_t launch_count<int64_t>(const TcArgs<int64_t> &, int, int, size_t, int, bool,
                                          hipStream_t);
template hipError_t count_occupancy<int32_t>(int, size_t, int, bool, int *);
template hipError_t count_occupancy<int64_t>(int, size_t, int, bool, int *);

}  // namespace trust
