// Dense core: the edges into a small set of high-degree vertices, counted
// with bit rows instead of hashed walks.  No counterpart in the reference;
// the count is the same.
//
// Let C be at most 32768 vertices with ids cid(x) in [0, |C|), and B(x) the
// row of N+(x) ∩ C over those ids.  A dense target is a v in C whose whole
// out-list lies in C, without repeats, with d+(v) >= t; a dense source is a
// u with d+(u) >= t whose core part has no repeats and holds a dense
// target.  For an edge u -> v from a dense source to a dense target every w
// in N+(u) ∩ N+(v) is in C, so
//
//     |N+(u) ∩ N+(v)| = popcount(B(u) & B(v)),
//
// which costs |C|/8 bytes of bit rows instead of min(d+(u), d+(v)) probes of
// 4-byte ids.  The walk index leaves these edges out (walk_index.hip, pass
// A) and one launch counts them.
//
// Choosing C.  Orientation runs from lower to higher degree (the degree the
// preprocessing ordered by), so the set of vertices above any such degree is
// closed under out-neighbours and all of its members with d+ >= t are dense
// targets.  Exact in-degrees would cost a
// global atomic per edge; an estimate (d+ plus 128x the in-count over every
// 128th entry of adj) picks the seed, the K0 highest estimates in a 64-bins-
// per-octave histogram, and the seed is then closed: each step adds the
// out-neighbours of the newest members, until nothing is added (at most
// kCoreSteps steps; a closure past 32768 vertices is retried from a halved
// seed, and below 256 the seed alone is kept).
// R-MAT's degrees come in classes (a vertex's expected degree depends on the
// bit pattern of its id): at scale 26 the 16k highest estimates close to
// 17.9k vertices whose edges carry 52% of the short-side walk's probes
// (43% with both ends' d+ >= 384), where the seed alone, cut inside one
// class by a noisy estimate, keeps 19%; sampling every 16th, 32nd, 64th or
// 128th entry closes to the same core.  The dense tests make the count exact
// for any C.
//
// Layout for the MI355X's eight XCDs: each row is cut into S slices of wd
// words (wd a power of two up to 32: a slice row is at most one 128-byte
// line) and the rows are stored slice-major, rows[s][cid][wd]; one slice of
// all rows is |C| x 128 bytes at most (2.3 MB for R-MAT 26's 17.9k-vertex
// core in 18 slices), within one XCD's 4 MB L2.  The index also stores each
// dense source's row B(u) (bsrc).  A work item is (dense source u, slice s):
// the wave reads u's slice of B(u), stages its dense targets' ids in LDS,
// and per target reads that target's slice row (16 bytes per lane) and adds
// the popcount of the AND.  Each slice has a queue; a wave serves its XCD's
// slices (x, x + 8, ...; hardware XCC_ID) first, then the others, so every
// item is counted once wherever the waves land and an XCD's L2 mostly
// serves its own slices.  (Slices of 36 words, two lines per row, measured
// 41 ms for R-MAT 26's dense edges.)
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <vector>

#include "core_items.h"
#include "engine.h"
#include "wave_ops.h"

namespace trust {

constexpr int kCoreSeedMax = 16384;  // K0
constexpr int kCoreSeedMin = 256;
constexpr int kCoreMax = 32768;      // |C| (int16 ids; at most 32 slices of 32 words)
constexpr int kCoreMaxSlices = 32;
constexpr int kCoreSteps = 6;        // closure steps
// The bound t on the degrees of dense edges, unless the caller gives one: a
// dense edge costs nC / 8 bytes of bit rows whatever its probes, so t grows
// with the core.  nC / 48 within [64, 384]: R-MAT 26 (17.9k vertices) fresh
// counts measured 253.6 ms at t = 256, 236.3 at 384, 236.8 at 512; R-MAT 24
// (12.9k) 44.4 ms at 192, 44.9 at 256, 45.3 at 384; counts of R-MAT 20 (6.2k)
// 1.81 ms at 96, 1.38 at 128, 1.46 at 192, 2.09 at 384.
constexpr int kCoreMinDegreeLow = 64, kCoreMinDegreeHigh = 384, kCorePerDegree = 48;
constexpr int kCoreSample = 128;     // in-degree sampled every 128th entry
constexpr int kCoreBins = 2048;      // histogram: est < 64 exact, then 64 bins per octave
constexpr int kCoreThreads = 256;
constexpr int kCoreQueueStride = 32; // one 128-byte line per slice queue
// misc words: the slice queues follow at 64
enum CoreMisc {
    kCmLong = 0,     // items of long lists (front of recs)
    kCmMembers = 2,  // vertices listed so far (past kCoreMax: the closure does not fit)
    kCmSources = 3,  // candidate rows: bsrc slots, and an item each (back of recs)
    kCmOver = 4,     // rows with d+ >= t
    kCmTake = 8,     // the seed's size
    kCmCut = 9,      // the seed's lowest histogram bin
    kCmDegree = 10,  // t
    kCmLevel = 16    // [k]: members before closure step k
};
constexpr int kCoreMiscWords = 64 + kCoreMaxSlices * kCoreQueueStride;

// A work item: dense targets pool[lo + t0, lo + t1) of the source whose
// row B(u) is bsrc[b].
template <typename OffT>
struct DenseRec {
    OffT lo;
    int32_t t0, t1, b;
};

__device__ __forceinline__ int core_bin(long long est)
{
    if (est < 64)
        return (int)max(est, 0ll);
    const int lg = 63 - __clzll((unsigned long long)est);
    return 64 + (lg - 6) * 64 + (int)((est >> (lg - 6)) & 63);
}

static int core_bin_host(long long est)
{
    if (est < 64)
        return (int)std::max(est, 0ll);
    int lg = 63;
    while (!((unsigned long long)est >> lg))
        lg--;
    return 64 + (lg - 6) * 64 + (int)((est >> (lg - 6)) & 63);
}

__global__ void __launch_bounds__(kCoreThreads)
core_sample_kernel(const int32_t *__restrict__ adj, long long E, int *__restrict__ din)
{
    const long long n = (E + kCoreSample - 1) / kCoreSample;
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x)
        atomicAdd(&din[adj[i * kCoreSample]], 1);
}

template <typename OffT>
__device__ __forceinline__ long long core_est(const OffT *beg, const int *din, long long x)
{
    const long long e = (long long)(beg[x + 1] - beg[x]) + (long long)kCoreSample * din[x];
    return min(e, (long long)INT32_MAX);
}

template <typename OffT>
__global__ void __launch_bounds__(kCoreThreads)
core_hist_kernel(const OffT *__restrict__ beg, long long V, const int *__restrict__ din,
                 unsigned *__restrict__ hist)
{
    __shared__ unsigned h[kCoreBins];
    for (int b = threadIdx.x; b < kCoreBins; b += blockDim.x)
        h[b] = 0;
    __syncthreads();
    for (long long x = (long long)blockIdx.x * blockDim.x + threadIdx.x; x < V;
         x += (long long)gridDim.x * blockDim.x)
        atomicAdd(&h[core_bin(core_est(beg, din, x))], 1u);
    __syncthreads();
    for (int b = threadIdx.x; b < kCoreBins; b += blockDim.x)
        if (h[b])
            atomicAdd(&hist[b], h[b]);
}

// The seed: the top bins, at most k0 vertices, no bin below bmin.  One
// workgroup; cut = the lowest bin, take = its vertices.
__global__ void __launch_bounds__(kCoreThreads)
core_cut_kernel(const unsigned *__restrict__ hist, int bmin, unsigned k0, unsigned *__restrict__ misc)
{
    constexpr int kPer = kCoreBins / kCoreThreads;
    __shared__ unsigned long long part[kCoreThreads];
    __shared__ unsigned best, cut;
    unsigned long long mine = 0;
    for (int k = 0; k < kPer; k++)
        mine += hist[threadIdx.x * kPer + k];
    part[threadIdx.x] = mine;
    if (threadIdx.x == 0) {
        best = 0;
        cut = kCoreBins;
    }
    __syncthreads();
    // suffix sums of the threads' counts: above = the bins past this thread's
    for (int off = 1; off < kCoreThreads; off <<= 1) {
        const unsigned long long y = threadIdx.x + off < kCoreThreads ? part[threadIdx.x + off] : 0;
        __syncthreads();
        part[threadIdx.x] += y;
        __syncthreads();
    }
    unsigned long long above = part[threadIdx.x] - mine;
    for (int k = kPer - 1; k >= 0; k--) {
        const int b = threadIdx.x * kPer + k;
        above += hist[b];
        if (above <= k0 && b >= bmin) {
            atomicMin(&cut, (unsigned)b);
            atomicMax(&best, (unsigned)above);
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        misc[kCmTake] = best;
        misc[kCmCut] = cut;
        misc[kCmMembers] = 0;
        misc[kCmLevel] = 0;
    }
}

// Appends x to the member list for the lanes with `add`.
__device__ __forceinline__ void core_append(bool add, int x, int *list, unsigned *members)
{
    const unsigned long long m = __ballot(add);
    if (!m)
        return;
    unsigned at = 0;
    if (lane_id() == 0)
        at = atomicAdd(members, (unsigned)__popcll(m));
    at = __builtin_amdgcn_readfirstlane(at) +
         __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0));
    if (add && at < (unsigned)kCoreMax)
        list[at] = x;
}

// flag[x] = 1 for the seed's vertices, 0 outside, and their list.
template <typename OffT>
__global__ void __launch_bounds__(kCoreThreads)
core_seed_kernel(const OffT *__restrict__ beg, long long V, const int *__restrict__ din,
                 int *__restrict__ flag, int *__restrict__ list, unsigned *__restrict__ misc)
{
    const int cut = (int)misc[kCmCut];
    const long long step = (long long)gridDim.x * blockDim.x;
    for (long long x0 = (long long)blockIdx.x * blockDim.x + (threadIdx.x & ~(kWave - 1)); x0 < V;
         x0 += step) {
        const long long x = x0 + lane_id();
        const bool in = x < V && core_bin(core_est(beg, din, x)) >= cut;
        if (x < V)
            flag[x] = in ? 1 : 0;
        core_append(in, (int)x, list, misc + kCmMembers);
    }
}

// Members listed before step k (the list's end as the step begins).
__global__ void core_level_kernel(unsigned *__restrict__ misc, int k)
{
    misc[kCmLevel + k + 1] = min(misc[kCmMembers], (unsigned)kCoreMax + 1u);
}

// Closure step k: a wave per member that step k - 1 added; its
// out-neighbours outside join the list.  Nothing once the list is full.
template <typename OffT>
__global__ void __launch_bounds__(kCoreThreads)
core_expand_kernel(const OffT *__restrict__ beg, const int32_t *__restrict__ adj,
                   int *__restrict__ flag, int *__restrict__ list, unsigned *__restrict__ misc, int k)
{
    constexpr int kWaves = kCoreThreads / kWave;
    const unsigned lo = misc[kCmLevel + k], hi = misc[kCmLevel + k + 1];
    if (hi > (unsigned)kCoreMax)
        return;
    const int lane = lane_id();
    for (unsigned m = lo + blockIdx.x * kWaves + threadIdx.x / kWave; m < hi;
         m += gridDim.x * kWaves) {
        const int x = __builtin_amdgcn_readfirstlane(list[m]);
        const long long p0 = (long long)beg[x], p1 = (long long)beg[x + 1];
        for (long long p = p0; p < p1; p += kWave) {
            const int w = p + lane < p1 ? adj[p + lane] : -1;
            const bool add = w >= 0 && flag[w] == 0 && atomicCAS(&flag[w], 0, 1) == 0;
            core_append(add, w, list, misc + kCmMembers);
        }
    }
}

// t of the core found, unless the caller gave one.
__global__ void core_degree_kernel(unsigned *__restrict__ misc, int thr)
{
    const int n = (int)min(misc[kCmMembers], (unsigned)kCoreMax);
    misc[kCmDegree] = (unsigned)(thr > 0 ? thr
                                         : min(max(n / kCorePerDegree, kCoreMinDegreeLow),
                                               kCoreMinDegreeHigh));
}

// flag (0/1) and its exclusive scan -> cid (int16, -1 outside) and coreV
__global__ void __launch_bounds__(kCoreThreads)
core_assign_kernel(long long V, const int *__restrict__ flag, const int *__restrict__ pos,
                   int16_t *__restrict__ cid, int *__restrict__ coreV)
{
    for (long long x = (long long)blockIdx.x * blockDim.x + threadIdx.x; x < V;
         x += (long long)gridDim.x * blockDim.x) {
        if (flag[x]) {
            cid[x] = (int16_t)pos[x];
            coreV[pos[x]] = (int)x;
        } else {
            cid[x] = -1;
        }
    }
}

// One workgroup per core vertex v: its Kb-bit row, kept (and v made a dense
// target) when d+(v) >= thr and every out-neighbour is a core vertex, once.
template <typename OffT>
__global__ void __launch_bounds__(kCoreThreads)
core_rows_kernel(const OffT *__restrict__ beg, const int32_t *__restrict__ adj,
                 const int16_t *__restrict__ cid, const int *__restrict__ coreV, int Kb, int S,
                 int thr, uint32_t *__restrict__ rows, uint32_t *__restrict__ dst_bits,
                 uint32_t *__restrict__ dense_cid)
{
    __shared__ uint32_t bits[kCoreMax / 32];
    __shared__ int bad;
    const int r = blockIdx.x;
    const int v = coreV[r];
    const OffT b0 = beg[v];
    const long long d = (long long)(beg[v + 1] - b0);
    if (d < thr || d > Kb)
        return;  // the whole workgroup
    const int words = Kb / 32;
    for (int i = threadIdx.x; i < words; i += blockDim.x)
        bits[i] = 0;
    if (threadIdx.x == 0)
        bad = 0;
    __syncthreads();
    for (long long j = threadIdx.x; j < d; j += blockDim.x) {
        const int c = cid[adj[(long long)b0 + j]];
        if (c < 0) {
            bad = 1;  // outside the core
            break;
        }
        const uint32_t m = 1u << (c & 31);
        if (atomicOr(&bits[c >> 5], m) & m) {
            bad = 1;  // a repeated neighbour
            break;
        }
    }
    __syncthreads();
    if (bad)
        return;
    const int wd = words / S;  // words of one slice
    for (int i = threadIdx.x; i < words; i += blockDim.x) {
        const int s = i / wd;
        rows[((size_t)s * Kb + r) * wd + (i - s * wd)] = bits[i];
    }
    if (threadIdx.x == 0) {
        atomicOr(&dst_bits[v >> 5], 1u << (v & 31));
        atomicOr(&dense_cid[r >> 5], 1u << (r & 31));
    }
}

// The dense sources: a wave takes 64 rows, and each row with d+ >= thr in
// turn: its core ids into an LDS bitmap, which checks for repeats and is the
// row B(u) (stored to bsrc for a dense source), and its dense targets' ids
// from the row's start of pool (pool has adj's indexing); then the row's
// work items, targets cut into kCorePart pieces.  A candidate row's slot b in
// bsrc is also its place from the back of recs (an empty item where it is no
// dense source, or has more than kCorePart targets: those fill recs from the
// front, so that the long ones are handed out first).  With an atomic per
// item the kernel ended no earlier than one counter took them: 11.5 ns each.
//
// R-MAT's long rows crowd at low ids, so a wave's share of the rows is those
// that start in equal ranges of entries (grab_row), several ranges per wave.
template <typename OffT>
__global__ void __launch_bounds__(kCoreThreads)
core_lists_kernel(const OffT *__restrict__ beg, const int32_t *__restrict__ adj, long long V,
                  const int16_t *__restrict__ cid, const uint32_t *__restrict__ dense_cid, int Kb,
                  int thr, uint16_t *__restrict__ pool, DenseRec<OffT> *__restrict__ recs,
                  long long cap, uint32_t *__restrict__ bsrc, long long nsrc_cap,
                  const long long *__restrict__ grab_row, long long ngrab,
                  unsigned *__restrict__ misc, uint32_t *__restrict__ src_bits)
{
    constexpr int kWaves = kCoreThreads / kWave;
    __shared__ uint32_t dc[kCoreMax / 32];
    __shared__ uint32_t seen_s[kWaves][kCoreMax / 32];
    const int words = Kb / 32;
    for (int i = threadIdx.x; i < words; i += blockDim.x)
        dc[i] = dense_cid[i];
    const int wave = threadIdx.x / kWave, lane = lane_id();
    uint32_t *seen = seen_s[wave];
    for (int i = lane; i < words; i += kWave)
        seen[i] = 0;
    __syncthreads();
    // the workgroup's candidate rows, one atomic for their bsrc slots
    __shared__ unsigned cand_s[kWaves], base_s;
    unsigned ncand = 0;
    const long long q0 = (long long)wave * gridDim.x + blockIdx.x;
    const long long qstep = (long long)gridDim.x * kWaves;
    for (long long q = q0; q < ngrab; q += qstep) {
        const long long r0 = grab_row[q], r1 = grab_row[q + 1];
        for (long long u0 = r0; u0 < r1; u0 += kWave) {
            const bool in = u0 + lane < r1;
            const long long d = in ? (long long)(beg[u0 + lane + 1] - beg[u0 + lane]) : 0;
            ncand += (unsigned)__popcll(__ballot(d >= thr));
        }
    }
    if (lane == 0)
        cand_s[wave] = ncand;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned all = 0;
        for (int w = 0; w < kWaves; w++)
            all += cand_s[w];
        base_s = all ? atomicAdd(&misc[kCmSources], all) : 0u;
    }
    __syncthreads();
    unsigned slot = base_s;
    for (int w = 0; w < wave; w++)
        slot += cand_s[w];
    for (long long q = q0; q < ngrab; q += qstep) {
        const long long r0 = grab_row[q], r1 = grab_row[q + 1];
      for (long long u0 = r0; u0 < r1; u0 += kWave) {
        const int n = (int)min((long long)kWave, r1 - u0);
        const long long d = lane < n ? (long long)(beg[u0 + lane + 1] - beg[u0 + lane]) : 0;
        unsigned long long cand = __ballot(d >= thr);
        while (cand) {
            const int i = __builtin_ctzll(cand);
            const unsigned b = slot++;
            cand &= cand - 1;
            const long long u = u0 + i;
            const long long lo = (long long)beg[u], hi = (long long)beg[u + 1];
            int nd = 0, dup = 0;
            constexpr int kW = 4;  // windows in flight
            for (long long p0 = lo; p0 < hi; p0 += kW * kWave) {
                int cw[kW];
#pragma unroll
                for (int k = 0; k < kW; k++) {
                    const long long at = p0 + k * kWave + lane;
                    cw[k] = at < hi ? adj[at] : -1;
                }
#pragma unroll
                for (int k = 0; k < kW; k++)
                    cw[k] = cw[k] >= 0 ? (int)cid[cw[k]] : -1;
#pragma unroll
                for (int k = 0; k < kW; k++) {
                    const int c = cw[k];
                    const bool core = c >= 0;
                    const bool dense = core && ((dc[c >> 5] >> (c & 31)) & 1u);
                    int rep = 0;
                    if (core) {
                        const uint32_t m = 1u << (c & 31);
                        rep = (atomicOr(&seen[c >> 5], m) & m) ? 1 : 0;
                    }
                    dup |= __ballot(rep) != 0ull;
                    const unsigned long long bd = __ballot(dense);
                    const int rd = (int)__builtin_amdgcn_mbcnt_hi(
                        (unsigned)(bd >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)bd, 0));
                    if (dense)
                        pool[lo + nd + rd] = (uint16_t)c;
                    nd += __popcll(bd);
                }
            }
            wave_sync();
            if (!dup && nd > 0 && (long long)b < nsrc_cap) {
                uint32_t *row = bsrc + (size_t)b * words;
                for (int k = lane; k < words; k += kWave)
                    row[k] = seen[k];
            }
            wave_sync();
            for (int k = lane; k < words; k += kWave)
                seen[k] = 0;
            wave_sync();
            if ((long long)b >= nsrc_cap)
                continue;
            const bool source = !dup && nd > 0;
            const int parts = source ? (nd + kCorePart - 1) / kCorePart : 0;
            DenseRec<OffT> rc;
            rc.lo = (OffT)lo;
            rc.t0 = 0;
            rc.t1 = parts == 1 ? nd : 0;
            rc.b = (int32_t)b;
            if (lane == 0)
                recs[cap - 1 - (long long)b] = rc;
            if (!source)
                continue;
            if (parts > 1 && lane < parts) {
                rc.t0 = lane * kCorePart;
                rc.t1 = min(nd, (lane + 1) * kCorePart);
                recs[atomicAdd(&misc[kCmLong], 1u)] = rc;
            }
            if (lane == 0)
                atomicOr(&src_bits[u >> 5], 1u << (u & 31));
        }
      }
    }
}

// grab_row[q] = the first row starting at or after entry q 2^lg
// (q <= ngrab; grab_row[ngrab] = V).
template <typename OffT>
__global__ void __launch_bounds__(kCoreThreads)
core_grabs_kernel(const OffT *__restrict__ beg, long long V, long long ngrab, int lg,
                  long long *__restrict__ grab_row)
{
    const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (q > ngrab)
        return;
    if (q == ngrab) {
        grab_row[q] = V;
        return;
    }
    const long long at = q << lg;
    long long lo = 0, hi = V;  // the first u in [0, V] with beg[u] >= at
    while (lo < hi) {
        const long long mid = (lo + hi) >> 1;
        if ((long long)beg[mid] >= at)
            hi = mid;
        else
            lo = mid + 1;
    }
    grab_row[q] = lo;
}

// Rows with d+ >= t (an upper bound on the dense sources).
template <typename OffT>
__global__ void __launch_bounds__(kCoreThreads)
core_rows_over_kernel(const OffT *__restrict__ beg, long long V, unsigned *__restrict__ misc)
{
    const long long thr = misc[kCmDegree];
    unsigned k = 0;
    for (long long x = (long long)blockIdx.x * blockDim.x + threadIdx.x; x < V;
         x += (long long)gridDim.x * blockDim.x)
        k += (long long)(beg[x + 1] - beg[x]) >= thr;
    k = (unsigned)wave_sum((unsigned long long)k);
    if (lane_id() == 0 && k)
        atomicAdd(misc + kCmOver, k);
}

// The counting launch.  A wave's item (r, s): u's slice s of B(u) from bsrc
// (16 bytes per lane) and the item's dense targets' ids staged in LDS, then
// one slice row per target: rows of wd = Kb/(32 S) words read as 16-byte
// pieces, wd/4 lanes per target, 64/(wd/4) targets at a time (8 for 32-word
// slices), kIn per lane in flight.
template <typename OffT>
__global__ void __launch_bounds__(kCoreThreads) __attribute__((amdgpu_waves_per_eu(8, 8)))
core_dense_kernel(const DenseRec<OffT> *__restrict__ recs, long long cap,
                  const unsigned *__restrict__ misc_in, unsigned *__restrict__ queues,
                  const uint16_t *__restrict__ pool, const uint32_t *__restrict__ bsrc,
                  const uint32_t *__restrict__ rows, int Kb, int S, TcCtl *__restrict__ ctl)
{
    constexpr int kWaves = kCoreThreads / kWave;
    constexpr int kIn = 8;
    __shared__ uint16_t tg_s[kWaves][kCorePart];
    const int wave = threadIdx.x / kWave, lane = lane_id();
    uint16_t *tg = tg_s[wave];
    const int words = Kb >> 5;                        // of a whole row
    const int wd = words / S;                         // of a slice row: 4, 8, 16 or 32
    const int L = wd >> 2;                            // lanes per target, 4 words each
    const int G = kWave / L;                          // targets per step
    const int g = lane / L, w4 = lane - g * L;        // lanes with g >= G idle
    const unsigned n_long = misc_in[kCmLong];
    const unsigned n = n_long + misc_in[kCmSources];
    unsigned long long acc = 0;
    // slices in the order: this XCD's (x, x + 8, ...), then the others
    const int x = xcc_id() & (kXcds - 1);
    const int n_own = x < S ? (S - 1 - x) / kXcds + 1 : 0;
    auto slice_at = [&](int i) {
        if (i < n_own)
            return x + kXcds * i;
        int k = i - n_own;
        for (int c = 0;; c++)
            if (c % kXcds != x && k-- == 0)
                return c;
    };
    // items per grab: a slice's counter takes an atomic every 11.5 ns, which
    // at one item each bounded the launch (R-MAT 20: 0.48 ms); four grabs per
    // wave of an XCD still level it
    const unsigned grab = min(max(n / (4u * (unsigned)gridDim.x * kWaves / kXcds), 1u), 16u);
    int vis = 0, s = slice_at(0);
    unsigned qn = 0;  // the next grab, taken while this one is counted
    if (lane == 0)
        qn = atomicAdd(&queues[s * kCoreQueueStride], grab);
    for (;;) {
        const unsigned q = __builtin_amdgcn_readfirstlane(qn);
        if (q >= n) {
            if (++vis == S)
                break;
            s = slice_at(vis);
            if (lane == 0)
                qn = atomicAdd(&queues[s * kCoreQueueStride], grab);
            continue;
        }
        if (lane == 0)
            qn = atomicAdd(&queues[s * kCoreQueueStride], grab);
        // the grab's items, one per lane
        const unsigned qi = min(q + (unsigned)min(lane, (int)grab - 1), n - 1);
        const DenseRec<OffT> mine =
            recs[qi < n_long ? (long long)qi : cap - 1 - (long long)(qi - n_long)];
        const int items = (int)min(grab, n - q);
        const uint4 *base = (const uint4 *)(rows + (size_t)s * Kb * wd) + w4;
        for (int i = 0; i < items; i++) {
            const int t0 = readlane(mine.t0, i), nt = readlane(mine.t1, i) - t0;
            if (nt <= 0)
                continue;  // not a source, or among the long ones
            const int b = readlane(mine.b, i);
            const uint4 bu = ((const uint4 *)(bsrc + (size_t)b * words + (size_t)s * wd))[w4];
            const uint16_t *src = pool + (long long)readlane(mine.lo, i) + t0;
            for (int j = lane; j < nt; j += kWave)
                tg[j] = src[j];
            if (__ballot((bu.x | bu.y | bu.z | bu.w) != 0u) == 0ull)
                continue;  // no core neighbour of u in this slice
            wave_sync();
            int t = g < G ? g : nt;
            for (; t + (kIn - 1) * G < nt; t += kIn * G) {
                uint4 y[kIn];
#pragma unroll
                for (int k = 0; k < kIn; k++)
                    y[k] = base[(size_t)tg[t + k * G] * L];
#pragma unroll
                for (int k = 0; k < kIn; k++)
                    acc += (unsigned long long)(__popc(y[k].x & bu.x) + __popc(y[k].y & bu.y) +
                                                __popc(y[k].z & bu.z) + __popc(y[k].w & bu.w));
            }
            for (; t < nt; t += G) {
                const uint4 y = base[(size_t)tg[t] * L];
                acc += (unsigned long long)(__popc(y.x & bu.x) + __popc(y.y & bu.y) +
                                            __popc(y.z & bu.z) + __popc(y.w & bu.w));
            }
            wave_sync();  // before the next item overwrites tg
        }
    }
    acc = wave_sum(acc);
    if (lane == 0 && acc)
        atomicAdd(&ctl->sums[blockIdx.x % kSumLines].count, acc);
}

// ------------------------------------------------------------------ host
// Sizes that the automatic rules read count rows that are not empty, so that
// a graph keeps its core when empty rows stand for ids that no edge names (of
// a graph without such ids 98.4 to 100% of the rows have an edge: R-MAT 10 to
// 24, Chung-Lu, ER, BA).
//
// The automatic seed: a power of two near twice the square root of them.  With
// more, the closure of a smaller graph leaves its top degree class: R-MAT 20
// closes to 6.2k vertices from 2048, 9.9k from 4096 and 30.5k from 8192
// (counts of 1.38, 1.60 and 2.39 ms); R-MAT 22 closes to 9.1k from 4096 and
// from 16384, R-MAT 24 to 12.9k from 4096 up, R-MAT 26 to 17.9k from 16384.
static int core_auto_seed(long long rows)
{
    int k = kCoreSeedMin;
    while (k < kCoreSeedMax && (double)k * (double)k < 4.0 * (double)rows)
        k *= 2;
    return k;
}

// The automatic core's sizes.  It needs lists that meet often and a count
// that its build (300 us at R-MAT 20) does not outweigh.  Index and count
// without and with the core: R-MAT 20, 8.5 M edges of 0.55 M vertices (15 to
// one) 1.35, 1.75 ms; 10.5 M (18) 1.68, 1.53 ms; R-MAT 21, 14 M (14) 1.90,
// 2.03 ms; R-MAT 22, 20 M (11.7) 2.5, 3.1 ms; R-MAT 23, 33 M (10.6) 3.6, 4.0
// ms, 41 M (12.3) 6.1, 5.0 ms; R-MAT 24, 66 M (11.2) 8.0, 7.7 ms.  A context
// that counts once also pays 2 ms for the buffers: R-MAT 20, 16 M 8.6, 10.5
// ms; R-MAT 21, 47 M 24.3, 19.9 ms.
static bool core_pays(const Ctx *ctx)
{
    const long long rows = ctx->g.rows, E = ctx->g.E;
    if (ctx->counts_once)
        return E >= 24ll << 20 && E >= 16 * rows;
    return E >= 9ll << 20 && E >= (E < 32ll << 20 ? 14 : 11) * rows;
}

void core_config(const Ctx *ctx, const trust_params &p, int *K, int *thr, bool *automatic)
{
    *K = 0;
    *thr = 0;
    *automatic = false;
    if (p.core_vertices < 0 || p.total_process > 1 || ctx->batch_ngraphs > 0)
        return;
    const int low = p.core_min_degree > 0 ? p.core_min_degree : kCoreMinDegreeLow;
    if (p.core_vertices > 0) {
        *K = p.core_vertices;
    } else if (core_pays(ctx) && ctx->g.max_deg >= 4ll * low) {
        // (a graph without such out-degrees cannot have the heavy tail the
        // automatic core asks for below: Chung-Lu 3.8M's fresh count skips
        // the check)
        *K = core_auto_seed(ctx->g.rows);
        *automatic = true;
    }
    if (*K)
        *thr = p.core_min_degree;  // 0: by the core's size
}

void core_drop(Ctx *ctx)
{
    CoreIndex &c = ctx->core;
    c.built = c.active = false;
    c.K = c.thr = c.nC = c.Kb = c.S = 0;
    c.dense_edges = c.dense_probes = 0;
}

void core_release(Ctx *ctx)
{
    CoreIndex &c = ctx->core;
    core_drop(ctx);
    for (DevBuf *b : {&c.flag, &c.cid, &c.pos, &c.coreV, &c.bits, &c.rows, &c.pool, &c.recs,
                      &c.bsrc, &c.grabs, &c.misc, &c.hist})
        b->release();
}

template <typename OffT>
static int core_build_t(Ctx *ctx)
{
    CoreIndex &c = ctx->core;
    const DevCsr &g = ctx->g;
    const long long V = g.V, E = g.E;
    const int K0 = c.want_K;
    const OffT *beg = (const OffT *)g.beg.p;
    const int32_t *adj = (const int32_t *)g.adj.p;
    hipStream_t st = ctx->stream;
    c.words = (V + 31) / 32;
    int rc;
    if ((rc = c.flag.ensure(sizeof(int) * (size_t)V)) ||
        (rc = c.pos.ensure(sizeof(int) * (size_t)(V + 1))) ||
        (rc = c.cid.ensure(sizeof(int16_t) * (size_t)V)) ||
        (rc = c.coreV.ensure(sizeof(int) * (size_t)kCoreMax)) ||
        (rc = c.bits.ensure(sizeof(uint32_t) * (size_t)(2 * c.words + kCoreMax / 32))) ||
        (rc = c.misc.ensure(sizeof(unsigned) * kCoreMiscWords)) ||
        (rc = c.hist.ensure(sizeof(unsigned) * kCoreBins)) ||
        (rc = ctx->side_bsum.ensure(sizeof(long long) * (size_t)(scan_blocks(V) + 1))))
        return rc;
    int *flag = (int *)c.flag.p;
    int *din = (int *)c.pos.p;  // the sampled in-counts, until the scan
    int *list = (int *)c.coreV.p;  // the members as they are found, until the scan
    uint32_t *bits = (uint32_t *)c.bits.p;
    uint32_t *dst_bits = bits, *src_bits = bits + c.words, *dense_cid = bits + 2 * c.words;
    unsigned *misc = (unsigned *)c.misc.p;
    const int blocks = 4 * ctx->num_cus;
    HIPCHK(launch_fill_u32((uint32_t *)din, 0u, V, st));
    HIPCHK(launch_fill_u32((uint32_t *)c.hist.p, 0u, kCoreBins, st));
    HIPCHK(launch_fill_u32(bits, 0u, 2 * c.words + kCoreMax / 32, st));
    HIPCHK(launch_fill_u32(misc, 0u, kCoreMiscWords, st));
    hipLaunchKernelGGL(core_sample_kernel, dim3(blocks), dim3(kCoreThreads), 0, st, adj, E, din);
    hipLaunchKernelGGL(core_hist_kernel<OffT>, dim3(blocks), dim3(kCoreThreads), 0, st, beg, V,
                       (const int *)din, (unsigned *)c.hist.p);
    HIPCHK(hipGetLastError());
    c.K = K0;
    c.built = true;
    c.active = false;
    // The seed and its closure, while it fits; a seed whose closure passes
    // kCoreMax vertices is halved and closed again (down to kCoreSeedMin),
    // and past that the last seed alone is the core (its targets are
    // whichever lists lie inside it).  All steps are queued at once (a step
    // with nothing to expand takes 3 us) and the host waits once.
    const int bmin = core_bin_host(c.want_thr > 0 ? c.want_thr : kCoreMinDegreeLow);
    unsigned h[kCmLevel];
    auto close = [&](int k0, int steps) -> int {
        hipLaunchKernelGGL(core_cut_kernel, dim3(1), dim3(kCoreThreads), 0, st,
                           (const unsigned *)c.hist.p, bmin, (unsigned)k0, misc);
        hipLaunchKernelGGL(core_seed_kernel<OffT>, dim3(blocks), dim3(kCoreThreads), 0, st, beg, V,
                           (const int *)din, flag, list, misc);
        for (int k = 0; k < steps; k++) {
            hipLaunchKernelGGL(core_level_kernel, dim3(1), dim3(1), 0, st, misc, k);
            // (the seed and what it adds are nearly all there is)
            hipLaunchKernelGGL(core_expand_kernel<OffT>, dim3(k < 2 ? 2 * blocks : blocks / 4),
                               dim3(kCoreThreads), 0, st, beg, adj, flag, list, misc, k);
        }
        hipLaunchKernelGGL(core_degree_kernel, dim3(1), dim3(1), 0, st, misc, c.want_thr);
        HIPCHK(launch_fill_u32(misc + kCmOver, 0u, 1, st));
        hipLaunchKernelGGL(core_rows_over_kernel<OffT>, dim3(blocks), dim3(kCoreThreads), 0, st, beg,
                           V, misc);
        HIPCHK(hipGetLastError());
        HIPCHK(hipMemcpyAsync(h, misc, sizeof(h), hipMemcpyDeviceToHost, st));
        HIPCHK(hipStreamSynchronize(st));
        return TRUST_OK;
    };
    for (int k0 = K0, steps = kCoreSteps;;) {
        if ((rc = close(k0, steps)))
            return rc;
        // The automatic core needs a heavy tail: its seed's smallest
        // estimates at least 2t (R-MAT 26: about 12k; a Chung-Lu graph capped
        // at degree 800 has no such vertices, and takes the reference walk
        // anyway)
        if (k0 == K0 && steps > 0 &&
            (h[kCmTake] == 0 ||
             (c.want_auto && (int)h[kCmCut] < core_bin_host(2ll * (long long)h[kCmDegree]))))
            return TRUST_OK;
        if (h[kCmTake] == 0) {  // no smaller seed: the last one alone
            k0 *= 2;
            steps = 0;
            continue;
        }
        if (h[kCmMembers] <= (unsigned)kCoreMax)
            break;
        if (k0 / 2 >= kCoreSeedMin)
            k0 /= 2;
        else
            steps = 0;  // the seed alone
    }
    const int thr = (int)h[kCmDegree];
    c.thr = thr;
    c.nsrc_cap = std::max<long long>(h[kCmOver], 1);
    c.cap = core_item_slots(c.nsrc_cap, E);
    const unsigned members = h[kCmMembers];
    // bit rows: S slices of wd words, wd a power of two in [4, 32]: a slice
    // row is at most one 128-byte line (a lane reads 16 bytes of it)
    const int nC = (int)members;
    int wd = 4;
    while (wd < 32 && wd * 32 * kXcds < nC)
        wd <<= 1;
    const int S = (nC + 32 * wd - 1) / (32 * wd);
    const int Kb = wd * 32 * S;
    c.nC = nC;
    c.Kb = Kb;
    c.S = S;
    // ranges of entries that the lists kernel's waves take, four per wave
    const unsigned lblocks = (unsigned)(8 * ctx->num_cus);
    int grab_lg = 9;
    while (grab_lg < 20 && (E >> grab_lg) > 16ll * lblocks)
        grab_lg++;
    const long long ngrab = (E >> grab_lg) + 1;
    if ((rc = c.rows.ensure((size_t)Kb * (size_t)Kb / 8)) ||
        (rc = c.pool.ensure(sizeof(uint16_t) * (size_t)E)) ||
        (rc = c.recs.ensure(sizeof(DenseRec<OffT>) * (size_t)c.cap)) ||
        (rc = c.bsrc.ensure((size_t)c.nsrc_cap * (size_t)Kb / 8)) ||
        (rc = c.grabs.ensure(sizeof(long long) * (size_t)(ngrab + 1))))
        return rc;
    HIPCHK(launch_scan<int32_t>(flag, nullptr, V, (long long *)ctx->side_bsum.p, (int32_t *)c.pos.p,
                                st));
    hipLaunchKernelGGL(core_assign_kernel, dim3(blocks), dim3(kCoreThreads), 0, st, V,
                       (const int *)flag, (const int *)c.pos.p, (int16_t *)c.cid.p,
                       (int *)c.coreV.p);
    hipLaunchKernelGGL(core_rows_kernel<OffT>, dim3((unsigned)nC), dim3(kCoreThreads), 0, st, beg,
                       adj, (const int16_t *)c.cid.p, (const int *)c.coreV.p, Kb, S, thr,
                       (uint32_t *)c.rows.p, dst_bits, dense_cid);
    hipLaunchKernelGGL(core_grabs_kernel<OffT>,
                       dim3((unsigned)((ngrab + kCoreThreads) / kCoreThreads)), dim3(kCoreThreads),
                       0, st, beg, V, ngrab, grab_lg, (long long *)c.grabs.p);
    hipLaunchKernelGGL(core_lists_kernel<OffT>, dim3(lblocks),
                       dim3(kCoreThreads), 0, st, beg, adj, V, (const int16_t *)c.cid.p,
                       (const uint32_t *)dense_cid, Kb, thr, (uint16_t *)c.pool.p,
                       (DenseRec<OffT> *)c.recs.p, c.cap, (uint32_t *)c.bsrc.p, c.nsrc_cap,
                       (const long long *)c.grabs.p, ngrab, misc, src_bits);
    HIPCHK(hipGetLastError());
    c.active = true;
    return TRUST_OK;
}

int core_build(Ctx *ctx)
{
    CoreIndex &c = ctx->core;
    core_drop(ctx);
    const int K = c.want_K;
    if (K == 0 || ctx->g.V <= 0 || ctx->g.E <= 0) {
        c.built = true;
        return TRUST_OK;
    }
    if (K < kCoreSeedMin || K > kCoreSeedMax || (K & (K - 1)))
        return fail(TRUST_ERR_ARG, "core_vertices %d: a power of two in [%d, %d]", K,
                    kCoreSeedMin, kCoreSeedMax);
    if (c.want_thr < 0 || c.want_thr == 1)
        return fail(TRUST_ERR_ARG, "core_min_degree %d: 0 or >= 2", c.want_thr);
    return ctx->g.off64 ? core_build_t<int64_t>(ctx) : core_build_t<int32_t>(ctx);
}

int core_enqueue(Ctx *ctx, TcCtl *ctl, hipStream_t s)
{
    CoreIndex &c = ctx->core;
    if (!c.active)
        return TRUST_OK;
    unsigned *misc = (unsigned *)c.misc.p;
    HIPCHK(launch_fill_u32(misc + 64, 0u, kCoreMaxSlices * kCoreQueueStride, s));
    const int blocks = 8 * ctx->num_cus;
    if (ctx->g.off64)
        hipLaunchKernelGGL(core_dense_kernel<int64_t>, dim3(blocks), dim3(kCoreThreads), 0, s,
                           (const DenseRec<int64_t> *)c.recs.p, c.cap, (const unsigned *)misc,
                           misc + 64, (const uint16_t *)c.pool.p, (const uint32_t *)c.bsrc.p,
                           (const uint32_t *)c.rows.p, c.Kb, c.S, ctl);
    else
        hipLaunchKernelGGL(core_dense_kernel<int32_t>, dim3(blocks), dim3(kCoreThreads), 0, s,
                           (const DenseRec<int32_t> *)c.recs.p, c.cap, (const unsigned *)misc,
                           misc + 64, (const uint16_t *)c.pool.p, (const uint32_t *)c.bsrc.p,
                           (const uint32_t *)c.rows.p, c.Kb, c.S, ctl);
    HIPCHK(hipGetLastError());
    return TRUST_OK;
}

}  // namespace trust
