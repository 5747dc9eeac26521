// Cell-binned dk/dv: scatter turned into register accumulation.
//
// A sample's four bilinear taps are the 2x2 pixel block whose top-left pixel is
// (y0, x0) = floor of its pixel coordinate -- its "cell". Which cell a sample
// falls in depends on the coordinates only, not on the head, so one counting
// sort per (batch, key view) -- bin_count / bin_scan / bin_fill below -- orders
// the samples (s1, l, p) of every key view by cell, and all H heads reuse it.
//
// The dk/dv kernel then gives one wave to one (plane (b, h, s2), cell): the
// cell's four K and four V tap rows are loaded ONCE into registers; for every
// sample in the cell's list the wave gathers the sample's query row (q, dout,
// log-sum-exp, delta), recomputes p and ds, and adds w_t*ds*scale*q and
// w_t*p*dout into register accumulators for the four pixels. Only the cell's
// final sums go to memory: 8*D float atomics per non-empty cell instead of 8*D
// per sample (each pixel is shared by four cells, hence atomics for that last
// step). Heavy cells (clustered coordinates) are the best case, not the worst.
//
// Cells are indexed on a (Himg+1) x (Wimg+1) grid, y0 in [-1, Himg-1] and x0 in
// [-1, Wimg-1]: border cells hold the samples with some taps outside the image
// (weight 0 there, zero padding per tap). Samples with all four taps outside
// contribute nothing to dk/dv and are left out of the lists.
#pragma once
#include "dsdpa_common.h"

namespace dsdpa {

constexpr int kBinThreads = 256;
// Waves per workgroup of the dk/dv kernel. One: items differ in length by orders of magnitude (a heavy
// list's piece beside lists of a few entries), and a workgroup keeps its LDS and its place on the CU until
// its longest wave ends -- with four waves a workgroup the SIMDs held 2.1 waves on average where the
// registers allow 3 (64x64, 64 samples per view, clustered: 4.88 ms with four, 4.13 ms with one).
constexpr int kCellWaves = 1;

__device__ __forceinline__ int cell_of(const Taps &tp, int Wimg) { return (tp.y0 + 1) * (Wimg + 1) + (tp.x0 + 1); }

// Fractional position of a sample inside its cell: the bilinear weights are (1-fx)(1-fy), fx(1-fy), (1-fx)fy, fx*fy.
// The binning pass stores it beside the sample id (same order), so that the dk/dv kernel reads it in list order
// instead of gathering the coordinate pair again (a random 8-byte read per entry, per head).
__device__ __forceinline__ float2 cell_fraction(float2 xy, const Dims &dm)
{
    // (fused, so that the position keeps the bits that the rounded pixel coordinate drops, whatever the compiler
    // would contract where this is inlined)
    const float ax = (xy.x * 2.0f - 1.0f) + 1.0f, kx = (float)(dm.Wimg - 1) * 0.5f;
    const float ay = (xy.y * 2.0f - 1.0f) + 1.0f, ky = (float)(dm.Himg - 1) * 0.5f;
    return make_float2(fmaf(ax, kx, -floorf(ax * kx)), fmaf(ay, ky, -floorf(ay * ky)));
}

__device__ __forceinline__ bool taps_any(const Taps &tp)
{
    return (tp.w[0] != 0.f) | (tp.w[1] != 0.f) | (tp.w[2] != 0.f) | (tp.w[3] != 0.f);
}

// Lists are kept per key = (group of query views s1 / vpg, cell), NK = groups * NC keys per (batch, key view).
// With more than one group the dk/dv kernel works through a key view's lists one group of query views at a
// time, so that the query rows it gathers (q and dout of that group only) stay in the XCD's L2.
//
// One thread per coordinate pair, in memory order (b, s1, l, s2, p).
// mode 0: count[(b*V+s2)*NK + key] += 1
// mode 1: the sample's list entry at place (b*V+s2)*M + cursor[(b*V+s2)*NK + key]++: with `records` a 12-byte
//         record (id = (s1*L + l)*P + p, then its position (fx, fy) inside the cell as two floats) in `sorted` taken
//         as an array of records -- one scattered store per sample, and the dk/dv kernel reads id and position in
//         list order instead of gathering the coordinate pair again; without, the id alone as sorted[place] (the
//         deterministic backward sorts the ids of every list before use).
struct CellEntry { unsigned id; float fx, fy; };
__device__ __forceinline__ void store_cell_entry(unsigned *sorted, size_t place, unsigned id, const float2 &ff, int records)
{
    if (records) {
        unsigned *r = sorted + 3 * place;
        r[0] = id;
        r[1] = __float_as_uint(ff.x);
        r[2] = __float_as_uint(ff.y);
    } else {
        sorted[place] = id;
    }
}

template <int MODE>
__global__ __launch_bounds__(kBinThreads) void bin_samples_kernel(const float *__restrict__ coords_, Dims dm,
                                                                  int NC, int NK, int vpg,
                                                                  unsigned *__restrict__ counters,
                                                                  unsigned *__restrict__ sorted, int records)
{
    const long long total = (long long)dm.B * dm.V * dm.L * dm.N;
    const long long i = (long long)blockIdx.x * kBinThreads + threadIdx.x;
    if (i >= total) return;
    const float2 xy = reinterpret_cast<const float2 *>(coords_)[i];
    const Taps tp = make_taps(xy.x, xy.y, dm.Wimg, dm.Himg);
    if (!taps_any(tp)) return;
    const int p = (int)(i % dm.P);
    long long t = i / dm.P;
    const int s2 = (int)(t % dm.V);
    t /= dm.V;                                   // t = (b*V + s1)*L + l
    const int ql = (int)(t % ((long long)dm.V * dm.L));   // s1*L + l
    const int b = (int)(t / ((long long)dm.V * dm.L));
    const size_t grp = (size_t)b * dm.V + s2;
    unsigned *ctr = counters + grp * NK + (ql / dm.L / vpg) * NC + cell_of(tp, dm.Wimg);
    if (MODE == 0) {
        atomicAdd(ctr, 1u);
    } else {
        const unsigned pos = atomicAdd(ctr, 1u);
        const size_t M = (size_t)dm.V * dm.L * dm.P;
        store_cell_entry(sorted, grp * M + pos, (unsigned)ql * (unsigned)dm.P + (unsigned)p, cell_fraction(xy, dm), records);
    }
}

// LDS-aggregated variant of the two passes above. A workgroup takes kBinRunThreads * PER consecutive samples of one (b, s2), PER
// of them a thread, requested together and kept in registers, and histograms them in LDS first, so the contended global
// atomics drop from one per sample to one per (workgroup, non-empty cell).
// mode 0: global count[cell] += local count
// mode 1: every sample's rank among the workgroup's in its cell comes from the counting atomic; reserve
//         [base, base+local count) from the global cursor of each cell, then place every sample at base + rank.
// Bound by the chain load -> LDS atomic -> global atomic -> scattered store, and by the counters that every workgroup walks: one key
// view's, not all V views' of a run of query rows (V * NC counters, twice that LDS, and each sample read and worked out twice in
// the fill). Count, scan and fill, us, before / now: 48x48, 6 views x 32 samples, batch 2 148 / 72; 64x64, 4 x 64, batch 2,
// clustered 165 / 95; 32x32, 6 x 16 38 / 21; 40x28, 4 x 8, batch 2 30 / 14; 18x18, 6 x 6, batch 2 22 / 13.
// 512 threads: 1024 with half the samples each are even, but beside the staged dq kernel, whose 14 to 16 waves on every CU
// leave workgroups of 16 waves or of more than 64 registers no place until dq ends, dk/dv would wait behind them (14x14, 8 views x
// 32 samples: the three launches 41 us from first to last with four samples a thread, 194 with eight).
constexpr int kBinRunThreads = 512, kBinRunKeys = 20 * 1024;
template <int MODE, int PER>
__global__ __launch_bounds__(kBinRunThreads, PER <= 4 ? 8 : 4) void bin_samples_lds_kernel(
    const float *__restrict__ coords_, Dims dm, int NC, int NK, int vpg, int nlc,
    unsigned *__restrict__ counters, unsigned *__restrict__ sorted, int records)
{
    constexpr int THREADS = kBinRunThreads;
    extern __shared__ unsigned s_hist[];                 // [NC] local counts; mode 1: then the places reserved
    // (b, s2, group of query views, run): the lists of a (b, s2) are filled by the workgroups of one XCD or two, whose L2 joins
    // their stores. Sample ids (s1*L + l)*P + p of a group are consecutive.
    const unsigned work = (unsigned)xcd_logical_block(blockIdx.x, gridDim.x), ngrp = (unsigned)(NK / NC);
    const unsigned t = work / (unsigned)nlc, lc = work - t * (unsigned)nlc;
    const unsigned grp = t / ngrp, qg = t - grp * ngrp, b = grp / (unsigned)dm.V, s2 = grp - b * (unsigned)dm.V;
    const unsigned n = (unsigned)dm.L * (unsigned)dm.P, end = min((qg + 1u) * (unsigned)vpg, (unsigned)dm.V) * n;
    const unsigned first = qg * (unsigned)vpg * n + lc * (unsigned)(THREADS * PER) + threadIdx.x;
    const float2 *crd = reinterpret_cast<const float2 *>(coords_) + (size_t)b * dm.V * dm.L * dm.N + (size_t)s2 * dm.P;
    float2 xy[PER];
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        const unsigned id = min(first + (unsigned)(j * THREADS), end - 1u), ql = dm.divP.div(id);
        xy[j] = crd[(size_t)ql * dm.N + (id - ql * (unsigned)dm.P)];
    }
    for (int i = threadIdx.x; i < NC; i += THREADS) s_hist[i] = 0u;
    __syncthreads();
    unsigned key[PER], rank[PER];                        // key NC: in no list
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        const Taps tp = make_taps(xy[j].x, xy[j].y, dm.Wimg, dm.Himg);
        const bool counted = first + (unsigned)(j * THREADS) < end && taps_any(tp);
        key[j] = counted ? (unsigned)cell_of(tp, dm.Wimg) : (unsigned)NC;
        rank[j] = 0u;
        if (counted) rank[j] = atomicAdd(&s_hist[key[j]], 1u);
    }
    __syncthreads();
    // the keys of this (b, s2) and group, four counters a thread in flight
    unsigned *gctr = counters + (size_t)grp * NK + (size_t)qg * NC;
    for (int i0 = threadIdx.x; i0 < NC; i0 += 4 * THREADS) {
        unsigned c[4], base[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int i = i0 + u * THREADS;
            c[u] = i < NC ? s_hist[i] : 0u;
            base[u] = 0u;
            if (c[u]) {
                if (MODE == 0) atomicAdd(gctr + i, c[u]);
                else base[u] = atomicAdd(gctr + i, c[u]);
            }
        }
        if (MODE == 1) {
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (c[u]) s_hist[i0 + u * THREADS] = base[u];
        }
    }
    if (MODE == 1) {
        __syncthreads();
        const size_t place0 = (size_t)grp * ((size_t)dm.V * n);
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            if (key[j] == (unsigned)NC) continue;
            store_cell_entry(sorted, place0 + s_hist[key[j]] + rank[j], first + (unsigned)(j * THREADS),
                             cell_fraction(xy[j], dm), records);
        }
    }
}

// One workgroup per (b, s2): exclusive scan of the list lengths (NC here = the number of keys, group-major). Writes
// start[grp*(NC+1) + c] (with the total at c = NC) and resets counters to the
// same starts, so that the fill pass can use them as cursors.
//
// It also makes the dk/dv kernel's work list of this (b, s2): one item (cell, first entry, end) per run of at
// most `piece` consecutive entries of a non-empty list, in list order -- items[grp*wmax + i]; the slots after
// the last item are marked empty (first = end). Empty lists get no item (clustered coordinates leave most
// of the grid empty), and a list much longer than the average is cut into pieces that different waves take,
// so that the longest list no longer sets the kernel's duration. wmax >= NC + M/piece bounds the number of
// items (M = entries of all lists). An item carries all a wave needs to start on it: one read, where the
// list's bounds would be a second, dependent one.
//
// Bound by its chain of waits (one workgroup per (b, s2), a few of them on the whole chip): four keys a thread, both
// sums by lane shifts inside a wave and over the waves' totals in LDS, two barriers per THREADS * 4 keys.
// (8450 keys, 8 workgroups: 29.4 -> 15.2 us against a scan of 1024 keys at a time with 20 barriers; 2401 keys 10.4 -> 6.0.)
constexpr int kScanKeys = 4;
struct ScanCarry { unsigned entries, pieces; };
// One turn of the scan for a workgroup of THREADS threads: keys [c0, c0 + 4) of each thread, v their list lengths;
// returns the first key's start in `first`, writes start and items, advances the carry. s_wave: a place per wave.
template <int THREADS>
__device__ __forceinline__ void scan_keys(const unsigned (&v)[kScanKeys], int c0, int NC, int grid_cells, unsigned piece,
                                          unsigned wmax, unsigned *__restrict__ st, uint4 *__restrict__ it,
                                          uint2 *s_wave, ScanCarry &carry, unsigned &first)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    unsigned np[kScanKeys], sum = 0, psum = 0;
#pragma unroll
    for (int i = 0; i < kScanKeys; ++i) {
        np[i] = (v[i] + piece - 1) / piece;                        // pieces of this list
        sum += v[i];
        psum += np[i];
    }
    unsigned incl = sum, pincl = psum;                             // inclusive scans over the wave
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
        const unsigned add = (unsigned)__shfl_up((int)incl, off, kWave), padd = (unsigned)__shfl_up((int)pincl, off, kWave);
        incl += lane >= off ? add : 0u;
        pincl += lane >= off ? padd : 0u;
    }
    __syncthreads();                                               // (the totals of the keys before have been read)
    if (lane == kWave - 1) s_wave[wave] = make_uint2(incl, pincl);
    __syncthreads();
    unsigned excl = carry.entries + incl - sum, pexcl = carry.pieces + pincl - psum;
#pragma unroll 4                                                      // (unrolled whole: 100 bytes of scratch a lane at 64 registers)
    for (int w = 0; w < THREADS / kWave; ++w) {
        const uint2 t = s_wave[w];
        excl += w < wave ? t.x : 0u;
        pexcl += w < wave ? t.y : 0u;
        carry.entries += t.x;
        carry.pieces += t.y;
    }
    asm volatile("" : "+v"(excl), "+v"(pexcl));                    // (summed here, not from two dozen parts behind each branch below)
    first = excl;
#pragma unroll
    for (int i = 0; i < kScanKeys; ++i) {
        if (c0 + i < NC) {
            st[c0 + i] = excl;
            const unsigned cell = (unsigned)((c0 + i) % grid_cells);
            for (unsigned j = 0; j < np[i]; ++j)
                if (pexcl + j < wmax)
                    it[pexcl + j] = make_uint4(cell, excl + j * piece, min(excl + v[i], excl + (j + 1) * piece), 0u);
        }
        excl += v[i];
        pexcl += np[i];
    }
}

// after the last turn: the total, the empty slots behind the items, and (where `spread` is asked for) the number of items, with
// kSpreadLong set unless the lists are the patch kernel's: `mean` or fewer entries a non-empty list and at most kSpreadLongest
// in the longest, or where the lists are fewer than `few`, `mean` in the longest
struct Spread { unsigned *items, mean, few; };
constexpr unsigned kSpreadLongest = 1024, kSpreadLong = 0x80000000u;
// Whether more than a third of the n groups (b, s2) have long lists: then all are the cell kernel's. (Half the views by
// patches and half by cells fill the chip twice by half: 40x28, batch 2, 4 views x 8 heads, P = 1, clustered, D = 128, bf16, all by cells
// 133 us a step, by patches 175, so mixed 185; 18x18, 6 x 16, P = 6 around the query's place, D = 32 183 / 192 / 206.)
__device__ __forceinline__ bool mostly_long(const unsigned *__restrict__ left, int n)
{
    const int lane = threadIdx.x & 63;
    int longs = 0;
    for (int i = 0; i < n; i += kWave) longs += __popcll(__ballot(i + lane < n && (left[min(i + lane, n - 1)] & kSpreadLong) != 0u));
    return 3 * longs > n;
}
// items that the cell kernel has to do in the planes of a group with left[] = l, 0 if they are the patch kernel's
__device__ __forceinline__ unsigned items_left(unsigned l, bool all) { return all || (l & kSpreadLong) ? l & ~kSpreadLong : 0u; }
template <int THREADS>
__device__ __forceinline__ void scan_end(const ScanCarry &carry, int NC, unsigned wmax, unsigned *__restrict__ st, uint4 *__restrict__ it,
                                         const Spread &spread, unsigned grp, unsigned longest)
{
    if (spread.items) {
        const int any_long = __syncthreads_or(longest > (carry.pieces < spread.few ? spread.mean : kSpreadLongest));
        if (threadIdx.x == 0) {
            const bool is_long = any_long || (unsigned long long)carry.entries > (unsigned long long)spread.mean * carry.pieces;
            spread.items[grp] = min(carry.pieces, wmax) | (is_long ? kSpreadLong : 0u);
        }
    }
    if (threadIdx.x == 0) st[NC] = carry.entries;
    for (unsigned i = min(carry.pieces, wmax) + threadIdx.x; i < wmax; i += THREADS) it[i] = make_uint4(0u, 0u, 0u, 0u);
}

// (512 threads and at most 64 registers beside the staged dq kernel, as above)
template <int THREADS>
__global__ __launch_bounds__(THREADS, THREADS == 512 ? 8 : 4) void bin_scan_kernel(
    unsigned *__restrict__ counters, unsigned *__restrict__ start, int NC, int grid_cells,
    unsigned piece, unsigned wmax, uint4 *__restrict__ items, Spread spread)
{
    __shared__ uint2 s_wave[THREADS / kWave];                      // (entries, pieces) of each wave's keys
    unsigned *cnt = counters + (size_t)blockIdx.x * NC;
    unsigned *st = start + (size_t)blockIdx.x * (NC + 1);
    uint4 *it = items + (size_t)blockIdx.x * wmax;
    ScanCarry carry{0u, 0u};
    unsigned longest = 0u;
    for (int base = 0; base < NC; base += THREADS * kScanKeys) {
        const int c0 = base + (int)threadIdx.x * kScanKeys;
        unsigned v[kScanKeys], at;
#pragma unroll
        for (int i = 0; i < kScanKeys; ++i) v[i] = c0 + i < NC ? cnt[c0 + i] : 0u;
#pragma unroll
        for (int i = 0; i < kScanKeys; ++i) longest = max(longest, v[i]);
        scan_keys<THREADS>(v, c0, NC, grid_cells, piece, wmax, st, it, s_wave, carry, at);
#pragma unroll
        for (int i = 0; i < kScanKeys; ++i) {
            if (c0 + i < NC) cnt[c0 + i] = at;
            at += v[i];
        }
    }
    scan_end<THREADS>(carry, NC, wmax, st, it, spread, blockIdx.x, longest);
}

// Count, scan and fill by one workgroup, for lists short enough that one workgroup holds all samples of a (b, s2) in
// its registers, kBinOneSamples / THREADS of them a thread: every sample's rank in its list comes from the counting atomic itself, so
// there is one round of LDS atomics, no counters in memory (nothing to clear) and no wait between launches; 1024 threads read the coordinates
// once, 256 (in the row dq launch, whose registers do not hold them and the scan) again for the fill. Bound by that chain of latencies (a few workgroups on the whole chip), as the three
// launches are: 1296 samples a list group (18x18, 2 views x 2 samples) 6.2 us against 13.7 for the three and the gaps
// between them. One workgroup's throughput then takes over: 5184 (4 x 4, six samples a thread) 13.9 against 17.4, a step
// no faster; 11664 34.8 against 24.1, 17871 59 against 19.
// Keys: one per cell, (Himg + 1)(Wimg + 1) <= 2 Himg Wimg + 2 of them, in LDS; the query views are one group (their rows
// take at most 2 * 2048 * 256 * 4 bytes, below where views_per_group splits them).
constexpr int kBinOneKeys = 2 * kBinOneSamples + 2, kBinOneKeyBits = 13;
static_assert(kBinOneKeys < (1 << kBinOneKeyBits), "a key fits below its rank");
static_assert(2ull * kBinOneSamples * 256 * 4 <= kGroupRowsBytes, "one group of query views");
// What it makes of coords: lists (starts, entries, as ids or `records`), work list, and the counts for the patch kernel (see above).
// `groups` of them; 0: nothing to do.
struct BinJob { unsigned groups; int NC; unsigned piece, wmax; unsigned *start; uint4 *items; unsigned *sorted; int records; Spread spread; };
// One (b, s2) = grp, by a workgroup of THREADS threads. s_hist: NC words of LDS.
template <int THREADS>
__device__ __forceinline__ void bin_one_group(const float *__restrict__ coords_, const Dims &dm, const BinJob &bj, unsigned grp, unsigned *s_hist)
{
    constexpr int PER = kBinOneSamples / THREADS;
    __shared__ uint2 s_wave[THREADS / kWave];
    const int NC = bj.NC;
    const unsigned s2 = grp % (unsigned)dm.V, b = grp / (unsigned)dm.V;
    const unsigned M = (unsigned)dm.V * (unsigned)dm.L * (unsigned)dm.P;
    const float2 *crd = reinterpret_cast<const float2 *>(coords_) + ((size_t)b * dm.V * dm.L * dm.V + s2) * (size_t)dm.P;
    unsigned tid = threadIdx.x;
    auto fetch = [&](int i) {
        const unsigned id = min((unsigned)(i * THREADS) + tid, M - 1u);                // id = ql * P + p
        const unsigned ql = dm.divP.div(id), p = id - ql * (unsigned)dm.P;
        return crd[(size_t)ql * dm.N + p];
    };
    float2 xy[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) xy[i] = fetch(i);
    for (int i = threadIdx.x; i < NC; i += THREADS) s_hist[i] = 0u;
    __syncthreads();
    unsigned key_rank[PER];                                        // key, rank above; all ones: in no list
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const unsigned id = (unsigned)(i * THREADS) + threadIdx.x;
        const Taps tp = make_taps(xy[i].x, xy[i].y, dm.Wimg, dm.Himg);
        key_rank[i] = 0xffffffffu;
        if (id < M && taps_any(tp)) {
            const unsigned key = (unsigned)cell_of(tp, dm.Wimg);
            key_rank[i] = key | (atomicAdd(&s_hist[key], 1u) << kBinOneKeyBits);
        }
        if (PER > 2) __builtin_amdgcn_sched_barrier(0);            // (one after the other: registers)
    }
    __syncthreads();
    ScanCarry carry{0u, 0u};
    unsigned longest = 0u;
    unsigned *st = bj.start + (size_t)grp * (NC + 1);
    uint4 *it = bj.items + (size_t)grp * bj.wmax;
    for (int base = 0; base < NC; base += THREADS * kScanKeys) {
        const int c0 = base + (int)threadIdx.x * kScanKeys;
        unsigned v[kScanKeys], at;
#pragma unroll
        for (int i = 0; i < kScanKeys; ++i) v[i] = c0 + i < NC ? s_hist[c0 + i] : 0u;
#pragma unroll
        for (int i = 0; i < kScanKeys; ++i) longest = max(longest, v[i]);
        scan_keys<THREADS>(v, c0, NC, NC, bj.piece, bj.wmax, st, it, s_wave, carry, at);
#pragma unroll
        for (int i = 0; i < kScanKeys; ++i) {
            if (c0 + i < NC) s_hist[c0 + i] = at;                  // (this thread's own keys)
            at += v[i];
        }
    }
    __syncthreads();
    if constexpr (PER > 2) asm volatile("" : "+v"(tid)::"memory");       // (coordinates and ids made anew: not held through the scan)
    constexpr int AT_ONCE = PER > 2 ? PER / 2 : PER;
#pragma unroll
    for (int i0 = 0; i0 < PER; i0 += AT_ONCE) {
#pragma unroll
        for (int i = i0; PER > 2 && i < i0 + AT_ONCE; ++i) xy[i] = fetch(i);
#pragma unroll
        for (int i = i0; i < i0 + AT_ONCE; ++i) {
            if (key_rank[i] != 0xffffffffu)
                store_cell_entry(bj.sorted, (size_t)grp * M + s_hist[key_rank[i] & ((1u << kBinOneKeyBits) - 1u)] + (key_rank[i] >> kBinOneKeyBits),
                                 (unsigned)(i * THREADS) + tid, cell_fraction(xy[i], dm), bj.records);
        }
        if (PER > 2) __builtin_amdgcn_sched_barrier(0);
    }
    scan_end<THREADS>(carry, NC, bj.wmax, st, it, bj.spread, grp, longest);
}

// In a launch of its own: before the dq kernels that take no BinJob (the row kernel does), and before the sort of the deterministic backward.
static __global__ __launch_bounds__(1024) void bin_one_kernel(const float *__restrict__ coords_, Dims dm, BinJob bj)
{
    __shared__ unsigned s_hist[kBinOneKeys];                       // list lengths, then starts
    bin_one_group<1024>(coords_, dm, bj, blockIdx.x, s_hist);
}

// Deterministic backward: begin / end of every cell list as positions in the flat id array
// [B*V][M] (one thread per (group, cell)), the segment bounds of the sort that orders each list.
static __global__ void cell_segments_kernel(const unsigned *__restrict__ start, int NC, unsigned M, unsigned nseg,
                                            unsigned *__restrict__ seg_begin, unsigned *__restrict__ seg_end)
{
    const unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nseg) return;
    const unsigned grp = i / (unsigned)NC, cell = i - grp * (unsigned)NC;
    const unsigned *st = start + (size_t)grp * (NC + 1) + cell;
    seg_begin[i] = grp * M + st[0];
    seg_end[i] = grp * M + st[1];
}

template <typename S, int DC>
__device__ __forceinline__ void load_tap_or_zero(const char *base, int pix, int D, int lane_elem, bool valid,
                                                 float (&dst)[DC])
{
    if (valid) {
        load_chunk<S, DC>(base + ((size_t)pix * D + lane_elem) * S::kBytes, dst);
    } else {
#pragma unroll
        for (int d = 0; d < DC; ++d) dst[d] = 0.f;
    }
}

// Deterministic backward: the sorted ids as records, so that the dk/dv kernel finds the positions beside them there too (one
// thread per list place; `total` = B*V*M, places beyond a group's lists are skipped).
static __global__ __launch_bounds__(256) void records_kernel(const float *__restrict__ coords_, const unsigned *__restrict__ start,
                                                             const unsigned *__restrict__ ids, unsigned *__restrict__ records,
                                                             int NC, unsigned total, Dims dm)
{
    const unsigned M = (unsigned)dm.V * (unsigned)dm.L * (unsigned)dm.P;
    const unsigned at = blockIdx.x * 256u + threadIdx.x;
    const unsigned grp = at / M, i = at - grp * M;                                   // (b, s2), place
    if (at >= total || i >= start[(size_t)grp * (NC + 1) + NC]) return;
    const unsigned b = grp / (unsigned)dm.V, s2 = grp - b * (unsigned)dm.V;
    const unsigned id = ids[at], ql = dm.divP.div(id), p = id - ql * (unsigned)dm.P;
    const float2 xy = reinterpret_cast<const float2 *>(coords_)[((size_t)b * dm.V * dm.L + ql) * dm.N + s2 * (unsigned)dm.P + p];
    store_cell_entry(records, at, id, cell_fraction(xy, dm), 1);
}

// A lane's part of one query row as it comes from memory: q and dout words (storage type), and the row's
// (lse, delta) pair.
template <int WORDS> struct RowFetch { uint32_t qw[WORDS], dw[WORDS]; float2 ld; };

// Which cells one launch of the dk/dv kernel covers, and the divisors that decode a work index into
// (b, h, s2, cell) with multiply-shift instead of integer division (the decode is scalar code every
// wave runs before it knows whether its cell is empty).
// All cells by the work list that the binning made, work index -> (b, h, s2, item), `ncells` being the
// list's capacity wmax per (b, s2) (empty slots leave at once); per-cell sums are flushed with float
// atomics (a pixel belongs to four cells).
// FIXED (deterministic backward): every cell of the grid, one wave each and no pieces, and the sums are stored: a pixel's
// four contributions come from four cells, as a different one of the four taps of each, so tap t of every cell has a
// buffer of its own, [dk, dv][tap][plane][pixel][D], every place of which one wave writes (zeros from an empty list).
// combine_taps_kernel then adds a pixel's four in a fixed order. (Four launches, each for the cells of one row and column parity
// and with read-add-write into dk and dv, took 222 us at 18x18, 6 views x 32 samples, D = 32, where the one and the sums take 142: a quarter
// of the cells are 8664 waves, a third of what the chip holds, four times.)
struct CellGrid {
    int ncells;
    int bh0;                                // first (batch, head) pair of this launch (b * H + h)
    unsigned t0, nplanes;                   // deterministic: first plane (b, h, s2) of this launch, counted from pair bh0, and planes
    unsigned nwork;                         // planes of this launch * ncells < 2^31
    FastDiv div_cells, div_ncx, div_v, div_h;
};

// HANDED: the dq kernel has left (p, sm_scale * ds) of every sample in `handed_` (per query row of this head,
// in the order of the row's coordinates): an entry then costs a gather of that pair and the two rank-1 updates --
// no taps in registers, no dot products, no exponential.
// The lists hold 12-byte records (sample id and position in the cell).
// FIXED: the deterministic backward's launch (see CellGrid).
// What an item costs beside its entries is about 300 vector instructions (bounds, taps, tables, the sum over the
// slots, the flush), which is most of the kernel where lists are short: 18x18, D = 32, 2 views x 2 samples (3.6
// entries a list, fp32) 43.0 -> 39.8 us, 6 x 6 (32 entries, bf16) 172 -> 161, 14x14 with 8 x 32 (223, fp32) 244.5 -> 241,
// with the slots summed on a quarter of the values where the step that halves them comes first, and no tables made
// for a block that is not there.
template <typename S, int D, int DC, bool HANDED, bool FIXED>
__device__ __forceinline__ void cell_sums(
    unsigned t, int ci, const void *__restrict__ q_, const void *__restrict__ k_, const void *__restrict__ v_,
    const float2 *__restrict__ stats_,
    const void *__restrict__ dout_, const unsigned *__restrict__ start, const unsigned *__restrict__ sorted,
    const uint4 *__restrict__ items, const float2 *__restrict__ handed_,
    float *__restrict__ dk_acc, float *__restrict__ dv_acc, const GradDims &dm, int NC, const CellGrid &cg)
{
    constexpr int G = D / DC;
    constexpr int NS = kWave / G;
    static_assert(G >= 4 && G <= 64 && G * DC == D, "lane split (a block of four lanes must not straddle two samples)");
    __shared__ float4 s_w[kCellWaves][2 * kWave];           // two sets of entry tables, used in turn
    __shared__ unsigned s_row[kCellWaves][2 * kWave];       // byte offset of the entry's query row in dout (and its (lse, delta))
    __shared__ unsigned s_qrow[kCellWaves][2 * kWave];      // ... in q (which may be strided)
    __shared__ float2 s_f[S::kBytes == 2 ? kCellWaves : 1][2 * kWave];      // 16-bit storage: (fx, fy) of the entry
    __shared__ __attribute__((aligned(16))) float s_flush[kCellWaves][4 * D];                 // the flush: four rows of dk, then of dv
    // four-entry trips (below), whose coefficients are two 16-bit parts; the deterministic backward keeps fp32 ones
    constexpr bool kQuad = HANDED && !FIXED && S::kBytes == 2 && DC >= 8;
    // kQuad: a ring of merged entries; the coefficients as [tap][place]
    __shared__ __attribute__((aligned(16))) float s_ckq[kQuad ? kCellWaves : 1][2 * 4 * kWave], s_cvq[kQuad ? kCellWaves : 1][2 * 4 * kWave];
    __shared__ __attribute__((aligned(16))) unsigned s_rowq[kQuad ? kCellWaves : 1][2 * kWave], s_qrowq[kQuad ? kCellWaves : 1][2 * kWave];

    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;   // wave index is uniform: keep it in an SGPR
    // t = plane (b, h, s2) of the launch, ci = its cell or work item
    const unsigned bhl = cg.div_v.div(t);                      // pair within this launch
    const int s2 = (int)(t - bhl * (unsigned)dm.V);
    const unsigned bh = (unsigned)cg.bh0 + bhl;
    const int b = (int)cg.div_h.div(bh);
    const int h = (int)(bh - (unsigned)b * (unsigned)dm.H);
    const size_t grp = (size_t)b * dm.V + s2;
    int cy, cx, cell;
    unsigned lo, hi;
    if constexpr (!FIXED) {
        const uint4 item = items[grp * (size_t)cg.ncells + ci];              // (cell, first entry, end)
        cell = (int)item.x;
        cy = (int)cg.div_ncx.div(item.x);                      // div_ncx: by Wimg + 1 in this mode
        cx = cell - cy * (dm.Wimg + 1);
        lo = item.y;
        hi = item.z;
    } else {
        cell = ci;
        cy = (int)cg.div_ncx.div((unsigned)ci);
        cx = ci - cy * (dm.Wimg + 1);                          // on the (Himg+1) x (Wimg+1) grid
        lo = start[grp * (NC + 1) + cell];
        hi = start[grp * (NC + 1) + cell + 1];
    }
    if (!FIXED && lo >= hi) return;

    const int g = lane % G, slot = lane / G, lane_elem = g * DC;
    const int y0 = cy - 1, x0 = cx - 1;
    const bool vy0 = y0 >= 0, vy1 = y0 + 1 < dm.Himg, vx0 = x0 >= 0, vx1 = x0 + 1 < dm.Wimg;
    const bool tv[4] = { vy0 && vx0, vy0 && vx1, vy1 && vx0, vy1 && vx1 };
    // where tap r of this cell goes (deterministic backward), `which` 0: dk, 1: dv; its pixel has to be inside the image
    auto tap_place = [&](int which, int r, int pix) -> float * {
        return (which == 0 ? dk_acc : dv_acc) + (((size_t)r * cg.nplanes + (t - cg.t0)) * dm.L + pix) * (size_t)D;
    };
    if constexpr (FIXED) {
        if (lo >= hi) {
            for (int idx = lane; idx < 8 * D; idx += kWave) {
                const int r = (idx / D) & 3;
                if (((r & 2) ? vy1 : vy0) && ((r & 1) ? vx1 : vx0))
                    tap_place(idx / (4 * D), r, (y0 + (r >> 1)) * dm.Wimg + x0 + (r & 1))[idx & (D - 1)] = 0.f;
            }
            return;
        }
    }
    const int tpix[4] = { y0 * dm.Wimg + x0, y0 * dm.Wimg + x0 + 1, (y0 + 1) * dm.Wimg + x0,
                          (y0 + 1) * dm.Wimg + x0 + 1 };
    const size_t plane_base = dm.acc_plane<S, D>(b, s2, h);                     // elements in dk/dv
    const size_t kv_base = dm.kv_plane(b, s2, h);                               // ... in k and v
    const char *kb = (const char *)k_ + kv_base * S::kBytes;
    const char *vb = (const char *)v_ + kv_base * S::kBytes;
    // fp32 storage: the taps widened in registers; 16-bit storage: the taps as packed pairs (half the
    // registers) feeding the packed dot-product instructions
    constexpr bool kPacked = S::kBytes == 2;
    float kt[4][kPacked ? 1 : DC], vt[4][kPacked ? 1 : DC], aK[4][DC], aV[4][DC];
    uint32_t ktp[4][kPacked ? DC / 2 : 1], vtp[4][kPacked ? DC / 2 : 1];
    // The per-sample rank-1 updates aK[t][d] += c_t * q[d], aV[t][d] += c'_t * dout[d] run on the 4x4 block
    // matrix instruction (see block_outer_fma): mK[d][t] / mV[d][t] are the same sums as aK[t][d] / aV[t][d].
    floatx4 mK[DC], mV[DC];
    // The row of the update that lane (lane & 3) supplies is a product a_x(fx) * a_y(fy) of two linear forms
    // with per-lane constants, so no lane ever selects among the four: packed (the bilinear weight of tap
    // lane & 3): a_x = 1 - fx or fx, a_y = 1 - fy or fy; fp32 (the moment 1, fx, fy, fx*fy): a_x = 1 or fx,
    // a_y = 1 or fy.
    const float row_sx = (lane & 1) ? 1.0f : (kPacked ? -1.0f : 0.0f), row_ox = (lane & 1) ? 0.0f : 1.0f;
    const float row_sy = (lane & 2) ? 1.0f : (kPacked ? -1.0f : 0.0f), row_oy = (lane & 2) ? 0.0f : 1.0f;
#pragma unroll
    for (int tpi = 0; tpi < (HANDED ? 0 : 4); ++tpi) {
        if constexpr (kPacked) {
#pragma unroll
            for (int i = 0; i < DC / 2; ++i) { ktp[tpi][i] = 0u; vtp[tpi][i] = 0u; }
            if (tv[tpi]) {
                load_packed<S, DC>(kb + ((size_t)tpix[tpi] * dm.kv_sl + lane_elem) * S::kBytes, ktp[tpi]);
                load_packed<S, DC>(vb + ((size_t)tpix[tpi] * dm.kv_sl + lane_elem) * S::kBytes, vtp[tpi]);
            }
        } else {
            load_tap_or_zero<S, DC>(kb, tpix[tpi], dm.kv_sl, lane_elem, tv[tpi], kt[tpi]);
            load_tap_or_zero<S, DC>(vb, tpix[tpi], dm.kv_sl, lane_elem, tv[tpi], vt[tpi]);
        }
    }
#pragma unroll
    for (int d = 0; d < DC; ++d) { mK[d] = floatx4{0.f, 0.f, 0.f, 0.f}; mV[d] = floatx4{0.f, 0.f, 0.f, 0.f}; }
    // fp32 storage: the cell's taps are turned, once, into the coefficients of the bilinear form
    //   blend(fx, fy) = T00 + fx*(T01 - T00) + fy*(T10 - T00) + fx*fy*(T00 - T01 - T10 + T11)
    // so that a sample's blend costs 3 multiply-adds per element instead of 4, and the sums are kept as the
    // matching moments (sum c, sum c*fx, sum c*fy, sum c*fx*fy times the query row), turned back into the
    // four pixels' sums after the loop. (Taps outside the image were loaded as zero rows.)
    if constexpr (!kPacked && !HANDED) {
#pragma unroll
        for (int d = 0; d < DC; ++d) {
            kt[3][d] = (kt[3][d] - kt[2][d]) - (kt[1][d] - kt[0][d]);
            kt[1][d] -= kt[0][d];
            kt[2][d] -= kt[0][d];
            vt[3][d] = (vt[3][d] - vt[2][d]) - (vt[1][d] - vt[0][d]);
            vt[1][d] -= vt[0][d];
            vt[2][d] -= vt[0][d];
        }
    }
    const float qscale = dm.sm_scale * kLog2e;
    const size_t M = (size_t)dm.V * dm.L * dm.P;
    const unsigned *list = sorted + grp * M * 3u;                       // records (id, fx, fy)
    // Query rows of this wave's (b, h) are addressed as a uniform base plus a 32-bit byte offset
    // (s1*H*L + l) * ROW < V*H*L*D*e <= 2^32 (the shape limits keep one batch item of a tensor below 2^30
    // elements): one add per gather instead of 64-bit address arithmetic per lane.
    constexpr unsigned kRowBytes = D * S::kBytes;
    constexpr int kRowWords = DC * S::kBytes / 4;                           // 32-bit words of a row held by one lane
    constexpr int kRowToPairShift = __builtin_ctz(kRowBytes) - 3;          // row byte offset -> offset of the row's (lse, delta)
    const size_t bh_row0 = ((size_t)b * dm.V * dm.H + h) * dm.L;              // row of (b, s1 = 0, h, l = 0)
    const char *q_bh = (const char *)q_ + dm.q_row(b, 0, h, 0) * S::kBytes;
    const char *do_bh = (const char *)dout_ + bh_row0 * kRowBytes;
    const char *stats_bh = (const char *)(stats_ + bh_row0);                 // (lse, delta) per row
    const unsigned lane_byte = (unsigned)lane_elem * S::kBytes;
    const unsigned view_rows = (unsigned)dm.H * (unsigned)dm.L;

    // HANDED: the entry's pair, gathered one chunk ahead (so the ids are fetched two chunks ahead). The pairs of
    // this launch's (batch, head) pairs lie as [pair][s1][l][sample]; those of this wave's pair are a uniform base
    // plus a 32-bit byte offset (the host checks V*L*N*8 < 2^32).
    const char *handed_bh = (const char *)(handed_ + (size_t)bhl * dm.V * dm.L * (size_t)dm.N);
    auto load_pair = [&](unsigned sid) -> float2 {
        const unsigned qlx = dm.divP.div(sid), px = sid - qlx * (unsigned)dm.P;       // qlx = s1*L + l
        const unsigned off = (qlx * (unsigned)dm.N + (unsigned)s2 * (unsigned)dm.P + px) * 8u;
        return *reinterpret_cast<const float2 *>(handed_bh + off);
    };
    if constexpr (kQuad) {
        // 16-bit storage with the pairs handed over, eight elements per lane (at four the trips are too short for
        // the requests to arrive in time: 1.14 -> 1.22 ms at 48x48, D = 64): FOUR entries per slot and trip on the
        // 4x4x4 block matrix instruction. k runs over the four entries, i over the four taps (lane 4b+i supplies
        // the four entries' coefficients of tap i, high and low parts in two instructions), j over the block's
        // lanes with their elements of the four query rows -- as stored, regrouped by two byte permutes per pair
        // of rows. 4 * DC instructions do what 4 * 2 * DC rank-1 updates and as many bf16 -> fp32 conversions did.
        //
        // Entries of ONE query in one cell are merged before their rows are requested: a query's samples cluster,
        // the fill pass of the binning leaves the samples that one wave places in one list next to each other (the
        // ranks that one returning LDS atomic hands out), and the sums are linear in the coefficients -- so a run
        // of up to four neighbouring entries with the same query row becomes one entry with the summed tap
        // coefficients: one gather of q and dout and one set of matrix instructions instead of up to four.
        //
        // The merged entries of the list's 64-entry blocks are appended to a ring of kRing places in LDS (tables
        // [tap][place] of coefficients and [place] of row offsets); trips of QT merged entries are taken off its
        // head. Everything is requested ahead: the q and dout rows of the next trip while this trip is worked on
        // (one set of registers each), which needs the next trip's places filled -- so blocks are merged two ahead
        // of the trips, and trips run while two whole trips are in the ring (all of them once the last block is in;
        // the places after the last entry then hold zero coefficients and the row of a live entry).
        constexpr int QT = 4 * NS, kRing = 2 * kWave;
        static_assert(QT % 4 == 0 && kRing % QT == 0 && kRing >= 2 * kWave && kRing >= kWave + 3 * QT,
                      "two blocks fit before the first trip; places written by one block never reach the trips in flight");
        // (requests past the end of the list repeat its last entry: no request sits under a branch, and the number
        // of requests in flight at any point is the same on every path -- the compiler's waits are exact then)
        auto load_entry_q = [&](unsigned cstart) -> CellEntry {
            const unsigned *r = list + 3u * min(cstart + (unsigned)lane, hi - 1u);
            return CellEntry{r[0], __uint_as_float(r[1]), __uint_as_float(r[2])};
        };
        // fp16: what the coefficients of ds are multiplied by at the split (lower_scale). The ring holds them as they are, so
        // that a scale lowered for a new block holds for what is left of the old ones too; the sums are brought down to it.
        constexpr bool kScaled = !S::kBf16;
        float scale_ds = kScaled ? kScaleDs : 1.0f;
        auto prepare = [&](unsigned cstart, int tail, unsigned sid, float2 ff, float2 pdv) -> int {
            const unsigned ql = dm.divP.div(sid);                                  // ql = s1*L + l
            const unsigned s1 = dm.divL.div(ql), l = ql - s1 * (unsigned)dm.L;
            const bool live = cstart + (unsigned)lane < hi;                        // a dead entry adds nothing
            const unsigned before = (unsigned)__shfl_up((int)ql, 1, kWave);
            const unsigned long long below = (1ull << lane) - 1ull;                // the lanes under this one
            const unsigned long long first = __ballot(lane == 0 || ql != before);  // first entries of the runs of one row
            const int run0 = 63 - __builtin_clzll(first & (below | (1ull << lane)));
            const bool lead = live && ((lane - run0) & 3) == 0;                    // runs are cut into merged entries of up to four
            const unsigned long long leads = __ballot(lead);
            const int idx = __builtin_popcountll(leads & below);                   // a leader's place after the tail
            const int n = __builtin_popcountll(leads);
            // the entries after this one that belong to the same merged entry: the lanes up to the next leader
            const bool f1 = lane < 63 && !((leads >> (lane + 1)) & 1ull);
            const bool f2 = f1 && lane < 62 && !((leads >> (lane + 2)) & 1ull);
            const float m1 = f1 ? 1.0f : 0.0f, m2 = f2 ? 1.0f : 0.0f;
            const float pn = live ? pdv.x : 0.f, dsn = live ? pdv.y : 0.f;
            const float gx = 1.0f - ff.x, gy = 1.0f - ff.y;
            const float wt[4] = { gx * gy, ff.x * gy, gx * ff.y, ff.x * ff.y };
            float c[8];
#pragma unroll
            for (int tpi = 0; tpi < 4; ++tpi) { c[tpi] = wt[tpi] * dsn; c[4 + tpi] = wt[tpi] * pn; }
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float pairsum = fmaf(m1, __shfl_down(c[i], 1, kWave), c[i]);
                c[i] = fmaf(m2, __shfl_down(pairsum, 2, kWave), pairsum);
            }
            float top = 0.f;
            if constexpr (kScaled) top = lead ? fmaxf(fmaxf(fabsf(c[0]), fabsf(c[1])), fmaxf(fabsf(c[2]), fabsf(c[3]))) : 0.f;
            const unsigned row = (s1 * view_rows + l) * kRowBytes;
            const unsigned qrow = (s1 * (unsigned)dm.q_sv + l * (unsigned)dm.q_sl) * S::kBytes;
            float *ck = s_ckq[wave], *cv = s_cvq[wave];
            if (lead) {
                const int at = (tail + idx) & (kRing - 1);
#pragma unroll
                for (int tpi = 0; tpi < 4; ++tpi) { ck[tpi * kRing + at] = c[tpi]; cv[tpi * kRing + at] = c[4 + tpi]; }
                s_rowq[wave][at] = row;
                s_qrowq[wave][at] = qrow;
            }
            // the places up to the end of a last, partial trip: no coefficients, and a row that is in this list
            // (no further: the two blocks merged before the first trip may fill the ring to its last place)
            if (tail + n + lane < ((tail + n + QT - 1) & ~(QT - 1))) {
                const int at = (tail + n + lane) & (kRing - 1);
#pragma unroll
                for (int tpi = 0; tpi < 4; ++tpi) { ck[tpi * kRing + at] = 0.f; cv[tpi * kRing + at] = 0.f; }
                s_rowq[wave][at] = (unsigned)__builtin_amdgcn_readfirstlane((int)row);
                s_qrowq[wave][at] = (unsigned)__builtin_amdgcn_readfirstlane((int)qrow);
            }
            if constexpr (kScaled) {
                const float by = lower_scale(first_lane(wave_max(top)), scale_ds);
                if (by != 1.0f) {
#pragma unroll
                    for (int d = 0; d < DC; ++d) mK[d] *= by;
                }
            }
            return n;
        };
        uint32_t rq[4][kRowWords], rd[4][kRowWords];
        auto issue_q = [&](int at0) {
            const uint4 r = reinterpret_cast<const uint4 *>(s_qrowq[wave])[((at0 >> 2) + slot) & (kRing / 4 - 1)];
            load_words<kRowWords>(q_bh + (r.x + lane_byte), rq[0]);
            load_words<kRowWords>(q_bh + (r.y + lane_byte), rq[1]);
            load_words<kRowWords>(q_bh + (r.z + lane_byte), rq[2]);
            load_words<kRowWords>(q_bh + (r.w + lane_byte), rq[3]);
        };
        auto issue_d = [&](int at0) {
            const uint4 r = reinterpret_cast<const uint4 *>(s_rowq[wave])[((at0 >> 2) + slot) & (kRing / 4 - 1)];
            load_words<kRowWords>(do_bh + (r.x + lane_byte), rd[0]);
            load_words<kRowWords>(do_bh + (r.y + lane_byte), rd[1]);
            load_words<kRowWords>(do_bh + (r.z + lane_byte), rd[2]);
            load_words<kRowWords>(do_bh + (r.w + lane_byte), rd[3]);
        };
        // (places that were never written are read for requests that nothing uses: any row of the pair will do)
        s_rowq[wave][lane] = 0u;
        s_rowq[wave][kWave + lane] = 0u;
        s_qrowq[wave][lane] = 0u;
        s_qrowq[wave][kWave + lane] = 0u;
        int head = 0, tail;
        CellEntry e_a;
        {
            const CellEntry e0 = load_entry_q(lo), e1 = load_entry_q(lo + kWave);
            e_a = load_entry_q(lo + 2 * kWave);
            const float2 pd0 = load_pair(e0.id), pd1 = load_pair(e1.id);
            tail = prepare(lo, 0, e0.id, make_float2(e0.fx, e0.fy), pd0);
            if (lo + kWave < hi) tail += prepare(lo + kWave, tail, e1.id, make_float2(e1.fx, e1.fy), pd1);
        }
        wave_lds_sync();
        issue_q(0);
        issue_d(0);
        const int tap_lane = (lane & 3) * (kRing / 4) + slot;                       // this lane's tap, its slot's four entries (in float4 units)
        for (unsigned cnext = lo + 2 * kWave;; cnext += kWave) {
            const bool more = cnext < hi;                      // a block is left to merge
            const float2 pd_a = load_pair(e_a.id);
            const CellEntry e_n = load_entry_q(cnext + kWave);
            __builtin_amdgcn_sched_barrier(0);                 // (requested here, not where they are used)
            // (at least one trip: a whole block adds QT merged entries or more to the QT or more that the trips before left)
            const int stop = more ? tail - 2 * QT : tail - 1;
            do {
                const int at = (head & (kRing - 1)) >> 2;
                const float4 ck4 = reinterpret_cast<const float4 *>(s_ckq[wave])[tap_lane + at];
                const float4 cv4 = reinterpret_cast<const float4 *>(s_cvq[wave])[tap_lane + at];
                const float by_p = kScaled ? kScaleP : 1.0f;
                const uint4 sk = split_coefficients<S>(ck4.x * scale_ds, ck4.y * scale_ds, ck4.z * scale_ds, ck4.w * scale_ds);
                const uint4 sv = split_coefficients<S>(cv4.x * by_p, cv4.y * by_p, cv4.z * by_p, cv4.w * by_p);
                __builtin_amdgcn_sched_barrier(0);
                block_blend4_pair<S, DC>(rq, __builtin_bit_cast(shortx4, make_uint2(sk.x, sk.y)),
                                         __builtin_bit_cast(shortx4, make_uint2(sk.z, sk.w)), mK);
                __builtin_amdgcn_sched_barrier(0);
                issue_q(head + QT);
                __builtin_amdgcn_sched_barrier(0);
                block_blend4_pair<S, DC>(rd, __builtin_bit_cast(shortx4, make_uint2(sv.x, sv.y)),
                                         __builtin_bit_cast(shortx4, make_uint2(sv.z, sv.w)), mV);
                __builtin_amdgcn_sched_barrier(0);
                issue_d(head + QT);
                __builtin_amdgcn_sched_barrier(0);
                head += QT;
            } while (head <= stop);
            if (!more) break;
            wave_lds_sync();
            tail += prepare(cnext, tail, e_a.id, make_float2(e_a.fx, e_a.fy), pd_a);
            wave_lds_sync();
            e_a = e_n;
        }
        if constexpr (kScaled) {
            const float un = 1.0f / scale_ds;
#pragma unroll
            for (int d = 0; d < DC; ++d) { mK[d] *= un; mV[d] *= 1.0f / kScaleP; }
        }
    }
    if constexpr (!kQuad) {
        // One list entry per lane and 64-entry block: weights and query row go into tables in LDS, which the slots
        // walk NS entries a trip. Two sets of tables, used in turn: the next block's are made while this block is
        // worked on, so that the last trip of a block can request the rows of the next block's first. The NS
        // samples of a trip need their query rows (q, dout, lse, delta) from memory, a round trip of several
        // hundred nanoseconds that the other waves of the SIMD do not cover: the rows of trip t+1 are requested
        // before trip t is worked on (two sets of row registers, the loop unrolled by two so that no set is ever
        // copied). Every request is unconditional -- entries past the end of the list repeat its last one, with
        // zero weights, and the last request of a list is never used -- and the trip loop runs at least once: the
        // number of requests in flight is the same on every path, so the compiler's waits name exactly the
        // younger requests instead of "everything" (a request under a branch, or a loop that may run zero times,
        // makes the wait at the join a wait for all outstanding loads, which undoes the overlap).
        auto load_entry_c = [&](unsigned cstart) -> CellEntry {
            const unsigned *r = list + 3u * min(cstart + (unsigned)lane, hi - 1u);
            return CellEntry{r[0], __uint_as_float(r[1]), __uint_as_float(r[2])};
        };
        auto tables = [&](unsigned cstart, int buf, const CellEntry &e, const float2 &pdv) {
            const unsigned ql = dm.divP.div(e.id);                     // ql = s1*L + l
            const unsigned s1 = dm.divL.div(ql), l = ql - s1 * (unsigned)dm.L;
            // Plain bilinear weights, not masked: every sample of this list lies in this cell, whose taps
            // outside the image were loaded as zeros above and are skipped by the flush below.
            const float fx = e.fx, fy = e.fy;
            const float gx = 1.0f - fx, gy = 1.0f - fy;
            const bool live = cstart + (unsigned)lane < hi;           // a dead entry adds nothing
            const int at = buf * kWave + lane;
            if constexpr (HANDED) {
                s_w[wave][at] = make_float4(fx, fy, live ? pdv.x : 0.f, live ? pdv.y : 0.f);     // (fx, fy, p, sm_scale * ds)
            } else if constexpr (kPacked) {
                s_w[wave][at] = live ? make_float4(gx * gy, fx * gy, gx * fy, fx * fy) : make_float4(0.f, 0.f, 0.f, 0.f);
                s_f[wave][at] = make_float2(fx, live ? fy : __int_as_float(0x7fc00000));          // NaN marks a dead entry
            } else {
                s_w[wave][at] = make_float4(fx, fy, fx * fy, live ? 1.0f : 0.0f);
            }
            s_row[wave][at] = (s1 * view_rows + l) * kRowBytes;
            s_qrow[wave][at] = (s1 * (unsigned)dm.q_sv + l * (unsigned)dm.q_sl) * S::kBytes;
        };
        auto issue = [&](int buf, int j0, RowFetch<kRowWords> &f) {
            const unsigned r = s_row[wave][buf * kWave + j0 + slot];
            const unsigned roff = r + lane_byte, soff = r >> kRowToPairShift;
            load_words<kRowWords>(q_bh + (s_qrow[wave][buf * kWave + j0 + slot] + lane_byte), f.qw);
            load_words<kRowWords>(do_bh + roff, f.dw);
            if constexpr (!HANDED) f.ld = *(const float2 *)(stats_bh + soff);
        };
        auto consume = [&](int buf, int j0, const RowFetch<kRowWords> &f) {
            float qf[DC], dof[DC];
            widen_words<S, DC>(f.qw, qf);
            widen_words<S, DC>(f.dw, dof);
            if constexpr (HANDED) {
                const float4 w4 = s_w[wave][buf * kWave + j0 + slot];                 // (fx, fy, p, sm_scale * ds)
                const float cl = fmaf(w4.x, row_sx, row_ox) * fmaf(w4.y, row_sy, row_oy);
                const float ck = cl * w4.w, cv = cl * w4.z;
#pragma unroll
                for (int d = 0; d < DC; ++d) {
                    mK[d] = block_outer_fma(ck, qf[d], mK[d]);
                    mV[d] = block_outer_fma(cv, dof[d], mV[d]);
                }
            } else {
            const float4 w = s_w[wave][buf * kWave + j0 + slot];
            const float lse = f.ld.x, delta = f.ld.y;
            float dot = 0.f, dp = 0.f;
            if constexpr (kPacked) {
                // q . k~ = sum_t w_t (q . K_t): packed dot products on the raw 16-bit pairs
                dot = fmaf(w.x, packed_dot<S, DC>(f.qw, ktp[0]),
                           fmaf(w.y, packed_dot<S, DC>(f.qw, ktp[1]),
                                fmaf(w.z, packed_dot<S, DC>(f.qw, ktp[2]), w.w * packed_dot<S, DC>(f.qw, ktp[3]))));
                dp = fmaf(w.x, packed_dot<S, DC>(f.dw, vtp[0]),
                          fmaf(w.y, packed_dot<S, DC>(f.dw, vtp[1]),
                               fmaf(w.z, packed_dot<S, DC>(f.dw, vtp[2]), w.w * packed_dot<S, DC>(f.dw, vtp[3]))));
            } else {
                // w = (fx, fy, fx*fy, live)
#pragma unroll
                for (int d = 0; d < DC; ++d) {
                    const float kk = fmaf(w.z, kt[3][d], fmaf(w.y, kt[2][d], fmaf(w.x, kt[1][d], kt[0][d])));
                    const float vv = fmaf(w.z, vt[3][d], fmaf(w.y, vt[2][d], fmaf(w.x, vt[1][d], vt[0][d])));
                    dot = fmaf(qf[d], kk, dot);
                    dp = fmaf(dof[d], vv, dp);
                }
            }
            dot = group_sum<G>(dot);
            dp = group_sum<G>(dp);
            float p_n = __builtin_amdgcn_exp2f(dot * qscale - lse);
            if constexpr (!kPacked) p_n *= w.w;                    // entries past the end of the list
            const float dss = p_n * (dp - delta) * dm.sm_scale;
            // this lane's row of the update: packed: the weight of tap (lane & 3); fp32: the moment
            // (1, fx, fy, fx*fy)[lane & 3]. The four lanes of a block sit in one slot (G is a multiple of 4),
            // so they share the sample and supply its four coefficients between them.
            float fxs, fys;
            if constexpr (kPacked) {
                const float2 ff = s_f[wave][buf * kWave + j0 + slot];
                fxs = ff.x;
                fys = ff.y;
            } else {
                fxs = w.x;
                fys = w.y;
            }
            float cl = fmaf(fxs, row_sx, row_ox) * fmaf(fys, row_sy, row_oy);
            if constexpr (kPacked) cl = (fys == fys) ? cl : 0.0f;       // dead entry: p_n is finite, the row is 0
            const float ck = cl * dss, cv = cl * p_n;
#pragma unroll
            for (int d = 0; d < DC; ++d) {
                mK[d] = block_outer_fma(ck, qf[d], mK[d]);
                mV[d] = block_outer_fma(cv, dof[d], mV[d]);
            }
            }
        };
        static_assert(kWave % (2 * NS) == 0, "a block of 64 entries is a whole number of trip pairs");
        // entries are fetched one block ahead of their tables; with the pairs handed over two, and the pairs -- whose
        // addresses come from the ids -- one
        CellEntry e_a, e_b{0u, 0.f, 0.f};
        float2 pd_a = make_float2(0.f, 0.f);
        {
            const CellEntry e0 = load_entry_c(lo);
            e_a = load_entry_c(lo + kWave);
            float2 pd0 = make_float2(0.f, 0.f);
            if constexpr (HANDED) {
                e_b = load_entry_c(lo + 2 * kWave);
                pd0 = load_pair(e0.id);
                pd_a = load_pair(e_a.id);
            }
            tables(lo, 0, e0, pd0);
        }
        wave_lds_sync();
        RowFetch<kRowWords> fa, fb;
        issue(0, 0, fa);
        int cur = 0;
        for (unsigned c0 = lo;; c0 += kWave) {
            const bool has_next = c0 + kWave < hi;
            CellEntry e_c;
            float2 pd_b = make_float2(0.f, 0.f);
            if constexpr (HANDED) {
                pd_b = load_pair(e_b.id);
                e_c = load_entry_c(c0 + 3 * kWave);
            } else {
                e_c = load_entry_c(c0 + 2 * kWave);
            }
            __builtin_amdgcn_sched_barrier(0);         // (requested here, not where they are used)
            // (a list of one block, the common case where lists are short, makes no second set of tables)
            if (has_next) {
                wave_lds_sync();
                tables(c0 + kWave, cur ^ 1, e_a, pd_a);
                wave_lds_sync();
            }
            const int cnt = (int)min((unsigned)kWave, hi - c0);
            int j0 = 0;
            do {
                issue(cur, j0 + NS, fb);
                __builtin_amdgcn_sched_barrier(0);     // (keeps the requests where they are written)
                consume(cur, j0, fa);
                __builtin_amdgcn_sched_barrier(0);
                // the next pair of trips: of this block, or the first of the next block
                const bool over = j0 + 2 * NS >= kWave && has_next;
                issue(over ? cur ^ 1 : cur, (j0 + 2 * NS) & (kWave - 1), fa);
                __builtin_amdgcn_sched_barrier(0);
                consume(cur, j0 + NS, fb);
                __builtin_amdgcn_sched_barrier(0);
                j0 += 2 * NS;
            } while (j0 < cnt);
            if (!has_next) break;
            if constexpr (HANDED) {
                e_a = e_b;
                pd_a = pd_b;
                e_b = e_c;
            } else {
                e_a = e_c;
            }
            cur ^= 1;
        }
    }
#pragma unroll
    for (int tpi = 0; tpi < 4; ++tpi) {
#pragma unroll
        for (int d = 0; d < DC; ++d) { aK[tpi][d] = mK[d][tpi]; aV[tpi][d] = mV[d][tpi]; }
    }
    if constexpr (!kPacked) {
        // moments -> pixels (linear, so it can be done on the slots' partial sums):
        // w00 = 1 - fx - fy + fx*fy, w01 = fx - fx*fy, w10 = fy - fx*fy, w11 = fx*fy
#pragma unroll
        for (int d = 0; d < DC; ++d) {
            aK[0][d] = (aK[0][d] - aK[1][d]) - (aK[2][d] - aK[3][d]);
            aK[1][d] -= aK[3][d];
            aK[2][d] -= aK[3][d];
            aV[0][d] = (aV[0][d] - aV[1][d]) - (aV[2][d] - aV[3][d]);
            aV[1][d] -= aV[3][d];
            aV[2][d] -= aV[3][d];
        }
    }
    // Sum the NS slots. First the steps that halve what a lane holds (lane bits 16 and 32), reduce-scatters on the
    // lane-swap instructions: a step adds the two halves and leaves each half with one half of the taps, so that in
    // the end lane bit 16 and lane bit 32 select the tap a lane holds (G <= 16), or bit 32 the tap pair
    // (G = 32), and all 64 lanes carry sums that go to memory. Then, on the quarter that is left, slots that differ
    // in lane bits below 16 by rotations of the 16 lanes (by 8, and by 4 once the lanes 8 apart agree).
    static_assert(G <= 32, "at least two slots");
    constexpr int kTapsHeld = G <= 16 ? 1 : 2;             // taps a lane holds after the reduce-scatters
    float hK[kTapsHeld][DC], hV[kTapsHeld][DC];
    if constexpr (G <= 16) {
#pragma unroll
        for (int d = 0; d < DC; ++d) {
            // bit 16: rows {0, 1} | {2, 3}; then bit 32: first | second of the pair
            const float k0 = swap_add_16(aK[0][d], aK[2][d]), k1 = swap_add_16(aK[1][d], aK[3][d]);
            const float v0 = swap_add_16(aV[0][d], aV[2][d]), v1 = swap_add_16(aV[1][d], aV[3][d]);
            hK[0][d] = swap_add_32(k0, k1);
            hV[0][d] = swap_add_32(v0, v1);
            if constexpr (G < 16) { hK[0][d] += row_rotate<8>(hK[0][d]); hV[0][d] += row_rotate<8>(hV[0][d]); }
            if constexpr (G < 8) { hK[0][d] += row_rotate<4>(hK[0][d]); hV[0][d] += row_rotate<4>(hV[0][d]); }
        }
    } else {
#pragma unroll
        for (int d = 0; d < DC; ++d) {
            hK[0][d] = swap_add_32(aK[0][d], aK[2][d]);
            hK[1][d] = swap_add_32(aK[1][d], aK[3][d]);
            hV[0][d] = swap_add_32(aV[0][d], aV[2][d]);
            hV[1][d] = swap_add_32(aV[1][d], aV[3][d]);
        }
    }
    // tap of hK[i] / hV[i] in this lane
    const int held0 = G <= 16 ? ((lane >> 4) & 1) * 2 + (lane >> 5) : (lane >> 5) * 2;
    // Through LDS into memory order: the four rows of dk (then of dv) as 4*D consecutive floats, which the
    // wave then adds to memory 64 consecutive floats per instruction (one or two cache lines a request,
    // where a lane adding its own DC consecutive floats would touch 64 / G lines with every instruction).
    const bool writer = (lane & 15) < G;                     // (lanes that differ below bit 16 hold copies)
    float *fl = s_flush[wave];
    constexpr int kLog2D = __builtin_ctz(D);
#pragma unroll
    for (int which = 0; which < 2; ++which) {
        wave_lds_sync();
        if (writer) {
#pragma unroll
            for (int i = 0; i < kTapsHeld; ++i) {
                float *dst = fl + (held0 + i) * D + lane_elem;
#pragma unroll
                for (int d = 0; d < DC; d += 4)
                    *reinterpret_cast<float4 *>(dst + d) = which == 0
                        ? make_float4(hK[i][d], hK[i][d + 1], hK[i][d + 2], hK[i][d + 3])
                        : make_float4(hV[i][d], hV[i][d + 1], hV[i][d + 2], hV[i][d + 3]);
            }
        }
        wave_lds_sync();
        float *acc = (which == 0 ? dk_acc : dv_acc) + plane_base;
#pragma unroll
        for (int idx0 = 0; idx0 < 4 * D; idx0 += kWave) {
            const int idx = idx0 + lane;
            const int r = idx >> kLog2D, dd = idx & (D - 1);
            const bool ok = ((r & 2) ? vy1 : vy0) && ((r & 1) ? vx1 : vx0);
            const int pix = (y0 + (r >> 1)) * dm.Wimg + x0 + (r & 1);
            const float val = fl[idx];
            if (ok) {
                if constexpr (FIXED) tap_place(which, r, pix)[dd] = val;
                else atomicAdd(acc + (size_t)pix * dm.acc_pixel<S, D>() + dd, val);
            }
        }
    }
}

#define DSDPA_CELL_ARGS                                                                                                    \
    const void *__restrict__ q_, const void *__restrict__ k_, const void *__restrict__ v_,                                 \
    const float2 *__restrict__ stats_, const void *__restrict__ dout_, const unsigned *__restrict__ start,                  \
    const unsigned *__restrict__ sorted, const uint4 *__restrict__ items, const float2 *__restrict__ handed_,               \
    float *__restrict__ dk_acc, float *__restrict__ dv_acc, GradDims dm, int NC, CellGrid cg

template <typename S, int D, int DC, bool HANDED, bool FIXED>
__global__ __launch_bounds__(kCellWaves *kWave, HANDED ? (DC <= 4 ? 5 : (S::kBytes == 2 ? 3 : 4))
                                                       : DC <= 4 ? (S::kBytes == 2 && D >= 64 ? 5 : 4) : (S::kBytes == 2 ? 3 : 2))
void bwd_dkdv_cell_kernel(DSDPA_CELL_ARGS)
{
    const unsigned work = (unsigned)xcd_logical_block(blockIdx.x, gridDim.x) * kCellWaves + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (work >= cg.nwork) return;
    const unsigned t = cg.div_cells.div(work);                 // plane-major
    cell_sums<S, D, DC, HANDED, FIXED>(t + cg.t0, (int)(work - t * (unsigned)cg.ncells), q_, k_, v_, stats_, dout_, start, sorted,
                                       items, handed_, dk_acc, dv_acc, dm, NC, cg);
}

// dk and dv of the planes [t0, t0 + nplanes) of the (batch, head, key view) order from the four taps' sums of the deterministic
// backward, in the order 00 + 01, 10 + 11, their sum. VE elements (16 bytes of the storage type) a thread. Bound by the
// eight floats read per element of dk and dv.
template <typename S, int D>
__global__ __launch_bounds__(256) void combine_taps_kernel(const float *__restrict__ dk_taps, const float *__restrict__ dv_taps,
                                                           void *__restrict__ dk_, void *__restrict__ dv_, GradDims dm, CellGrid cg)
{
    constexpr int VE = S::kBytes == 4 ? 4 : 8;
    const unsigned per = (unsigned)dm.L * (D / VE);                          // threads per plane
    const unsigned at = blockIdx.x * 256u + threadIdx.x, t = blockIdx.y;     // of the plane t of this launch
    if (at >= per) return;
    const unsigned bhl = cg.div_v.div(t + cg.t0), s2 = t + cg.t0 - bhl * (unsigned)dm.V, bh = (unsigned)cg.bh0 + bhl;
    const unsigned b = cg.div_h.div(bh), h = bh - b * (unsigned)dm.H;
    const unsigned pix = at / (D / VE);
    const size_t dst = dm.dkv_plane((int)b, (int)s2, (int)h) + pix * (unsigned)dm.dkv_sl + (at - pix * (D / VE)) * VE;
    const size_t tap = (size_t)cg.nplanes * dm.L * D;
#pragma unroll
    for (int which = 0; which < 2; ++which) {
        const float *src = (which == 0 ? dk_taps : dv_taps) + (size_t)t * dm.L * D + (size_t)at * VE;
        float x[4][VE];
#pragma unroll
        for (int r = 0; r < 4; ++r) load_chunk<F32, VE>(src + r * tap, x[r]);
#pragma unroll
        for (int d = 0; d < VE; ++d) x[0][d] = (x[0][d] + x[1][d]) + (x[2][d] + x[3][d]);
        store_chunk<S, VE>((char *)(which == 0 ? dk_ : dv_) + dst * S::kBytes, x[0]);
    }
}

// The planes that the patch kernel has left: a loop over their work lists, at once over where there are none. left[grp]:
// see scan_end. Every XCD takes one contiguous part of the planes. (A loop costs registers and, over whole launches, time: one
// wave per SIMD less.)
template <typename S, int D, int DC>
__global__ __launch_bounds__(kCellWaves *kWave) void bwd_dkdv_cell_rest_kernel(const unsigned *__restrict__ left, DSDPA_CELL_ARGS)
{
    const bool all = mostly_long(left, dm.B * dm.V);
    unsigned most = 0u;
    for (int i = threadIdx.x & 63; i < dm.B * dm.V; i += kWave) most = max(most, items_left(left[i], all));
    most = (unsigned)__builtin_amdgcn_readfirstlane((int)wave_all(most, [](unsigned x, unsigned y) { return max(x, y); }));
    if (most == 0u) return;
    const unsigned planes = cg.nwork / (unsigned)cg.ncells, total = planes * most, parts = gridDim.x / kXcds;
    const unsigned x = blockIdx.x % kXcds, end = (unsigned)((unsigned long long)total * (x + 1) / kXcds);
    for (unsigned i = (unsigned)((unsigned long long)total * x / kXcds) + blockIdx.x / kXcds; i < end; i += parts) {
        const unsigned t = i / most, ci = i - t * most;
        const unsigned bhl = cg.div_v.div(t), b = cg.div_h.div((unsigned)cg.bh0 + bhl);
        if (ci < items_left(left[b * (unsigned)dm.V + t - bhl * (unsigned)dm.V], all))
            cell_sums<S, D, DC, true, false>(t, (int)ci, q_, k_, v_, stats_, dout_, start, sorted, items, handed_, dk_acc, dv_acc,
                                            dm, NC, cg);
    }
}

}  // namespace dsdpa
