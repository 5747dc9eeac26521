// Host-side state shared by the translation units of libdsdpa.so: error slot, kernel-path selector,
// kernel timer. Defined in dsdpa_api.hip.
#pragma once
#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>

#include <atomic>
#include <mutex>
#include <vector>

#include "../../include/dsdpa.h"

namespace dsdpa {

extern thread_local int g_last_hip_error;
extern std::atomic<int> g_path;

// Optional kernel timer: while enabled, every main forward/backward kernel launch carries a pair of HIP
// events. Process-wide (a framework may run the backward pass on another thread than the forward).
// The events ride on the kernel's own dispatch (hipExtLaunchKernelGGL's start/stop events: the start and
// end timestamps of that dispatch), not on hipEventRecord: an event recorded between two kernels costs
// about 5 us of idle GPU each (measured: 10 us gaps between timed kernels, none between untimed ones),
// which would make the timed step slower than the untimed one.
struct EventPair { hipEvent_t start, stop; };
struct KernelTimer {
    std::atomic<bool> on{false};
    std::mutex mu;
    std::vector<EventPair> pairs[5];   // [0] forward, [1] backward dk/dv, [2] backward dq, [3] cell binning (one pair per launch), [4] descriptor table
};
extern KernelTimer g_timer;

// One timed item: a single launch (pass start() and stop() to it) or a run of launches (start() to the
// first, stop() to the last). record = true: the item contains launches made by a library routine, which
// cannot carry events; then the pair is recorded around the run with hipEventRecord.
struct ScopedKernelTimer {
    hipStream_t st;
    EventPair ev{nullptr, nullptr};
    int which;
    bool armed = false, record;
    mutable bool handed_out = false;       // a launch took the events (or they were recorded around a run)
    ScopedKernelTimer(int which_, hipStream_t st_, bool record_ = false) : st(st_), which(which_), record(record_)
    {
        if (!g_timer.on.load(std::memory_order_relaxed)) return;
        if (hipEventCreate(&ev.start) != hipSuccess) return;
        if (hipEventCreate(&ev.stop) != hipSuccess) { (void)hipEventDestroy(ev.start); return; }
        armed = record ? hipEventRecord(ev.start, st) == hipSuccess : true;
        handed_out = record && armed;
    }
    hipEvent_t start() const { handed_out = armed; return armed && !record ? ev.start : nullptr; }
    hipEvent_t stop() const { handed_out = armed; return armed && !record ? ev.stop : nullptr; }
    ~ScopedKernelTimer()
    {
        if (!armed) return;
        if (!handed_out) {                  // the launch never happened (an early error return)
            (void)hipEventDestroy(ev.start);
            (void)hipEventDestroy(ev.stop);
            return;
        }
        if (record) (void)hipEventRecord(ev.stop, st);
        std::lock_guard<std::mutex> lock(g_timer.mu);
        g_timer.pairs[which].push_back(ev);
    }
};

// Side lane of the backward: a second stream, per host thread and device, on which the cell binning runs
// next to the dq kernel (neither needs the other; dk/dv needs both). Fork and join are events on the
// caller's stream, so the caller sees one stream's worth of ordering. Created on first use, default
// priority, never destroyed (a handful of handles per thread that ever ran a backward).
struct SideLane {
    hipStream_t stream = nullptr;
    hipEvent_t fork = nullptr, join = nullptr;
    bool failed = false;
};
inline SideLane *side_lane()
{
    constexpr int kMaxDevices = 64;
    thread_local SideLane lanes[kMaxDevices];
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return nullptr;
    SideLane &s = lanes[dev];
    if (s.failed) return nullptr;
    if (!s.stream) {
        if (hipStreamCreateWithFlags(&s.stream, hipStreamNonBlocking) != hipSuccess ||
            hipEventCreateWithFlags(&s.fork, hipEventDisableTiming) != hipSuccess ||
            hipEventCreateWithFlags(&s.join, hipEventDisableTiming) != hipSuccess) {
            (void)hipGetLastError();
            s.failed = true;
            s.stream = nullptr;
            return nullptr;
        }
    }
    return &s;
}

// Compute units of the current device (asked once per device; 256 when the runtime will not say).
inline int device_cus()
{
    constexpr int kMaxDevices = 64;
    static std::atomic<int> cus[kMaxDevices];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) {
        (void)hipGetLastError();
        return 256;
    }
    int n = cus[dev].load(std::memory_order_relaxed);
    if (n > 0) return n;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) {
        (void)hipGetLastError();
        n = 256;
    }
    cus[dev].store(n, std::memory_order_relaxed);
    return n;
}

inline int check_launch()
{
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        g_last_hip_error = (int)e;
        return DSDPA_ERR_HIP;
    }
    return DSDPA_OK;
}

// The plane kernels (forward, dq) keep one K and one V plane of a (b, s2, h) in LDS next to their
// per-wave descriptors; they serve every shape for which that fits in the 160 KB of a gfx950 workgroup.
constexpr size_t kLdsBytes = 160 * 1024;
constexpr size_t kPlaneDescLdsBytes = 16 * 96 * (16 + 8);   // 16 waves x 96 places x (4 weights + 2 offsets)
constexpr size_t kPlaneGradLdsBytes = 16 * 96 * 8;         // + fx, fy per place (coordinate gradient)
inline bool plane_path_fits(size_t L, size_t D, size_t esize, bool coords_grad = false)
{
    return (L + 2) * 2 * D * esize + kPlaneDescLdsBytes + (coords_grad ? kPlaneGradLdsBytes : 0) <= kLdsBytes;
}

// Whether the staged dq kernel leaves dk/dv's workgroups, of some KB of LDS each, room beside its own, of which a CU holds one. Where it
// leaves little, they come in as its workgroups end, and a second round of those finds no CU with enough LDS free before dk/dv
// runs out. Backward on one stream over that on two, mean and range of 260 shapes (2 to 12 views x 4 to 63 samples, all types): one round
// of dq with 0 to 8 KB left 0.98 (0.94 to 1.05), 8 to 24 KB 1.05 (0.98 to 1.13), 24 KB and more 1.17 (0.99 to 1.50); more rounds with 0
// to 20 KB 0.93 (0.85 to 1.00), 24 KB and more 1.05 (1.00 to 1.11). A round: 256 workgroups of at most 16 waves and two blocks
// of rows (one with the coordinate gradient or 16 elements a lane).
inline bool dq_leaves_room(size_t planes, size_t V, size_t L, size_t D, size_t esize, bool coords_grad)
{
    const size_t lanes = D * esize / 16 < 16 ? D * esize / 16 : 16, rows = (coords_grad || D / lanes > 8 ? 16 : 32) * (64 / lanes);
    const bool one_round = planes * ((V * L + rows - 1) / rows) <= 256;
    const size_t used = (L + 2) * 2 * D * esize + kPlaneDescLdsBytes + (coords_grad ? kPlaneGradLdsBytes : 0);
    return used + (one_round ? 8 : 24) * 1024 <= kLdsBytes;
}

// With very few samples per view the staged kernels mostly stage: every workgroup loads all V plane pairs for P samples
// per row and view, while the row kernels touch only the rows they sample, and need no table. us a step, staged / rows, D = 32,
// 18x14: fp32 V = 8: P = 1 114 / 92, P = 2 165 / 163, P = 3 185 / 195; V = 12: P = 1 242 / 178, 2 293 / 277, 3 341 / 357; V = 4: P = 2
// 79 / 73, 3 89 / 86, 4 97 / 97; V = 2 (18x18): P = 3 85 / 78, 5 89 / 93; bf16 V = 8: P = 3 155 / 142, 4 177 / 172; V = 12: P = 3 276 /
// 262, 4 321 / 327.
inline bool few_samples_prefer_rows(size_t V, size_t P, size_t esize) { return P <= (esize == 2 ? 3 : 2) || V * P <= 6; }

// Row kernels (dsdpa_rows.h) against the gather kernels, a wave per row, for fewer than 64 samples per view. The less samples
// a row has the more the latter's empty lanes and the merge of its slots cost; the more it has the more its eight or four samples
// in flight per row pay where the launch has few rows to fill the chip with. us, gather / rows, forward: 40x40, D = 32, fp32, N = 8
// samples a row, 400 / 1600 waves of rows: 5 / 4, 10 / 6; N = 24, 1200: 12 / 16; N = 40, 400 / 1600: 9 / 14, 21 / 22; 44x20, 14080
// waves: N = 8 59 / 33. Rows of a wave sample all views at once: with the K and V planes of a (batch, head) well beyond an XCD's 4 MB of L2
// that costs misses (D = 128, 56x50, V = 5: bf16, 7 MB, forward 563 / 632, dq 930 / 689; fp32, 14 MB, 1851 / 2227 and 1023 / 2182; V = 4, dq,
// 5.5 MB, N = 100 over the image 0.82 to 0.95 of the gather kernel's speed).
//
// A workgroup of rows is long and its CU's share of the work: what the CU with the most of them has to do sets the launch's time,
// and `fill`, the mean over the most, is what is left of the rows' advantage. Gather's time over that of rows where the workgroups
// fill the CUs evenly, lower tenth and median over 2 to 12 views x 3 to 50 samples, 31x9 to 56x50, samples over the image, clustered
// and around the query's place:
//                       fp32, D = 32     64 and 128     256            bf16, D = 32     64             128 and 256
//   N <= 32, forward    1.14 1.27        1.07 1.14      1.16 1.66      1.41 1.85        1.34 1.46      1.21 1.30
//            dq         1.25 1.38        1.06 1.15      1.46 1.94      1.50 1.86        1.38 1.54      1.38 1.54
//   N <= 64, forward    1.05 1.10        1.03 1.07                     1.04 1.28        1.13 1.20      1.06 1.15
//            dq         1.10 1.18        1.02 1.08      1.58 1.88      1.20 1.39        1.14 1.26      1.20 1.38
//   beyond,  forward    1.02 1.05        1.01 1.04      1.47 1.81      0.97 1.08        1.02 1.08      1.01 1.06 (D = 256 1.08 1.15)
//            dq         1.03 1.09        1.00 1.03      1.54 2.07      1.13 1.19        1.04 1.12      1.12 1.22
// The fill that a launch needs is about the inverse of the medians. (One workgroup over five a CU, fp32, D = 64, 43x24, N = 40 to 200: 0.82 to 0.99
// without it; fp32, D = 64, 43x24, 4 views x 50 samples, clustered, 8.1 workgroups a CU: step 1035 us by rows, 948 by gather.)
inline bool row_path(size_t rows, size_t V, size_t L, size_t D, size_t P, size_t esize, bool dq)
{
    const size_t N = V * P, lanes = D * esize >= 512 ? 32 : D * esize / 16, waves = rows * lanes / 64, MB = (size_t)1 << 20;
    const bool fp32 = esize == 4;
    if (P >= 64) return false;
    if (N <= 16) return true;
    if (2 * V * L * D * esize > (!dq ? 4 : fp32 && D == 128 ? 5 : 8) * MB) return false;
    if (waves < (N <= 32 ? 2048 : N <= 64 ? 4096 : 8192)) return false;
    if (N > 32 && fp32 && D < 32) return false;
    if (N > 64 && (D < 64 || (!dq && !fp32 && D < 256))) return false;
    const size_t per = 4 * (64 / lanes), groups = rows / (V * L) * ((V * L + per - 1) / per);     // workgroups
    const size_t cus = (size_t)device_cus(), fill = 100 * groups / ((groups + cus - 1) / cus * cus);
    return fill >= (fp32 && D == 256 ? 65 : N <= 32 ? (fp32 && D >= 64 ? 88 : 80) : N <= 64 ? (fp32 ? 95 : 85) : fp32 ? 97 : 93);
}

// Samples whose taps the row dq kernel has in flight together. Two hold more registers, and in fp32 4 workgroups a CU instead of 6: there the
// number whose last round of workgroups is the fuller, two where they are even. dq, us, one / two: bf16 48x48, 6 views x 32 samples, D = 64
// 1889 / 1842; 60x50, 4 x 8, D = 16 160 / 143; 44x44, 6 x 20, D = 64 bf16 896 / 876, fp16 911 / 880, fp32 (11616 workgroups) 1653 /
// 1600; fp32 40x28, 4 x 8, D = 64 (4480: 2.9 and 4.4 rounds) 172 / 177, 37x23, 3 x 7, D = 128, one batch (1600: 1.04 and 1.6 rounds)
// 49.7 / 46.8. With the coordinate gradient one: 40x28, 4 x 8, D = 64 bf16 101 / 106, fp16 109 / 120.
inline int row_step(size_t esize, long long groups)
{
    if (esize == 2) return 2;
    const long long cus = device_cus();
    auto full = [&](long long at_once) { return (double)groups / (double)((groups + at_once - 1) / at_once * at_once); };
    return full(6 * cus) > full(4 * cus) ? 1 : 2;
}

// Whether the row dq kernel has a form that bins beside its rows: all but the one of 1 KB rows with the coordinate gradient, which would spill.
constexpr bool row_takes_bins(size_t D, size_t esize, bool coords_grad) { return !(coords_grad && D * esize >= 1024); }

// Descriptor table of the plane kernels: per coordinate pair 16 bytes of weights and 4 of packed slot
// codes (plus, for the coordinate gradient, 16 bytes of derivative weights), computed once per call by
// plane_descriptor_kernel. Empty when the plane kernels do not apply.
struct DescLayout { size_t w, e, g, bytes; };
inline size_t round256(size_t b) { return (b + 255) / 256 * 256; }
inline DescLayout desc_layout(size_t B, size_t V, size_t Himg, size_t Wimg, size_t D, size_t P, size_t esize,
                              bool coords_grad = false)
{
    DescLayout d{0, 0, 0, 0};
    const size_t L = Himg * Wimg;
    if (!plane_path_fits(L, D, esize, coords_grad)) return d;
    const size_t m = B * V * L * V * P;
    d.w = 0;
    d.e = round256(m * 16);
    d.g = d.e + round256(m * 4);
    d.bytes = d.g + (coords_grad ? round256(m * 16) : 0);
    return d;
}

// Dense-box forward (fwd_dense_kernel): for 16-bit storage and D = 64 or 128 on shapes whose planes do not fit in LDS, with
// at least a chunk's worth of samples per view. Its workspace is one flag per tile of 16 queries, telling which
// tiles are left to the gather kernel. bytes = 0: the shape does not take that path.
struct DenseLayout { size_t todo, bytes; int ntl; };
inline DenseLayout dense_layout(size_t B, size_t V, size_t H, size_t Himg, size_t Wimg, size_t D, size_t P, size_t esize)
{
    DenseLayout d{0, 0, 0};
    const size_t L = Himg * Wimg, chunks = V * ((P + 63) / 64);
    if (esize != 2 || (D != 64 && D != 128) || P < 64 || chunks > 4096 || Himg >= 65536 || Wimg >= 65536 || plane_path_fits(L, D, esize))
        return d;
    d.ntl = (int)((L + 15) / 16);
    d.todo = 0;
    d.bytes = round256(B * H * V * (size_t)d.ntl);
    return d;
}

// Slab kernels (fwd_slab_kernel, bwd_dq_slab_kernel): fp32 storage, 16 or 32 samples per view, planes that do not fit in LDS whole but do,
// twice, as slabs of 16 columns (64 bytes per pixel, image rows at a pitch of 2 mod 4 pixels), at most 1024 pixels,
// query rows of a (batch, head) within 31 bits of coordinate pairs. Needs no workspace.
inline size_t slab_buffer_bytes(size_t Himg, size_t Wimg)
{
    const size_t pitch = Wimg + ((6 - (Wimg & 3)) & 3);
    return round256(Himg * pitch * 64);
}
inline bool slab_path_fits(size_t V, size_t Himg, size_t Wimg, size_t D, size_t P, size_t esize)
{
    const size_t L = Himg * Wimg;
    // (a wave stages runs of 16 pixels of an image row, four per slab)
    // (64 samples per view go to the gather kernels, whose window mode pays where the samples cluster)
    return esize == 4 && (P == 16 || P == 32) && (D == 32 || D == 64 || D == 128) && Himg * ((Wimg + 15) / 16) <= 64 &&
           2 * slab_buffer_bytes(Himg, Wimg) + 12 * 1024 <= kLdsBytes && !plane_path_fits(L, D, esize) &&
           V * L * V * P < ((size_t)1 << 31);
}

// Forward workspace: the descriptor table, or the dense-box forward's flags (never both).
// Backward workspace, every segment rounded up to 256 bytes:
//   delta    rows floats                     dout.out per query row
//   counters B*V*NC u32                      per (batch, key view) cell counts, then fill cursors
//   start    B*V*(NC+1) u32                  exclusive scan of the counts
//   sorted   B*V*(V*L*P) u32                 the cell lists: 12-byte records (sample id, its position (fx, fy) in the
//   frac     B*V*(V*L*P) x 8 bytes           cell) that run from `sorted` on through `frac`, which follows it; the
//                                            deterministic backward sorts plain ids first
//   items    B*V*wmax x 16 bytes             work list of the dk/dv kernel: (cell, first entry, end) per item
//   handed   bhg*V*L*(V*P) x 8 bytes         (p, sm_scale*ds) per query*sample of one GROUP of bhg (batch, head) pairs,
//                                            dq kernel -> dk/dv kernel (shapes on the gather kernels, and short lists);
//                                            at most kHandedCapBytes whatever the shape
//   acc      2*n floats                      fp32 dk/dv accumulators (16-bit storage, not deterministic; in the place of `handed` where
//                                            patches of few samples need none)
//   desc     20 bytes per coordinate pair    descriptor table (only when the plane kernels apply); 36 with
//                                            the coordinate gradient
// deterministic backward only (DSDPA_FLAG_DETERMINISTIC):
//   sorted2  as sorted                       the lists with every cell's ids in ascending order
//   seg      2*B*V*NC u32                    begin / end of every list in the flat id array
//   sorttmp  sort_temp_bytes()               scratch of the segmented sort
//   taps     8 * L * D floats per plane      the sums of every cell's four taps, of dk and of dv, of a group of planes (b, h, s2)
// with NC = (Himg+1)*(Wimg+1) cells.
size_t sort_temp_bytes(size_t n, size_t segments);                       // dsdpa_sort.hip
int sort_cell_lists(void *temp, size_t temp_bytes, const unsigned *ids_in, unsigned *ids_out, size_t n,
                    size_t segments, const unsigned *seg_begin, const unsigned *seg_end, unsigned id_bits,
                    hipStream_t st);

// Samples of a (batch, key view) up to which the binning is one launch (bin_one_kernel).
constexpr int kBinOneSamples = 2 * 1024;

struct WorkspaceLayout {
    size_t delta, counters, start, sorted, frac, items, handed, handed_bytes, acc, desc, sorted2, seg, sorttmp, sorttmp_bytes, taps, total;
    int tap_planes;             // planes (b, h, s2) whose taps the buffer of the deterministic backward holds at a time
    int bh_group;               // (batch, head) pairs whose pairs the handed buffer holds at a time; 0: nothing is handed over
    bool patch;                 // dk/dv by patches where the lists are short (DSDPA_PATH_AUTO)
    unsigned spread_mean, spread_few;   // ... up to so many entries a non-empty list on average; few such lists
    DescLayout dl;
    size_t counters_bytes;
    int NC;                     // cells of the grid
    int NK, vpg;                // lists per (batch, key view) = groups of query views * NC; query views per group
    unsigned piece, wmax;       // work list of the dk/dv kernel: entries per item, items per (batch, key view)
};

// Work list of the dk/dv kernel: a cell list is cut into items of at most `piece` entries, four times the
// average list length over the whole cell grid (at least 768, a multiple of 64): lists near the average
// stay whole, the heavy ones of clustered coordinates are shared by several waves. Every item ends with a flush
// of 8*D float atomics, a quarter of the kernel's time where the lists are long (64x64, 64 samples per view,
// clustered, two groups of query views: pieces of 512 entries 1.63 ms, 768 1.58, 1024 1.60, 2048 1.68 -- the last
// pieces then run alone). NC + M/piece bounds the number of items per (batch, key view), M = V*L*P being all its
// entries.
inline void work_list_geometry(size_t V, size_t L, size_t P, size_t NC, unsigned *piece, unsigned *wmax)
{
    const size_t M = V * L * P;
    size_t pc = 4 * M / NC;
    if (pc < 768) pc = 768;
    pc = (pc + 63) / 64 * 64;
    if (pc > 0x40000000u) pc = 0x40000000u;
    *piece = (unsigned)pc;
    *wmax = (unsigned)(NC + M / pc + 1);
}
// Query views per group of the dk/dv lists (only where the dq kernel hands its pairs over: there the dk/dv kernel
// waits for the query rows it gathers and for little else). The rows of one (batch, head), q and dout, are
// 2*V*L*D*e bytes; where that is more than an XCD's 4 MB of L2, the entries -- which the cell order scatters over
// all of it -- miss L2. Lists per (group of query views, cell), worked through group by group, keep the rows in
// use to one group's: groups of at most 4 MB (64x64, D = 128, 16-bit, V = 4: 8 MB, two groups: 2.31 -> 2.07 ms;
// four groups 2.23 ms -- every group multiplies the items, each with its set-up and flush), as long as the lists
// stay long enough to pay for that (an average of 48 entries over the whole grid).
constexpr size_t kGroupRowsBytes = (size_t)4 << 20;
inline int views_per_group(size_t V, size_t L, size_t D, size_t esize, size_t P, size_t NC, bool handed)
{
    const size_t rows_bytes = 2 * V * L * D * esize, M = V * L * P, cap = kGroupRowsBytes;
    if (!handed || rows_bytes <= cap) return (int)V;
    size_t groups = (rows_bytes + cap - 1) / cap;
    if (groups > V) groups = V;
    while (groups > 1 && M / (groups * NC) < 48) --groups;
    return (int)((V + groups - 1) / groups);
}
// The dq kernel can hand (p, sm_scale * ds) of every query*sample over to the dk/dv kernel, which then neither
// recomputes them nor needs the cell's taps. The whole backward's pairs would be rows * V*P * 8 bytes (0.54 GB
// for 2 x 4 views x 8 heads x 64x64, 64 samples per view): more than the tensors, and more than the memory-side
// cache holds. So the backward runs in GROUPS of (batch, head) pairs -- dq of a group, then dk/dv of the same
// group, the cell lists being shared by all heads -- and the buffer holds one group's pairs: at most
// kHandedCapBytes, which also stay in the memory-side cache between the two kernels. Returns the (batch, head)
// pairs per group, 0 when nothing is handed over: one pair's samples beyond the cap or beyond 32-bit byte offsets. Not asked
// for by shapes on the staged kernels (dq and dk/dv run side by side there), short lists apart.
constexpr size_t kHandedCapBytes = (size_t)128 << 20;
// The deterministic backward's taps (8 floats per element of dk): a launch covers the planes whose taps fit, and ends with its
// longest list.
constexpr size_t kTapsCapBytes = (size_t)256 << 20;
inline int handed_group(size_t B, size_t V, size_t H, size_t L, size_t P)
{
    const size_t per_bh = V * L * (V * P) * 8;
    if (per_bh >= ((size_t)1 << 32) || per_bh > kHandedCapBytes) return 0;
    size_t g = kHandedCapBytes / per_bh;
    if (g > B * H) g = B * H;
    // groups of equal size (the last one may be smaller by less than one pair per group)
    const size_t ngroups = (B * H + g - 1) / g;
    return (int)((B * H + ngroups - 1) / ngroups);
}
// dk/dv by patches of 4x4 pixels (dsdpa_patch.h) where the lists are short: what the cell kernel pays per list -- 300
// instructions and 8*D float atomics, which the memory side takes at 0.3 a ns -- is then most of its time. From 1024 patches,
// which fill the chip, and up to 48 entries a list over the whole grid in 16-bit storage (32 at D = 16, where a row's products are
// the least of a visit), where the products run at 16 times the vector rate; 12 in fp32, where they run at twice. us a step,
// cells / patches, 40x28, batch 2, 4 views, 8 heads, P = 4, 8, 10 (15, 30, 38 entries): bf16 D = 16 136 / 118, 170 / 162, 181 / 185;
// D = 32 161 / 135, 225 / 217, 262 / 260; D = 64 232 / 166, 312 / 270, 353 / 325; D = 128 426 / 261, 580 / 448, 657 / 543; D = 256
// 902 / 529, 1330 / 1028, 1510 / 1249; fp32 P = 1, 3 (4, 11) D = 32 114 / 81, 149 / 134; D = 64 184 / 114, 256 / 218. bf16 18x18,
// 6 views x 8, 16 heads (43): D = 16 167 / 181, D = 32 213 / 211, D = 64 383 / 321. At 184 entries (48x48, D = 64, bf16) the kernels
// take 1150 / 1680, at 223 (14x14, D = 32, fp32) 235 / 500.
//
// The lists are counted when they are made: spread_mean is the mean of the non-empty ones up to which the patches go ahead. Behind
// it the second launch works by cells, which with the launch of patches that only clear costs up to 7 % more than cells alone. us a
// step, cells by that second launch / patches, bf16, the first shape with samples in the middle 0.7 of the image each way, P = 4, 6,
// 8, 10 (34, 50, 66, 82): D = 16 116 / 115, 133 / 141, 153 / 166, 173 / 192; D = 32 142 / 132, 176 / 173, 212 / 215, 248 / 256; D = 64
// 192 / 163, 236 / 220, 282 / 273, 330 / 329; D = 128 330 / 256, 408 / 357, 482 / 451, 565 / 551; D = 256 637 / 470, 852 / 711, 1007 / 891,
// 1190 / 1093 (105: even). P = 8 around the query's own place (56): D = 64 cells alone 271, patches 275; D = 128 474 / 439.
// Where few cells hold samples (spread_few, less than 1024 patches' worth in a launch) the longest list takes the mean's place, since
// the patch around it is most of the launch. The first shape with P = 1, bf16, 121 such cells of 37 entries, the longest 120
// (clustered): cells alone / patches D = 64 95 / 120, D = 128 133 / 175, D = 256 257 / 236; 117 cells of 38, the longest 59: D = 128
// 132 / 135, D = 256 255 / 202.
inline unsigned spread_mean(size_t D, size_t esize)
{
    return esize == 4 ? 16u : D == 16 ? 36u : D == 32 ? 52u : D == 64 ? 72u : D == 128 ? 80u : 128u;
}
inline unsigned spread_few(size_t planes) { return (unsigned)((1024 * 16 + planes - 1) / planes); }
inline bool patch_path(size_t B, size_t V, size_t H, size_t Himg, size_t Wimg, size_t D, size_t P, size_t esize, bool deterministic)
{
    const size_t L = Himg * Wimg, mean = V * L * P / ((Himg + 1) * (Wimg + 1));
    return !deterministic && L >= 16 && mean <= (esize == 4 ? 12 : D == 16 ? 32 : 48) && B * V * H * L * V * P >= ((size_t)1 << 15) &&
           B * V * H * ((Himg + 3) / 4) * ((Wimg + 3) / 4) >= 1024;
}
inline WorkspaceLayout workspace_layout(size_t B, size_t V, size_t H, size_t Himg, size_t Wimg, size_t D, size_t P,
                                        bool storage16, bool deterministic, bool coords_grad)
{
    WorkspaceLayout w;
    const size_t rows = B * V * H * Himg * Wimg;
    w.NC = (int)((Himg + 1) * (Wimg + 1));
    size_t off = 0;
    w.delta = off; off += round256(rows * 8);           // (lse, delta) per row
    const size_t L = Himg * Wimg, esize = storage16 ? 2 : 4, acc_bytes = storage16 && !deterministic ? round256(2 * rows * D * 4) : 0;
    const bool planes = plane_path_fits(L, D, esize);
    w.patch = patch_path(B, V, H, Himg, Wimg, D, P, esize, deterministic);
    w.bh_group = planes && !w.patch ? 0 : handed_group(B, V, H, L, P);
    w.patch = w.patch && w.bh_group > 0;
    w.spread_mean = spread_mean(D, esize);
    w.spread_few = w.patch ? spread_few((size_t)w.bh_group * V) : 0;
    const bool grouped = w.bh_group > 0 && !planes && !deterministic;
    w.vpg = views_per_group(V, L, D, esize, P, (size_t)w.NC, grouped);
    w.NK = w.NC * (int)((V + w.vpg - 1) / w.vpg);       // (short lists are never split: NK = NC where there are patches)
    w.counters = off; w.counters_bytes = round256(B * V * (size_t)w.NK * 4); off += w.counters_bytes;
    w.start = off; off += round256(B * V * ((size_t)w.NK + 1) * 4);
    w.sorted = off; off += round256(B * V * (V * Himg * Wimg * P) * 4);
    w.frac = off; off += round256(B * V * (V * Himg * Wimg * P) * 8);
    work_list_geometry(V, Himg * Wimg, P, (size_t)w.NK, &w.piece, &w.wmax);
    w.items = off; off += round256(B * V * (size_t)w.wmax * 16);
    // (p, sm_scale * ds) per query*sample of one group of (batch, head) pairs, handed from the dq kernel to the
    // dk/dv kernel (see handed_group)
    w.handed = off;
    w.handed_bytes = round256((size_t)w.bh_group * V * L * (V * P) * 8);
    // (the few samples of 16-bit patches that no cell kernel follows: one room for the pairs, or for the accumulators of a
    // path that was forced, whichever is in use. 18x18, 2 views x 2 samples, 32 heads, D = 32, batch 2: 12 -> 10.6 MB)
    const bool shared = w.patch && storage16 && V * L * P <= kBinOneSamples;
    w.acc = shared ? off : off + w.handed_bytes;
    off = shared ? off + (w.handed_bytes > acc_bytes ? w.handed_bytes : acc_bytes) : w.acc + acc_bytes;
    // with the coordinate gradient the staged dq kernel needs more LDS; where it no longer fits, dq takes the
    // gather kernel and no table is needed
    w.dl = desc_layout(B, V, Himg, Wimg, D, P, storage16 ? 2 : 4, coords_grad);
    w.desc = off; off += w.dl.bytes;
    w.sorted2 = w.seg = w.sorttmp = w.taps = off;
    w.tap_planes = 0;
    w.sorttmp_bytes = 0;
    if (deterministic) {
        const size_t ids = B * V * (V * Himg * Wimg * P), segs = B * V * (size_t)w.NC;
        w.sorted2 = off; off += round256(ids * 4);
        w.seg = off; off += round256(2 * segs * 4);
        w.sorttmp_bytes = round256(sort_temp_bytes(ids, segs));
        w.sorttmp = off; off += w.sorttmp_bytes;
        // dk and dv as four taps each: groups of equal size, at most kTapsCapBytes or one plane (there are no accumulators)
        const size_t per = 8 * L * D * 4, planes_all = B * H * V;
        size_t g = kTapsCapBytes / per;
        g = g < 1 ? 1 : g > planes_all ? planes_all : g;
        g = g > 32768 ? 32768 : g;                          // (a dimension of the grid)
        const size_t ngroups = (planes_all + g - 1) / g;
        w.tap_planes = (int)((planes_all + ngroups - 1) / ngroups);
        w.taps = off; off += round256((size_t)w.tap_planes * per);
    }
    w.total = off;
    return w;
}

// One storage type's forward / backward entry (argument checks, kernel selection, launches); each is
// instantiated in its own translation unit (dsdpa_f32.hip, dsdpa_bf16.hip, dsdpa_f16.hip) so that the
// three compile in parallel.
// `strides`: null (everything contiguous) or the 8 element strides of q and of k/v over (batch, view, head, pixel).
// dense_ok: the workspace has room for dense_layout() (false: the gather kernels alone do those shapes).
template <typename S>
int fwd_impl(const void *q, const void *k, const void *v, const float *coords, void *out, float *lse,
             void *workspace, int B, int V, int H, int Himg, int Wimg, int D, int P, float sm_scale,
             const long long *strides, void *stream, bool dense_ok = true);
template <typename S>
int bwd_impl(const void *q, const void *k, const void *v, const float *coords, const void *out,
             const float *lse, const void *dout, void *dq, void *dk, void *dv, float *dcoords, void *workspace,
             int B, int V, int H, int Himg, int Wimg, int D, int P, float sm_scale, const long long *strides,
             unsigned flags, void *stream);

}  // namespace dsdpa
