// dk/dv by patches of 4x4 pixels: the scatter as a matrix product, no atomics.
//
// A workgroup owns the 16 pixels of a patch of one plane (b, h, s2). The samples that touch them lie in the 5x5 cells
// around it, and since the lists of the binning are in cell order, those are five contiguous runs of list entries, one
// per row of cells. With (p, sm_scale * ds) of every sample left by the dq kernel,
//
//   dK[16 x D] = Cds[16 x entries] . Q[entries x D]          Cds[pixel][n] = w_pixel(n) * sm_scale * ds_n
//   dV[16 x D] = Cp [16 x entries] . dO[entries x D]         Cp [pixel][n] = w_pixel(n) * p_n
//
// where an entry's column of C has the bilinear weights of its (up to four) pixels inside the patch and zeros
// elsewhere. The sums are complete when the entries are done: they are stored once, in the storage type, by
// the workgroup that owns them. The price is that an entry near a patch border is visited by two or four patches
// (25/16 visits on average) and that four of a column's sixteen places are used; the matrix unit has that to spare.
//
// Per 64 entries: one lane per entry fetches its record and pair, forms the four weights times p and ds and scatters
// them into the wave's C matrices in LDS ([pixel][entry], all 64 columns or half at a time; the rest is zero and is made zero again);
// then steps of STEP entries: the lanes read their row of C as the A operand, and the query rows -- requested a step
// ahead, straight from memory into the layout of the B operand -- are multiplied:
//   16-bit storage  v_mfma_f32_16x16x32: lane group lane/16 holds eight entries, lane % 16 = column n: E = D/16
//                   consecutive elements of each row, element t of every lane in product t (so output column n of
//                   product t is element E*n + t: no data crosses lanes). The coefficients are split in parts of the storage
//                   type, one product each: two in fp16 (good to 2^-23 down to a floor, see lower_scale), three in bf16 (two
//                   are good to 2^-17, which rows that cancel show); two byte permutes make the operand of a pair of rows.
//                   The third part costs a third of the tables' LDS. us a step with 64 columns in LDS (kPatchColumns), cells / two
//                   parts / three, bf16: 18x18, 32 heads, D = 32, 6 views x 6 samples 351 / 274 / 292, 12 x 4 797 / 670 / 701; 20x20,
//                   4 x 6, D = 64 229 / 182 / 186; 40x28, 4 x 8, coherent, D = 128 581 / 425 / 441.
//   fp32            v_mfma_f32_16x16x4_f32: one entry per lane group and instruction, everything in fp32.
// fp16 has 5 bits of exponent: its coefficients are scaled by powers of two (lower_scale).
//
// A non-finite query row times the zeros of its column would reach all sixteen pixels: where a patch's sums
// come out non-finite, the workgroup works it out again entry by entry, each for the pixels it touches only.
//
// Short lists only. A patch costs its visits; the cell kernel costs its lists (300 instructions and 8*D atomics each) and
// entries, and is ahead where lists are long. The host asks for patches where the lists would be short with the samples
// spread over the image, and the binning, which counts them, decides by the mean of the non-empty lists and the longest, per
// (batch, key view) or, where many are long, for all (mostly_long). Where they are not short (samples that cluster leave
// most cells empty and the others full), the patch kernel only clears its pixels' accumulators, and a second
// launch, the cell kernel as a loop over the work list, does the sums.
#pragma once
#include "dsdpa_cell.h"
#include "dsdpa_dense.h"

namespace dsdpa {

constexpr int kPatchSide = 4, kPatchPixels = kPatchSide * kPatchSide;
constexpr int kPatchMaxWaves = 4;
// Entries whose columns of C are in LDS at a time: a block of 64, or half of it, where the tables' LDS is what limits the waves on
// a CU (bf16's three tables with 64 columns leave room for 11, with 32 for 21). dk/dv, us, 64 / 32: bf16 D = 32, 18x18, 6 views x 6
// samples, 32 heads 117 / 105, 50x50, 4 x 4 171 / 148; bf16 D = 16, 40x28, 4 x 2, 24 heads 73 / 55; fp32 D = 16, same 62 / 52. Elsewhere
// registers limit them, and the second turn of writing and clearing is not won back: a step, D = 64, 40x28, 4 x 8, bf16 273 / 275, fp16 265 /
// 269; D = 128, 4 x 4 271 / 276; fp16 D = 32, 18x18, 6 x 6 268 / 269.
template <typename S, int DP> constexpr int kPatchColumns = DP <= (S::kBf16 ? 32 : S::kBytes == 4 ? 16 : 0) ? kWave / 2 : kWave;
// dwords between two rows of C: 16-byte reads of 16 rows cover all banks
template <typename S, int DP> constexpr int kPatchPitch = kPatchColumns<S, DP> + 4;
// per wave: C of ds, C of p (bf16: and their third parts), over which the sums of DP columns pass at the end; row offsets in q and
// dout, list bounds, a flag
template <typename S, int DP> constexpr int kPatchC = kPatchPixels * kPatchPitch<S, DP>;
template <typename S> constexpr int kPatchTables = S::kBf16 ? 3 : 2;
template <typename S, int DP>
constexpr int kPatchRoom = kPatchTables<S> * kPatchC<S, DP> > kPatchPixels * DP ? kPatchTables<S> * kPatchC<S, DP> : kPatchPixels * DP;
template <typename S, int DP> constexpr int kPatchWaveDwords = kPatchRoom<S, DP> + 2 * kWave + 5 * 8 + 4;
template <typename S, int DP> constexpr size_t patch_lds_bytes(int waves) { return (size_t)waves * kPatchWaveDwords<S, DP> * 4; }

struct PatchGrid {
    int npx, npatch;                        // patches per row and per plane
    int bh0;                                // first (batch, head) pair of this launch (b * H + h)
    FastDiv div_patch, div_npx, div_v, div_h;
};

// One list entry of a patch: sample id, position in its cell, and where that cell lies: 8 * row + column of the 5x5.
struct PatchEntry { unsigned id; float fx, fy; unsigned code; };

// E elements of a row as they lie in memory (2 bytes, or 4 to 32)
template <int BYTES>
__device__ __forceinline__ void load_piece(const char *p, uint32_t (&w)[(BYTES + 3) / 4])
{
    if constexpr (BYTES == 2) w[0] = *reinterpret_cast<const uint16_t *>(p);
    else if constexpr (BYTES == 4) w[0] = *reinterpret_cast<const uint32_t *>(p);
    else load_words<BYTES / 4>(p, w);
}

// A coefficient as (high part | low part << 16) of the storage type, and in `rest` what they leave of it: a third part in
// bf16 (2^-17 without it), not used in fp16.
template <typename S>
__device__ __forceinline__ uint32_t split_pack(float c, float &rest)
{
    using T = std::conditional_t<S::kBf16, __bf16, _Float16>;
    typedef T pair_t __attribute__((ext_vector_type(2)));
    const T hi = (T)c;
    const float r = c - (float)hi;
    const T lo = (T)r;
    rest = r - (float)lo;
    return __builtin_bit_cast(uint32_t, pair_t{hi, lo});
}

template <typename S, int D, int DP>
__global__ __launch_bounds__(kPatchMaxWaves *kWave, DP > 64 ? 2 : DP > 32 && S::kBf16 ? 3 : 4) void bwd_dkdv_patch_kernel(
    const void *__restrict__ q_, const void *__restrict__ dout_, const unsigned *__restrict__ start,
    const unsigned *__restrict__ sorted, const unsigned *__restrict__ left, const float2 *__restrict__ handed_,
    void *__restrict__ dk_, void *__restrict__ dv_, float *__restrict__ dk_acc, float *__restrict__ dv_acc, GradDims dm, int NC,
    PatchGrid pg)
{
    constexpr bool k16 = S::kBytes == 2, kBf16 = S::kBf16, kF16 = k16 && !kBf16;
    constexpr int E = DP / 16;                        // elements of a row per lane
    constexpr int EPL = k16 ? 8 : 4;                  // entries per lane group and step
    constexpr int STEP = 4 * EPL, NSTEP = kWave / STEP;
    constexpr int PITCH = kPatchPitch<S, DP>, COLS = kPatchColumns<S, DP>, SPC = COLS / STEP;     // steps of the columns in LDS
    constexpr int PIECE = E * S::kBytes, WORDS = (PIECE + 3) / 4;
    static_assert(DP % 16 == 0 && D % DP == 0 && DP <= 128, "columns of a workgroup");
    extern __shared__ __attribute__((aligned(16))) unsigned smem_patch[];

    const int nw = (int)(blockDim.x >> 6);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    unsigned *const base = smem_patch + wave * kPatchWaveDwords<S, DP>;
    unsigned *const ck = base, *const cv = base + kPatchC<S, DP>, *const cl = base + 2 * kPatchC<S, DP>;       // cl: bf16's third parts, ds | p << 16
    unsigned *const s_qrow = base + kPatchRoom<S, DP>, *const s_row = s_qrow + kWave, *const s_bnd = s_row + kWave;

    // plane-major: (b, h, s2, patch)
    const unsigned work = (unsigned)xcd_logical_block(blockIdx.x, gridDim.x);
    const unsigned t = pg.div_patch.div(work);
    const int patch = (int)(work - t * (unsigned)pg.npatch);
    const unsigned bhl = pg.div_v.div(t);
    const int s2 = (int)(t - bhl * (unsigned)dm.V);
    const unsigned bh = (unsigned)pg.bh0 + bhl;
    const int b = (int)pg.div_h.div(bh), h = (int)(bh - (unsigned)b * (unsigned)dm.H);
    const int py = (int)pg.div_npx.div((unsigned)patch), px = patch - py * pg.npx;
    const size_t grp = (size_t)b * dm.V + s2;
    const int col0 = (int)blockIdx.y * DP;                               // first column of this workgroup

    const size_t M = (size_t)dm.V * dm.L * dm.P;
    const unsigned *list = sorted + grp * M * 3u;                         // 12-byte records (id, fx, fy)
    const unsigned *st = start + grp * ((size_t)NC + 1);
    const unsigned kRowBytes = D * S::kBytes;
    const size_t bh_row0 = ((size_t)b * dm.V * dm.H + h) * dm.L;
    const unsigned lane_byte = (unsigned)(col0 + (lane & 15) * E) * S::kBytes;
    const char *q_bh = (const char *)q_ + dm.q_row(b, 0, h, 0) * S::kBytes;
    const char *do_bh = (const char *)dout_ + bh_row0 * kRowBytes;
    const char *handed_bh = (const char *)(handed_ + (size_t)bhl * dm.V * dm.L * (size_t)dm.N);
    const unsigned view_rows = (unsigned)dm.H * (unsigned)dm.L;

    const size_t plane_base = dm.dkv_plane(b, s2, h);
    constexpr int VE = k16 ? 8 : 4;                               // elements of a 16-byte store
    auto pixel_of = [&](int m, unsigned &pix) -> bool {
        const int y = kPatchSide * py + (m >> 2), x = kPatchSide * px + (m & 3);
        pix = (unsigned)(y * dm.Wimg + x);
        return y < dm.Himg && x < dm.Wimg;
    };
    auto pixel_at = [&](int m, size_t &elem) -> bool {
        unsigned pix;
        const bool in = pixel_of(m, pix);
        elem = plane_base + pix * (unsigned)dm.dkv_sl + col0;
        return in;
    };
    if (left && items_left(left[grp], mostly_long(left, dm.B * dm.V)) != 0u) {
        for (int i = threadIdx.x; i < kPatchPixels * DP / 4; i += (int)blockDim.x) {
            unsigned pix;
            if (pixel_of(i * 4 / DP, pix)) {
                const size_t elem = dm.acc_plane<S, D>(b, s2, h) + pix * dm.acc_pixel<S, D>() + col0;
                *reinterpret_cast<float4 *>(dk_acc + elem + i * 4 % DP) = make_float4(0.f, 0.f, 0.f, 0.f);
                *reinterpret_cast<float4 *>(dv_acc + elem + i * 4 % DP) = make_float4(0.f, 0.f, 0.f, 0.f);
            }
        }
        return;
    }

    // The patch's entries: five runs of the list, numbered through.
    unsigned pre1, pre2, pre3, pre4, total;
    {
        const int r = lane / 6, c = lane - 6 * r;
        const int cy = kPatchSide * py + r, cx = min(kPatchSide * px + c, dm.Wimg + 1);
        unsigned v = 0u;
        if (lane < 30 && cy <= dm.Himg) v = st[cy * (dm.Wimg + 1) + cx];
        auto len = [&](int row) {
            return (unsigned)(__builtin_amdgcn_readlane((int)v, 6 * row + 5) - __builtin_amdgcn_readlane((int)v, 6 * row));
        };
        pre1 = len(0);
        pre2 = pre1 + len(1);
        pre3 = pre2 + len(2);
        pre4 = pre3 + len(3);
        total = pre4 + len(4);
        const unsigned pre = r == 0 ? 0u : r == 1 ? pre1 : r == 2 ? pre2 : r == 3 ? pre3 : pre4;
        if (lane < 30 && c < 5) s_bnd[8 * r + c] = c == 0 ? v - pre : v;     // c = 0: from the number to the place in the list
        wave_lds_sync();
    }
    // (numbers past the end repeat the last entry: no request sits under a branch)
    auto load_entry = [&](unsigned first) -> PatchEntry {
        const unsigned n = min(first + (unsigned)lane, total - 1u);
        const unsigned r = (n >= pre1 ? 1u : 0u) + (n >= pre2 ? 1u : 0u) + (n >= pre3 ? 1u : 0u) + (n >= pre4 ? 1u : 0u);
        const uint4 bd = reinterpret_cast<const uint4 *>(s_bnd)[2 * r];
        const unsigned b4 = s_bnd[8 * r + 4], at = n + bd.x;
        const unsigned c = (at >= bd.y ? 1u : 0u) + (at >= bd.z ? 1u : 0u) + (at >= bd.w ? 1u : 0u) + (at >= b4 ? 1u : 0u);
        const unsigned *rec = list + 3 * (size_t)at;
        return PatchEntry{rec[0], __uint_as_float(rec[1]), __uint_as_float(rec[2]), 8u * r + c};
    };
    // (p, sm_scale * ds) of the entry, and its query row
    struct Fetched { float2 pd; unsigned ql; };
    auto fetch = [&](unsigned id) -> Fetched {
        const unsigned ql = dm.divP.div(id), p = id - ql * (unsigned)dm.P;          // ql = s1*L + l
        const unsigned n = (unsigned)s2 * (unsigned)dm.P + p;
        Fetched f;
        f.ql = ql;
        f.pd = *reinterpret_cast<const float2 *>(handed_bh + (ql * (unsigned)dm.N + n) * 8u);
        return f;
    };
    auto offsets = [&](unsigned ql, unsigned &qrow, unsigned &row) {
        const unsigned s1 = dm.divL.div(ql), l = ql - s1 * (unsigned)dm.L;
        qrow = (s1 * (unsigned)dm.q_sv + l * (unsigned)dm.q_sl) * S::kBytes;
        row = (s1 * view_rows + l) * kRowBytes;
    };
    floatx4 mK[E], mV[E];
#pragma unroll
    for (int i = 0; i < E; ++i) { mK[i] = floatx4{0.f, 0.f, 0.f, 0.f}; mV[i] = floatx4{0.f, 0.f, 0.f, 0.f}; }
    constexpr float kByP = kF16 ? kScaleP : 1.0f;
    float scale_ds = kF16 ? kScaleDs : 1.0f, rescale = 1.0f;
    (void)rescale;

    // The coefficients of a block of 64 entries, a lane each, and the entries' row offsets. They go into C COLS entries at a time, the
    // `part`-th COLS lanes' at once, and are cleared when they have been read.
    int zat = 0;
    unsigned zmask = 0u;
    uint32_t zk[4], zv[4], zl[kBf16 ? 4 : 1];
    auto tables = [&](unsigned first, const PatchEntry &e, const Fetched &f) {
        const bool live = first + (unsigned)lane < total;
        const float2 ff = make_float2(e.fx, e.fy);
        const float gx = 1.0f - ff.x, gy = 1.0f - ff.y;
        const float w[4] = { gx * gy, ff.x * gy, gx * ff.y, ff.x * ff.y };
        const int r = (int)(e.code >> 3), c = (int)(e.code & 7u);
        const unsigned rows = (r >= 1 ? 3u : 0u) | (r <= 3 ? 12u : 0u), cols = (c >= 1 ? 5u : 0u) | (c <= 3 ? 10u : 0u);
        float ds = f.pd.y;
        if constexpr (kF16) {
            rescale = lower_scale(first_lane(wave_max(live ? fabsf(ds) : 0.f)), scale_ds);
            ds *= scale_ds;
        }
        const float p = f.pd.x * kByP;
        zmask = live ? rows & cols : 0u;
        zat = ((r - 1) * kPatchSide + (c - 1)) * PITCH + (lane & (COLS - 1));
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if constexpr (k16) {
                float rk, rv;
                zk[i] = split_pack<S>(w[i] * ds, rk);
                zv[i] = split_pack<S>(w[i] * p, rv);
                if constexpr (kBf16) zl[i] = __builtin_bit_cast(uint32_t, dsdpa_bf16x2{(__bf16)rk, (__bf16)rv});
            } else {
                zk[i] = __float_as_uint(w[i] * ds);
                zv[i] = __float_as_uint(w[i] * p);
            }
        }
        unsigned qrow, row;
        offsets(f.ql, qrow, row);
        s_qrow[lane] = qrow;
        s_row[lane] = row;
    };
    auto put_tables = [&](int part, bool clear) {
        const unsigned here = lane / COLS == part ? zmask : 0u;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (here & (1u << i)) {
                const int at = zat + ((i >> 1) * kPatchSide + (i & 1)) * PITCH;
                ck[at] = clear ? 0u : zk[i];
                cv[at] = clear ? 0u : zv[i];
                if constexpr (kBf16) cl[at] = clear ? 0u : zl[i];
            }
        }
    };

    uint32_t rq[EPL][WORDS], rd[EPL][WORDS];
    auto issue = [&](const char *src, const unsigned *offs, int s, uint32_t (&r)[EPL][WORDS]) {
        const uint4 *o = reinterpret_cast<const uint4 *>(offs + s * STEP + (lane >> 4) * EPL);
#pragma unroll
        for (int i = 0; i < EPL / 4; ++i) {
            const uint4 v = o[i];
            load_piece<PIECE>(src + (v.x + lane_byte), r[4 * i + 0]);
            load_piece<PIECE>(src + (v.y + lane_byte), r[4 * i + 1]);
            load_piece<PIECE>(src + (v.z + lane_byte), r[4 * i + 2]);
            load_piece<PIECE>(src + (v.w + lane_byte), r[4 * i + 3]);
        }
    };
    struct Coefs { uint4 x[EPL / 4]; };
    auto read_coefs = [&](const unsigned *c, int s) -> Coefs {
        Coefs f;
        const uint4 *src = reinterpret_cast<const uint4 *>(c + (lane & 15) * PITCH + s * STEP % COLS + (lane >> 4) * EPL);
#pragma unroll
        for (int i = 0; i < EPL / 4; ++i) f.x[i] = src[i];
        return f;
    };
    // (g, half: bf16's third parts, in the low or the high halves)
    auto multiply = [&](const Coefs &f, const Coefs &g, unsigned half, const uint32_t (&r)[EPL][WORDS], floatx4 (&acc)[E]) {
        if constexpr (k16) {
            auto pick = [](unsigned y, unsigned x, unsigned sel) { return __builtin_amdgcn_perm(y, x, sel); };
            auto part = [&](const Coefs &t, unsigned sel) {
                const uint4 a = t.x[0], c = t.x[EPL / 4 - 1];
                return make_uint4(pick(a.y, a.x, sel), pick(a.w, a.z, sel), pick(c.y, c.x, sel), pick(c.w, c.z, sel));
            };
            const uint4 hi = part(f, 0x05040100u), lo = part(f, 0x07060302u), third = kBf16 ? part(g, half) : hi;
#pragma unroll
            for (int i = 0; i < E; ++i) {
                const unsigned sel = (i & 1) ? 0x07060302u : 0x05040100u;
                const uint4 x = make_uint4(pick(r[1][i / 2], r[0][i / 2], sel), pick(r[3][i / 2], r[2][i / 2], sel),
                                           pick(r[EPL - 3][i / 2], r[EPL - 4][i / 2], sel), pick(r[EPL - 1][i / 2], r[EPL - 2][i / 2], sel));
                acc[i] = mfma_16x16x32<S>(hi, x, acc[i]);
                acc[i] = mfma_16x16x32<S>(lo, x, acc[i]);
                if constexpr (kBf16) acc[i] = mfma_16x16x32<S>(third, x, acc[i]);
            }
        } else {
            const uint32_t a[4] = { f.x[0].x, f.x[0].y, f.x[0].z, f.x[0].w };
#pragma unroll
            for (int j = 0; j < 4; ++j) {
#pragma unroll
                for (int i = 0; i < E; ++i)
                    acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a[j]), __uint_as_float(r[j][i]), acc[i], 0, 0, 0);
            }
        }
    };

    for (int i = lane; i < kPatchTables<S> * kPatchC<S, DP> / 4; i += kWave) reinterpret_cast<uint4 *>(base)[i] = make_uint4(0u, 0u, 0u, 0u);
    const unsigned stride = (unsigned)nw * kWave;
    unsigned first = (unsigned)wave * kWave;                      // the waves take the blocks of 64 entries in turn
    if (first < total) {
        // entries are fetched two blocks ahead of their tables, pairs one block, rows one step
        PatchEntry e1, e2;
        Fetched f1;
        {
            const PatchEntry e0 = load_entry(first);
            e1 = load_entry(first + stride);
            e2 = load_entry(first + 2 * stride);
            const Fetched f0 = fetch(e0.id);
            f1 = fetch(e1.id);
            tables(first, e0, f0);
            wave_lds_sync();                                      // (the zeros above are other lanes')
            put_tables(0, false);
        }
        wave_lds_sync();
        issue(q_bh, s_qrow, 0, rq);
        issue(do_bh, s_row, 0, rd);
        for (;;) {
            const bool more = first + stride < total;
            const Fetched f2 = fetch(e2.id);
            const PatchEntry e3 = load_entry(first + 3 * stride);
            __builtin_amdgcn_sched_barrier(0);                    // (requested here, not where they are used)
#pragma unroll
            for (int s = 0; s < NSTEP; ++s) {
                const Coefs fk = read_coefs(ck, s), fv = read_coefs(cv, s), fl = kBf16 ? read_coefs(cl, s) : Coefs{};
                if (s % SPC == SPC - 1 && (s < NSTEP - 1 || more)) {      // C has been read: the next columns
                    wave_lds_sync();
                    put_tables(s / SPC, true);
                    if (s == NSTEP - 1) tables(first + stride, e1, f1);
                    if constexpr (COLS < kWave) wave_lds_sync();      // (lanes l and l + 32 share a column: the zeros before the coefficients)
                    put_tables((s + 1) % NSTEP / SPC, false);
                    wave_lds_sync();
                }
                const int next = (s + 1) % NSTEP;
                __builtin_amdgcn_sched_barrier(0);
                multiply(fk, fl, 0x05040100u, rq, mK);
                __builtin_amdgcn_sched_barrier(0);
                issue(q_bh, s_qrow, next, rq);                    // (behind the last block: rows that nothing uses)
                __builtin_amdgcn_sched_barrier(0);
                multiply(fv, fl, 0x07060302u, rd, mV);
                __builtin_amdgcn_sched_barrier(0);
                issue(do_bh, s_row, next, rd);
                __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (kF16) {
                if (more && rescale != 1.0f) {
#pragma unroll
                    for (int i = 0; i < E; ++i) mK[i] *= rescale;
                }
            }
            if (!more) break;
            first += stride;
            e1 = e2;
            f1 = f2;
            e2 = e3;
        }
    }
    if constexpr (kF16) {
        const float uk = 1.0f / scale_ds;
#pragma unroll
        for (int i = 0; i < E; ++i) { mK[i] *= uk; mV[i] *= 1.0f / kByP; }
    }

    // Sum of the waves through LDS, and the stores: the patch as [pixel][column], dk and then dv.
    unsigned &s_bad = smem_patch[kPatchWaveDwords<S, DP> - 1];
    if (threadIdx.x == 0) s_bad = 0u;
    float z = 0.f;
#pragma unroll
    for (int i = 0; i < E; ++i) {
#pragma unroll
        for (int j = 0; j < 4; ++j) z = fmaf(mK[i][j], 0.f, fmaf(mV[i][j], 0.f, z));
    }
    __syncthreads();
    if (!(z == 0.f)) s_bad = 1u;
#pragma unroll
    for (int which = 0; which < 2; ++which) {
        float *mine = reinterpret_cast<float *>(base);
        __syncthreads();
#pragma unroll
        for (int j = 0; j < 4; ++j) {
#pragma unroll
            for (int i = 0; i < E; ++i)
                mine[(4 * (lane >> 4) + j) * DP + (lane & 15) * E + i] = which == 0 ? mK[i][j] : mV[i][j];
        }
        __syncthreads();
        const float *all = reinterpret_cast<const float *>(smem_patch);
        for (int i = threadIdx.x; i < kPatchPixels * DP / VE; i += (int)blockDim.x) {
            const int m = i * VE / DP, c = i * VE % DP;
            float sum[VE];
#pragma unroll
            for (int d = 0; d < VE; ++d) sum[d] = all[i * VE + d];
            for (int w = 1; w < nw; ++w) {
#pragma unroll
                for (int d = 0; d < VE; ++d) sum[d] += all[w * kPatchWaveDwords<S, DP> + i * VE + d];
            }
            size_t elem;
            if (pixel_at(m, elem)) store_chunk<S, VE>((char *)(which == 0 ? dk_ : dv_) + (elem + c) * S::kBytes, sum);
        }
    }
    if (s_bad == 0u) return;

    // The exact way: a wave per pixel, one entry at a time, only those that touch the pixel.
    __syncthreads();
    constexpr int CE = DP > kWave ? DP / kWave : 1;               // columns per lane: lane, lane + 64
    for (int m = wave; m < kPatchPixels; m += nw) {
        float aK[CE], aV[CE];
#pragma unroll
        for (int d = 0; d < CE; ++d) { aK[d] = 0.f; aV[d] = 0.f; }
        for (unsigned first = 0; first < total; first += kWave) {
            const PatchEntry e = load_entry(first);
            const Fetched f = fetch(e.id);
            const float2 ff = make_float2(e.fx, e.fy);
            const int dy = (m >> 2) - ((int)(e.code >> 3) - 1), dx = (m & 3) - ((int)(e.code & 7u) - 1);
            const bool on = first + (unsigned)lane < total && (dy == 0 || dy == 1) && (dx == 0 || dx == 1);
            const float w = (dy == 0 ? 1.0f - ff.y : ff.y) * (dx == 0 ? 1.0f - ff.x : ff.x);
            const float cds = w * f.pd.y, cp = w * f.pd.x;
            unsigned qrow, row;
            offsets(f.ql, qrow, row);
            unsigned long long left = __ballot(on);
            while (left) {
                const int j = __builtin_ctzll(left);
                left &= left - 1ull;
                const float a = __uint_as_float((unsigned)__builtin_amdgcn_readlane((int)__float_as_uint(cds), j));
                const float c = __uint_as_float((unsigned)__builtin_amdgcn_readlane((int)__float_as_uint(cp), j));
                const unsigned qo = (unsigned)__builtin_amdgcn_readlane((int)qrow, j), ro = (unsigned)__builtin_amdgcn_readlane((int)row, j);
#pragma unroll
                for (int d = 0; d < CE; ++d) {
                    const unsigned at = (unsigned)(col0 + min(lane + d * kWave, DP - 1)) * S::kBytes;
                    float x, y;
                    if constexpr (S::kBf16) {
                        x = bf16_to_f32(*reinterpret_cast<const uint16_t *>(q_bh + (qo + at)));
                        y = bf16_to_f32(*reinterpret_cast<const uint16_t *>(do_bh + (ro + at)));
                    } else {
                        x = (float)*reinterpret_cast<const typename S::type *>(q_bh + (qo + at));
                        y = (float)*reinterpret_cast<const typename S::type *>(do_bh + (ro + at));
                    }
                    aK[d] = fmaf(a, x, aK[d]);
                    aV[d] = fmaf(c, y, aV[d]);
                }
            }
        }
        size_t elem;
        if (!pixel_at(m, elem)) continue;
#pragma unroll
        for (int d = 0; d < CE; ++d) {
            const int c = lane + d * kWave;
            if (c >= DP) continue;
            typename S::type *pk = (typename S::type *)dk_ + elem + c, *pv = (typename S::type *)dv_ + elem + c;
            if constexpr (S::kBf16) { *pk = f32_to_bf16(aK[d]); *pv = f32_to_bf16(aV[d]); }
            else { *pk = (typename S::type)aK[d]; *pv = (typename S::type)aV[d]; }
        }
    }
}

}  // namespace dsdpa
