// "Row" kernels: query-stationary forward and dq with the K/V taps read straight from memory, one query row per slot.
//
// A wave's 64 lanes are NS = 64/G slots of G = D/DC lanes, as everywhere; a slot owns one query row of a (batch, head)
// from the first sample to the last, so nothing is merged across slots at the end, and every trip has a sample for
// every slot whatever P is. Per pass of G samples lane g of a slot turns sample c0 + g of its row into a descriptor (four
// weights, four byte offsets from the plane of view 0) and parks it in LDS; then the slot walks the pass, the K and V
// taps of a step's samples requested together. Samples are counted over all key views, so only a row's last pass may
// be part full.
//
// Against a wave per row (dsdpa_gather.h, which keeps the shapes whose samples may share a window): no merge of the slots'
// states (three steps over DC + 2 values), no empty lanes in the descriptors of rows of fewer than 64 samples. Against the
// staged kernels: every tap is a row from L1 or L2, 8 * D * e bytes a sample at 64 a clock and CU where LDS gives 128, but
// no table, no staging and no barrier.
#pragma once
#include "dsdpa_cell.h"
#include "dsdpa_gather.h"

namespace dsdpa {

constexpr int kRowWaves = 4;

struct RowGrid { int nblk; FastDiv div_nblk, div_h; int bh0; };       // workgroups per (batch, head); first pair of the launch

// workgroups before the rows': whole rounds over the XCDs, so that the rows' stay where xcd_logical_block takes them to be
__host__ __device__ inline unsigned bin_blocks(unsigned groups) { return (groups + kXcds - 1) / kXcds * kXcds; }

// A slot's place: its row, clamped to the last of the (batch, head) for the slots beyond it.
struct RowSlot { bool have; unsigned bhl, b, h, s1, l, qidx; };
// (`skip`: workgroups of the launch, a multiple of 8, before those of the rows)
template <int NS>
__device__ __forceinline__ RowSlot decode_row_slot(const Dims &dm, const RowGrid &rg, int wave, int slot, unsigned skip = 0u)
{
    const unsigned bid = (unsigned)xcd_logical_block((int)(blockIdx.x - skip), (int)(gridDim.x - skip));
    RowSlot r;
    r.bhl = rg.div_nblk.div(bid);
    const unsigned bh = r.bhl + (unsigned)rg.bh0, nq = (unsigned)(dm.V * dm.L);
    r.b = rg.div_h.div(bh);
    r.h = bh - r.b * (unsigned)dm.H;
    const unsigned at = (bid - r.bhl * (unsigned)rg.nblk) * (kRowWaves * NS) + (unsigned)(wave * NS + slot);
    r.have = at < nq;
    r.qidx = min(at, nq - 1u);
    r.s1 = dm.divL.div(r.qidx);
    r.l = r.qidx - r.s1 * (unsigned)dm.L;
    return r;
}

// The descriptor of sample n (of the row's V*P) at coordinates xy: weights (0 beyond the row) and byte offsets from the
// plane of view 0 of this (batch, head).
template <int BYTES>
__device__ __forceinline__ void row_descriptor(const Taps &tp, bool valid, unsigned n, const Dims &dm, float4 &w, uint4 &e)
{
    const unsigned view = dm.divP.div(n) * (unsigned)dm.kv_sv;
    w = valid ? make_float4(tp.w[0], tp.w[1], tp.w[2], tp.w[3]) : make_float4(0.f, 0.f, 0.f, 0.f);
    const unsigned sl = (unsigned)dm.kv_sl;
    e = make_uint4((view + (unsigned)tp.pix[0] * sl) * BYTES, (view + (unsigned)tp.pix[1] * sl) * BYTES,
                   (view + (unsigned)tp.pix[2] * sl) * BYTES, (view + (unsigned)tp.pix[3] * sl) * BYTES);
}

template <typename S, int D, int DC>
__global__ __launch_bounds__(kRowWaves *kWave) void fwd_rows_kernel(
    const void *__restrict__ q_, const void *__restrict__ k_, const void *__restrict__ v_, const float *__restrict__ coords_,
    void *__restrict__ out_, float *__restrict__ lse_, Dims dm, RowGrid rg)
{
    constexpr int G = D / DC, NS = kWave / G;
    constexpr bool kPacked = S::kBytes == 2;
    constexpr int kStep = DC * S::kBytes <= 16 ? 2 : 1;           // samples per step: their eight taps in flight together
    constexpr int RW = kPacked ? DC / 2 : DC;                    // 32-bit words of a tap held by one lane
    static_assert(G >= 2 && G <= 32 && G * DC == D, "lane split");
    __shared__ float4 s_w[kRowWaves][NS * (G + 1)];             // (a pad place per slot: neither side has bank conflicts)
    __shared__ uint4 s_e[kRowWaves][NS * (G + 1)];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int g = lane % G, slot = lane / G, lane_elem = g * DC;
    const RowSlot rs = decode_row_slot<NS>(dm, rg, wave, slot);
    const unsigned lane_byte = (unsigned)lane_elem * S::kBytes;
    const size_t kv_base = dm.kv_plane((int)rs.b, 0, (int)rs.h) * S::kBytes;
    const char *kb = (const char *)k_ + kv_base, *vb = (const char *)v_ + kv_base;
    const float2 *crow = reinterpret_cast<const float2 *>(coords_) + ((size_t)rs.b * dm.V * dm.L + rs.qidx) * (size_t)dm.N;
    float4 *const my_w = s_w[wave] + slot * (G + 1);
    uint4 *const my_e = s_e[wave] + slot * (G + 1);

    const float qscale = dm.sm_scale * kLog2e;
    float qf[DC];
    uint32_t qp[kPacked ? DC / 2 : 1];
    const char *qsrc = (const char *)q_ + (dm.q_row((int)rs.b, (int)rs.s1, (int)rs.h, (int)rs.l) + lane_elem) * S::kBytes;
    if constexpr (kPacked) load_packed<S, DC>(qsrc, qp);
    else {
        load_chunk<S, DC>(qsrc, qf);
#pragma unroll
        for (int d = 0; d < DC; ++d) qf[d] *= qscale;
    }
    float m = kNegBig, lsum = 0.f, acc[DC];
#pragma unroll
    for (int d = 0; d < DC; ++d) acc[d] = 0.f;

    // the n samples of a pass from the t-th on
    auto step = [&](auto n, int t) {
        constexpr int U = decltype(n)::value;
        float4 wt[U];
        uint32_t kr[U][4][RW], vr[U][4][RW];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            wt[u] = my_w[t + u];
            const uint4 o = lane_offsets(my_e[t + u], lane_byte);
            load_words<RW>(kb + o.x, kr[u][0]);
            load_words<RW>(kb + o.y, kr[u][1]);
            load_words<RW>(kb + o.z, kr[u][2]);
            load_words<RW>(kb + o.w, kr[u][3]);
            load_words<RW>(vb + o.x, vr[u][0]);
            load_words<RW>(vb + o.y, vr[u][1]);
            load_words<RW>(vb + o.z, vr[u][2]);
            load_words<RW>(vb + o.w, vr[u][3]);
        }
        float s[U], mc = m;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const float4 x = wt[u];
            float dot = 0.f;
            if constexpr (kPacked) {
                const float d0 = packed_dot<S, DC>(qp, kr[u][0]), d1 = packed_dot<S, DC>(qp, kr[u][1]);
                const float d2 = packed_dot<S, DC>(qp, kr[u][2]), d3 = packed_dot<S, DC>(qp, kr[u][3]);
                dot = qscale * fmaf(x.x, d0, fmaf(x.y, d1, fmaf(x.z, d2, x.w * d3)));
            } else {
#pragma unroll
                for (int d = 0; d < DC; ++d) {
                    const float kk = fmaf(x.x, __uint_as_float(kr[u][0][d]), fmaf(x.y, __uint_as_float(kr[u][1][d]),
                                     fmaf(x.z, __uint_as_float(kr[u][2][d]), x.w * __uint_as_float(kr[u][3][d]))));
                    dot = fmaf(qf[d], kk, dot);
                }
            }
            s[u] = group_sum<G>(dot);
            mc = fmaxf(mc, s[u]);
        }
        const float alpha = __builtin_amdgcn_exp2f(m - mc);
        m = mc;
        lsum *= alpha;
#pragma unroll
        for (int d = 0; d < DC; ++d) acc[d] *= alpha;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const float p = __builtin_amdgcn_exp2f(s[u] - mc);
            lsum += p;
            const float c[4] = { p * wt[u].x, p * wt[u].y, p * wt[u].z, p * wt[u].w };
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float x[DC];
                widen_words<S, DC>(vr[u][i], x);
#pragma unroll
                for (int d = 0; d < DC; ++d) acc[d] = fmaf(c[i], x[d], acc[d]);
            }
        }
    };

    float2 xy = crow[min(g, dm.N - 1)];
    for (int c0 = 0; c0 < dm.N; c0 += G) {
        const int n = c0 + g, cnt = min(G, dm.N - c0);
        const Taps tp = make_taps(xy.x, xy.y, dm.Wimg, dm.Himg);
        xy = crow[min(n + G, dm.N - 1)];                          // (the next pass', a pass ahead)
        float4 w;
        uint4 e;
        row_descriptor<S::kBytes>(tp, n < dm.N, (unsigned)min(n, dm.N - 1), dm, w, e);
        wave_lds_sync();
        my_w[g] = w;
        my_e[g] = e;
        wave_lds_sync();
        // (an odd sample on its own: a second one of weight 0 would make NaN of an infinite V)
        int t = 0;
        for (; t + kStep <= cnt; t += kStep) step(std::integral_constant<int, kStep>{}, t);
        if (kStep > 1 && t < cnt) step(std::integral_constant<int, 1>{}, t);
    }
    if (!rs.have) return;
    const size_t row = (((size_t)rs.b * dm.V + rs.s1) * dm.H + rs.h) * dm.L + rs.l;
    const float inv = 1.0f / lsum;
#pragma unroll
    for (int d = 0; d < DC; ++d) acc[d] *= inv;
    store_chunk<S, DC>((char *)out_ + (row * D + lane_elem) * S::kBytes, acc);
    if (g == 0) lse_[row] = m + __log2f(lsum);
}

// dq, the rows' (lse, delta) (stats_ may be null), the pairs for the dk/dv kernel (handed_ may be null; see
// bwd_dq_gather_kernel) and, with CG, the gradient of the coordinates: per-tap dot products instead of blend-then-dot, each
// lane's part of the two derivatives summed over the slot, and one pair of atomics per pass from the lane that owns the sample.
// BIN: the binning of few samples, which reads coords only and is wanted by the kernel behind this one, takes the launch's first workgroups,
// one a (batch, key view): a launch less, and its chain of waits beside the rows'. Binning and dq, us, in two launches / in one: 18x18,
// 2 views x 2 samples, 32 heads, D = 32, fp32 6.6 + 13.1 / 12.5, bf16 6.2 + 8.3 / 9.8; 20x20, 2 x 2, 8 heads, D = 128, fp32
// 6.1 + 14.8 / 14.8; 20x18, 4 x 1, 8 heads, D = 16, fp32 6.9 + 5.1 / 7.6.
// STEP samples have their taps in flight together: two (fp32 112 to 114 registers, 16 bits 102 to 127: 4 waves a SIMD; also with the
// coordinate gradient and the binning) or one (fp32 up to D = 128 80, 6 waves; with the coordinate gradient 96, 5 waves, but bf16 121 and fp16, D =
// 16 107), see row_step.
// Waves a SIMD that the compiler is held to: six in fp32 with one sample and D <= 128 also where it bins (held to four it took 84 registers,
// five waves, where row_step counts six; dq of 18x18, 2 views x 2 samples, 16 to 96 heads, D = 32, is the same with either). Rows of 1 KB
// that bin get four and no more, the taps of a sample all in flight (16x20, 2 x 3, D = 256, us, with four / five 30 / 34).
template <typename S, int D, bool CG, int STEP, bool BIN>
constexpr int kRowDqWaves = !BIN || S::kBytes == 2 ? 1 : !CG && STEP == 1 && D <= 128 ? 6 : 4;
template <typename S, int D, bool BIN> constexpr int kRowDqWavesMost = BIN && D * S::kBytes >= 1024 ? 4 : 8;
template <typename S, int D, int DC, bool CG, int STEP, bool BIN>
__global__ __launch_bounds__(kRowWaves *kWave) __attribute__((
    amdgpu_waves_per_eu(kRowDqWaves<S, D, CG, STEP, BIN>, kRowDqWavesMost<S, D, BIN>))) void bwd_dq_rows_kernel(
    const void *__restrict__ q_, const void *__restrict__ k_, const void *__restrict__ v_, const float *__restrict__ coords_,
    const void *__restrict__ out_, const float *__restrict__ lse_, const void *__restrict__ dout_, void *__restrict__ dq_,
    float2 *__restrict__ stats_, float *__restrict__ dcoords_, float2 *__restrict__ handed_, GradDims dm, RowGrid rg, BinJob bj)
{
    constexpr int G = D / DC, NS = kWave / G;
    // dot products of 16-bit pairs as they are stored; with the coordinate gradient in bf16 only, where widening costs an instruction an
    // element: fp16's halves are widened by the multiply-add that takes them, and its forms differ by 5 % either
    // way (us, pairs / widened: 40x28, 4 views x 8, D = 64 99 / 104, 32x19, 2 x 3 21.8 / 19.9)
    constexpr bool kPacked = S::kBytes == 2 && (!CG || S::kBf16);
    constexpr int RW = DC * S::kBytes / 4;
    static_assert(G >= 2 && G <= 32 && G * DC == D, "lane split");
    __shared__ float4 s_w[kRowWaves][NS * (G + 1)];
    __shared__ uint4 s_e[kRowWaves][NS * (G + 1)];
    __shared__ float4 s_gx[CG ? kRowWaves : 1][CG ? NS * (G + 1) : 1], s_gy[CG ? kRowWaves : 1][CG ? NS * (G + 1) : 1];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int g = lane % G, slot = lane / G, lane_elem = g * DC;
    const unsigned skip = BIN ? bin_blocks(bj.groups) : 0u;
    if constexpr (BIN) {
        if (blockIdx.x < skip) {
            extern __shared__ unsigned s_hist[];
            if (blockIdx.x < bj.groups) bin_one_group<kRowWaves * kWave>(coords_, dm, bj, blockIdx.x, s_hist);
            return;
        }
    }
    const RowSlot rs = decode_row_slot<NS>(dm, rg, wave, slot, skip);
    const unsigned lane_byte = (unsigned)lane_elem * S::kBytes;
    const size_t kv_base = dm.kv_plane((int)rs.b, 0, (int)rs.h) * S::kBytes;
    const char *kb = (const char *)k_ + kv_base, *vb = (const char *)v_ + kv_base;
    const size_t crow_at = ((size_t)rs.b * dm.V * dm.L + rs.qidx) * (size_t)dm.N;
    const float2 *crow = reinterpret_cast<const float2 *>(coords_) + crow_at;
    float4 *const my_w = s_w[wave] + slot * (G + 1);
    uint4 *const my_e = s_e[wave] + slot * (G + 1);

    const size_t row = (((size_t)rs.b * dm.V + rs.s1) * dm.H + rs.h) * dm.L + rs.l;
    const size_t roff = (row * D + lane_elem) * S::kBytes;
    float qf[DC], dof[DC], dqa[DC];
    uint32_t dop[kPacked ? DC / 2 : 1], qp[kPacked && CG ? DC / 2 : 1];
    float delta = 0.f;
    {
        float of[DC];
        load_chunk<S, DC>((const char *)q_ + (dm.q_row((int)rs.b, (int)rs.s1, (int)rs.h, (int)rs.l) + lane_elem) * S::kBytes, qf);
        load_chunk<S, DC>((const char *)dout_ + roff, dof);
        load_chunk<S, DC>((const char *)out_ + roff, of);
        if constexpr (kPacked) load_packed<S, DC>((const char *)dout_ + roff, dop);
        if constexpr (kPacked && CG)
            load_packed<S, DC>((const char *)q_ + (dm.q_row((int)rs.b, (int)rs.s1, (int)rs.h, (int)rs.l) + lane_elem) * S::kBytes, qp);
#pragma unroll
        for (int d = 0; d < DC; ++d) { delta = fmaf(dof[d], of[d], delta); dqa[d] = 0.f; }
        delta = group_sum<G>(delta);
    }
    const float qscale = dm.sm_scale * kLog2e, lse = lse_[row];
    if (stats_ && rs.have && g == 0) stats_[row] = make_float2(lse, delta);
    float2 *handed_row = handed_ ? handed_ + ((size_t)rs.bhl * dm.V * dm.L + rs.qidx) * (size_t)dm.N : nullptr;

    float2 xy = crow[min(g, dm.N - 1)];
    for (int c0 = 0; c0 < dm.N; c0 += G) {
        const int n = c0 + g, cnt = min(G, dm.N - c0);
        const Taps tp = make_taps(xy.x, xy.y, dm.Wimg, dm.Himg);
        float4 w;
        uint4 e;
        row_descriptor<S::kBytes>(tp, n < dm.N, (unsigned)min(n, dm.N - 1), dm, w, e);
        wave_lds_sync();
        my_w[g] = w;
        my_e[g] = e;
        if constexpr (CG) {
            const TapGrads tg = make_tap_grads(xy.x, xy.y, dm.Wimg, dm.Himg);
            s_gx[wave][slot * (G + 1) + g] = make_float4(tg.gx[0], tg.gx[1], tg.gx[2], tg.gx[3]);
            s_gy[wave][slot * (G + 1) + g] = make_float4(tg.gy[0], tg.gy[1], tg.gy[2], tg.gy[3]);
        }
        xy = crow[min(n + G, dm.N - 1)];
        wave_lds_sync();
        float my_p = 0.f, my_ds = 0.f, my_gx = 0.f, my_gy = 0.f;
        auto one = [&](int t, const float4 &x, const uint32_t (&kr)[4][RW], const uint32_t (&vr)[4][RW]) {
            const float wt[4] = { x.x, x.y, x.z, x.w };
            float kk[DC], dot = 0.f, dp = 0.f, dk_t[4], dv_t[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float tk[DC];
                widen_words<S, DC>(kr[i], tk);
                dk_t[i] = dv_t[i] = 0.f;
#pragma unroll
                for (int d = 0; d < DC; ++d) {
                    kk[d] = i == 0 ? wt[0] * tk[d] : fmaf(wt[i], tk[d], kk[d]);
                    if constexpr (CG && !kPacked) dk_t[i] = fmaf(qf[d], tk[d], dk_t[i]);
                }
                if constexpr (CG && kPacked) dk_t[i] = packed_dot<S, DC>(qp, kr[i]);
                if constexpr (CG) dot = fmaf(wt[i], dk_t[i], dot);
                if constexpr (CG && S::kBf16) __builtin_amdgcn_sched_barrier(0);   // (widening tap by tap: registers for four waves a SIMD)
                if constexpr (kPacked) {
                    dv_t[i] = packed_dot<S, DC>(dop, vr[i]);
                    dp = fmaf(wt[i], dv_t[i], dp);
                } else {
                    float tv[DC];
                    widen_words<S, DC>(vr[i], tv);
#pragma unroll
                    for (int d = 0; d < DC; ++d) dv_t[i] = fmaf(dof[d], tv[d], dv_t[i]);
                    dp = fmaf(wt[i], dv_t[i], dp);
                }
            }
            if constexpr (!CG) {
#pragma unroll
                for (int d = 0; d < DC; ++d) dot = fmaf(qf[d], kk[d], dot);
            }
            dot = group_sum<G>(dot);
            dp = group_sum<G>(dp);
            const float p = __builtin_amdgcn_exp2f(dot * qscale - lse);
            const float ds = p * (dp - delta);
#pragma unroll
            for (int d = 0; d < DC; ++d) dqa[d] = fmaf(ds, kk[d], dqa[d]);
            if (t == g) { my_p = p; my_ds = ds; }
            if constexpr (CG) {
                const float4 ax = s_gx[wave][slot * (G + 1) + t], ay = s_gy[wave][slot * (G + 1) + t];
                const float a = ds * dm.sm_scale;
                const float g0 = fmaf(a, dk_t[0], p * dv_t[0]), g1 = fmaf(a, dk_t[1], p * dv_t[1]);
                const float g2 = fmaf(a, dk_t[2], p * dv_t[2]), g3 = fmaf(a, dk_t[3], p * dv_t[3]);
                const float gx = group_sum<G>(fmaf(ax.x, g0, fmaf(ax.y, g1, fmaf(ax.z, g2, ax.w * g3))));
                const float gy = group_sum<G>(fmaf(ay.x, g0, fmaf(ay.y, g1, fmaf(ay.z, g2, ay.w * g3))));
                if (t == g) { my_gx = gx; my_gy = gy; }
            }
        };
        // the n samples from the t-th on: their taps in flight together
        auto step = [&](auto n, int t) {
            constexpr int U = decltype(n)::value;
            float4 xs[U];
            uint32_t kr[U][4][RW], vr[U][4][RW];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                xs[u] = my_w[t + u];
                const uint4 o = lane_offsets(my_e[t + u], lane_byte);
                load_words<RW>(kb + o.x, kr[u][0]);
                load_words<RW>(kb + o.y, kr[u][1]);
                load_words<RW>(kb + o.z, kr[u][2]);
                load_words<RW>(kb + o.w, kr[u][3]);
                load_words<RW>(vb + o.x, vr[u][0]);
                load_words<RW>(vb + o.y, vr[u][1]);
                load_words<RW>(vb + o.z, vr[u][2]);
                load_words<RW>(vb + o.w, vr[u][3]);
            }
            // (the second: 96 registers for 100, five waves; 50x50, 4 views x 4 samples, D = 32, 16 heads, coordinate gradient, fp16 197 -> 185 us)
            if constexpr (U > 1 || (CG && S::kBytes == 2 && !S::kBf16 && D <= 32 && !BIN)) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < U; ++u) one(t + u, xs[u], kr[u], vr[u]);
        };
        int t = 0;
        for (; t + STEP <= cnt; t += STEP) step(std::integral_constant<int, STEP>{}, t);
        if (STEP > 1 && t < cnt) step(std::integral_constant<int, 1>{}, t);
        if (rs.have && n < dm.N) {
            if (handed_row) handed_row[n] = make_float2(my_p, my_ds * dm.sm_scale);
            if constexpr (CG) {
                float *dst = dcoords_ + 2 * (crow_at + (size_t)n);
                atomicAdd(dst, my_gx);
                atomicAdd(dst + 1, my_gy);
            }
        }
    }
    if (rs.have) {
        // (decoded anew: the row's place in dq is not kept in registers through the loop)
        int slot_here = slot;
        asm volatile("" : "+v"(slot_here));
        const RowSlot re = decode_row_slot<NS>(dm, rg, wave, slot_here, skip);
#pragma unroll
        for (int d = 0; d < DC; ++d) dqa[d] *= dm.sm_scale;
        store_chunk<S, DC>((char *)dq_ + (dm.dq_bh((int)re.b, (int)re.h) + dm.dq_at(re.s1, re.l) + lane_elem) * S::kBytes, dqa);
    }
}

}  // namespace dsdpa
