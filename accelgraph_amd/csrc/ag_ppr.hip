// ag_ppr.hip -- personalised PageRank pull of up to 64 columns.
//
// The plain iteration of pageRank.c:942-1109 applied to up to 64 rank vectors at once, each with
// its own restart vector. Contributions are stored vertex-major, W = 16, 32 or 64 per vertex, so
// an in-edge gathers one contiguous run (128 bytes in BF16/FP16 and 256 in FP32 for 64 columns): a
// group of W / 4 lanes (four columns per lane, 8-byte or 16-byte loads) reads it with one
// coalesced load, and a group keeps the lines of 16 in-edges in flight at once, their source ids
// fetched by coalesced loads and passed lane to lane. Work items reuse the pull plan's bins:
// THREAD and GROUP16 rows take one group each, WAVE rows a wavefront, BLOCK rows a whole
// workgroup, HUB rows fixed segments whose partials a one-workgroup finish kernel adds in segment
// order. The per-column L1 delta is reduced in FP64 in a fixed order; the run stops when every
// column is below the tolerance. A run of iterations is captured once per column width into a
// hipGraph and replayed until the solve stops.
#include <stdlib.h>
#include <string.h>
#include <time.h>

#include "ag_internal.h"
#include "ag_pull_kernel.h"

#define PPR_W 64          // most columns per vertex
#define PPR_CH 16         // in-edges of a chunk: their contribution lines are in flight together
#define PPR_REPLAY 16u    // iterations of the captured graph

namespace {

// Run options read by the kernels from device memory, so one captured solve serves any
// seeds, column count, storage and stop rule.
struct PprConf {
    uint32_t seed[PPR_W];     // device row of each column's seed, AG_PPR_UNIFORM = uniform
    // FP16 storage holds contribution * 2^-f16_bias (the sum is multiplied back by 2^f16_bias,
    // exactly): every scaled rank, so every contribution, is at most N, and N * 2^-f16_bias
    // stays below FP16's largest finite value
    int32_t f16_bias;
    uint32_t k;
    uint32_t storage;         // AG_STORE_*
    uint32_t stop_rule;
    uint32_t pad;
    double l1_tol, refine_l1;
};

struct PprArgs {
    const void *c16[2];       // 16-bit contributions [N][W] (bf16 or fp16 bits)
    const float *c32[2];      // f32 contributions [N][W]
    float *rank;              // [N][W]
    const uint32_t *outdeg;
    const PprConf *conf;
    float *hub_part;          // [n_segs][W]
    double *part;             // [grid][W] per-workgroup column error partials
    double *colerr;           // [64] last column errors
    double *hist;             // [max_iterations] max column error per iteration
    PrState *st;
    uint32_t nparts;
    uint32_t n;
    float base, damp, basen;
    double dn;
};

struct Mode {
    bool r16, w16, f16;
    uint32_t rd, wr;
};

__device__ __forceinline__ Mode ppr_mode(const PprArgs &A, uint32_t storage, uint32_t iter)
{
    Mode m;
    m.rd = iter & 1u;
    m.wr = m.rd ^ 1u;
    m.f16 = storage == AG_STORE_F16;
    if (storage == AG_STORE_F32) {
        m.r16 = m.w16 = false;
        return m;
    }
    const int32_t ri = *(volatile const int32_t *)&A.st->refine_iter;
    m.w16 = !(ri >= 0 && (int32_t)iter >= ri);
    m.r16 = !(ri >= 0 && (int32_t)iter >= ri + 1);
    return m;
}

__device__ __forceinline__ float2 unpack16(uint32_t v, bool f16)
{
    if (f16) {
        _Float16 lo = __builtin_bit_cast(_Float16, (uint16_t)(v & 0xFFFFu));
        _Float16 hi = __builtin_bit_cast(_Float16, (uint16_t)(v >> 16));
        return make_float2((float)lo, (float)hi);
    }
    return make_float2(__uint_as_float(v << 16), __uint_as_float(v & 0xFFFF0000u));
}

__device__ __forceinline__ uint32_t to_bf16(float x)
{
    uint32_t u = __float_as_uint(x);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return u >> 16;
}

__device__ __forceinline__ uint32_t pack16(float x, float y, bool f16)
{
    if (f16) {
        const uint16_t a = __builtin_bit_cast(uint16_t, (_Float16)x);
        const uint16_t b = __builtin_bit_cast(uint16_t, (_Float16)y);
        return (uint32_t)a | ((uint32_t)b << 16);
    }
    return to_bf16(x) | (to_bf16(y) << 16);
}

__device__ __forceinline__ void add4(float4 &a, const float4 &b)
{
    a.x += b.x;
    a.y += b.y;
    a.z += b.z;
    a.w += b.w;
}

// The kernels are built for W = 16, 32 and 64 columns per vertex, the least that holds the call's
// columns: a group of W / 4 lanes (four columns each) owns a row, so a wavefront carries 16, 8 or 4
// rows and gathers 32-, 64- or 128-byte lines (twice that in FP32). A call of few columns paid for
// all 64 before: one column on RMAT-18 12.1 -> 4.8 ms a solve, RMAT-20 46 -> 14.5 ms (BF16), 32
// columns 15.3 -> 7.6 and 60 -> 27 ms.
template <uint32_t W>
struct Ppr {
    static constexpr uint32_t GL = W / 4u;                 // lanes per group
    static constexpr uint32_t NG = AG_WG / GL;             // groups per workgroup
    static constexpr uint32_t FG = AG_FIN_WG / GL;         // groups of the finish workgroup
    static constexpr uint32_t NI = PPR_CH / GL;            // a lane's source ids of a chunk
    struct Ids {
        uint32_t v[NI];
    };
};

// This lane's source ids of the 16-edge chunk at `base` of in-edges below hi (0 past hi): edge
// u * GL + q of the chunk is lane q's u-th.
template <uint32_t W>
__device__ __forceinline__ typename Ppr<W>::Ids ppr_ids(const PullGeom &G, uint32_t base,
                                                        uint32_t hi, uint32_t q)
{
    typename Ppr<W>::Ids s;
#pragma unroll
    for (uint32_t u = 0; u < Ppr<W>::NI; u++) {
        const uint32_t j = base + u * Ppr<W>::GL + q;
        s.v[u] = base < hi && j < hi ? __builtin_nontemporal_load(&G.src[j]) : 0u;
    }
    return s;
}

// Sum of columns 4q..4q+3 over the in-edges [lo, hi) owned by group gi of the ng groups that
// share the row: the edges are cut into 16-edge chunks, chunk c belongs to group c % ng. A
// chunk's source ids arrive in coalesced loads (`sl` holds the first chunk's, loaded by the
// caller) and are passed lane to lane, so every contribution line of the chunk is in flight at
// once: 16 loads of 8 bytes per lane (16-bit storage) or two rounds of 8 loads of 16 bytes
// (FP32); the next chunk's ids are loaded before them. Per lane the terms are added in edge
// order into two accumulators (even and odd edges), combined at the end.
template <uint32_t W>
__device__ __forceinline__ float4 ppr_group_sum(const PullGeom &G, const PprArgs &A,
                                                const Mode &m, uint32_t lo, uint32_t hi,
                                                uint32_t gi, uint32_t ng, uint32_t q,
                                                typename Ppr<W>::Ids sl)
{
    constexpr uint32_t GL = Ppr<W>::GL;
    float4 a0 = make_float4(0.f, 0.f, 0.f, 0.f), a1 = a0;
    const uint2 *c16 = (const uint2 *)A.c16[m.rd];
    const float4 *c32 = (const float4 *)A.c32[m.rd];
    const uint32_t stride = ng * PPR_CH;
    for (uint32_t base = lo + gi * PPR_CH; base < hi; base += stride) {
        const uint32_t cnt = hi - base < PPR_CH ? hi - base : PPR_CH;
        const typename Ppr<W>::Ids next = ppr_ids<W>(G, base + stride, hi, q);
        if (m.r16) {
            uint2 v[PPR_CH];
#pragma unroll
            for (uint32_t t = 0; t < PPR_CH; t++) {
                const uint32_t sv = (uint32_t)__shfl((int)sl.v[t / GL], (int)(t % GL), (int)GL);
                v[t] = t < cnt ? c16[(size_t)sv * GL + q] : make_uint2(0u, 0u);
            }
            // one branch a chunk: the format chosen per value took RMAT-18 181 us an iteration
            // in BF16 (64 columns), against 148
            const auto add = [&](auto f16) {
#pragma unroll
                for (uint32_t t = 0; t < PPR_CH; t++) {
                    const float2 lo2 = unpack16(v[t].x, f16), hi2 = unpack16(v[t].y, f16);
                    add4((t & 1u) ? a1 : a0, make_float4(lo2.x, lo2.y, hi2.x, hi2.y));
                }
            };
            if (m.f16)
                add(std::true_type());
            else
                add(std::false_type());
        } else {
#pragma unroll
            for (uint32_t h = 0; h < PPR_CH; h += PPR_CH / 2) {
                float4 v[PPR_CH / 2];
#pragma unroll
                for (uint32_t t = 0; t < PPR_CH / 2; t++) {
                    const uint32_t sv = (uint32_t)__shfl((int)sl.v[(h + t) / GL],
                                                         (int)((h + t) % GL), (int)GL);
                    v[t] = h + t < cnt ? c32[(size_t)sv * GL + q]
                                       : make_float4(0.f, 0.f, 0.f, 0.f);
                }
#pragma unroll
                for (uint32_t t = 0; t < PPR_CH / 2; t++)
                    add4((t & 1u) ? a1 : a0, v[t]);
            }
        }
        sl = next;
    }
    add4(a0, a1);
    return a0;
}

// Damping update of columns 4q..4q+3 of row v; each column's |delta| / N is accumulated in
// err (FP64), the next contribution rank / out_degree stored in 16 bits or FP32.
template <uint32_t W>
__device__ __forceinline__ void ppr_finish(const PprArgs &A, const Mode &m, uint32_t v,
                                           uint32_t q, float4 sum, const uint32_t *seed,
                                           double *err)
{
    float sums[4] = {sum.x, sum.y, sum.z, sum.w};
    if (m.r16 && m.f16) {   // FP16 terms were stored scaled by 2^-bias: exact power-of-two undo
#pragma unroll
        for (int c = 0; c < 4; c++)
            sums[c] = ldexpf(sums[c], A.conf->f16_bias);
    }
    float nw[4];
#pragma unroll
    for (int c = 0; c < 4; c++) {
        const float p = seed[c] == AG_PPR_UNIFORM ? A.base : (seed[c] == v ? A.basen : 0.0f);
        nw[c] = __fadd_rn(p, __fmul_rn(A.damp, sums[c]));
    }
    float4 *rk = (float4 *)(A.rank + (size_t)v * W) + q;
    const float4 old = *rk;
    *rk = make_float4(nw[0], nw[1], nw[2], nw[3]);
    const float olds[4] = {old.x, old.y, old.z, old.w};
#pragma unroll
    for (int c = 0; c < 4; c++)
        err[c] += __ddiv_rn((double)fabsf(__fsub_rn(nw[c], olds[c])), A.dn);
    const uint32_t od = A.outdeg[v];
    const float inv = od ? __uint2float_rn(od) : 1.0f;
    float qv[4];
#pragma unroll
    for (int c = 0; c < 4; c++)
        qv[c] = od ? __fdiv_rn(nw[c], inv) : 0.0f;
    if (m.w16) {
        if (m.f16) {
#pragma unroll
            for (int c = 0; c < 4; c++)
                qv[c] = ldexpf(qv[c], -A.conf->f16_bias);
        }
        ((uint2 *)A.c16[m.wr])[(size_t)v * (W / 4u) + q] =
            make_uint2(pack16(qv[0], qv[1], m.f16), pack16(qv[2], qv[3], m.f16));
    }
    else
        ((float4 *)A.c32[m.wr])[(size_t)v * (W / 4u) + q] = make_float4(qv[0], qv[1], qv[2], qv[3]);
}

// Column errors of one workgroup of NG groups: s_err[group][W] summed over groups in order.
template <uint32_t W, uint32_t NG>
__device__ __forceinline__ void ppr_column_errors(const double *err, double *s_err, double *out)
{
    const uint32_t tid = threadIdx.x, q = tid % (W / 4u), gi = tid / (W / 4u);
#pragma unroll
    for (int c = 0; c < 4; c++)
        s_err[gi * W + 4 * q + c] = err[c];
    __syncthreads();
    if (tid < W) {
        double t = 0.0;
        for (uint32_t w = 0; w < NG; w++)
            t += s_err[w * W + tid];
        out[tid] = t;
    }
    __syncthreads();
}

// One iteration's gather and update. Work items, heaviest first: hub segments and BLOCK rows
// (every group of the workgroup on one row; partials combined in LDS in group order), WAVE rows
// (the groups of a wavefront on one row; combined by lane exchanges), THREAD and GROUP16 rows
// (one group per row).
template <uint32_t W>
__global__ __launch_bounds__(AG_WG, 4) void ppr_kernel(PullGeom G, PprArgs A)
{
    constexpr uint32_t GL = Ppr<W>::GL, NG = Ppr<W>::NG;
    __shared__ float4 s_red[NG * GL];
    __shared__ double s_err[NG * W];
    __shared__ double s_tot[W];
    if (*(volatile const uint32_t *)&A.st->done)
        return;
    const uint32_t iter = *(volatile const uint32_t *)&A.st->iter;
    const Mode m = ppr_mode(A, A.conf->storage, iter);
    const uint32_t tid = threadIdx.x, q = tid % GL, gi = tid / GL;
    const uint32_t wl = (tid % AG_WAVE) / GL;   // group inside its wavefront
    uint32_t seed[4];
#pragma unroll
    for (int c = 0; c < 4; c++)
        seed[c] = A.conf->seed[4 * q + c];
    double err[4] = {0.0, 0.0, 0.0, 0.0};
    const uint32_t lite_rows = G.bin_row[AG_BIN_WAVE];    // THREAD + GROUP16 rows
    const uint32_t wave0 = G.bin_row[AG_BIN_WAVE], wave1 = G.bin_row[AG_BIN_WAVE + 1];
    const uint32_t nwave = (wave1 - wave0 + AG_WG / AG_WAVE - 1) / (AG_WG / AG_WAVE);
    const uint32_t nlite = (lite_rows + NG - 1) / NG;
    const uint32_t nblock = G.bin_row[AG_BIN_BLOCK + 1] - G.bin_row[AG_BIN_BLOCK];
    const uint32_t nseg = G.slot_blk0[1] - G.slot_blk0[0];
    const uint32_t heavy = nseg + nblock;
    const uint32_t total = heavy + nwave + nlite;
    const uint32_t lite0 = heavy + nwave;
    uint32_t it = blockIdx.x;
    for (; it < lite0; it += gridDim.x) {
        if (it < heavy) {
            uint32_t lo, hi, row = 0;
            const bool hub = it < nseg;
            if (hub) {
                lo = G.seg_lo[it];
                hi = G.seg_hi[it];
            } else {
                row = G.bin_row[AG_BIN_BLOCK] + (it - nseg);
                lo = G.off[row];
                hi = G.off[row + 1];
            }
            s_red[gi * GL + q] = ppr_group_sum<W>(G, A, m, lo, hi, gi, NG, q,
                                                   ppr_ids<W>(G, lo + gi * PPR_CH, hi, q));
            __syncthreads();
            if (gi == 0) {
                float4 t = s_red[q];
                for (uint32_t w = 1; w < NG; w++)
                    add4(t, s_red[w * GL + q]);
                if (hub)
                    ((float4 *)(A.hub_part + (size_t)it * W))[q] = t;
                else
                    ppr_finish<W>(A, m, row, q, t, seed, err);
            }
            __syncthreads();
        } else if (it < heavy + nwave) {
            const uint32_t row = wave0 + (it - heavy) * (AG_WG / AG_WAVE) + tid / AG_WAVE;
            const bool valid = row < wave1;
            float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
            if (valid) {
                const uint32_t lo = G.off[row], hi = G.off[row + 1];
                a = ppr_group_sum<W>(G, A, m, lo, hi, wl, AG_WAVE / GL, q,
                                  ppr_ids<W>(G, lo + wl * PPR_CH, hi, q));
            }
            // (g0 + g1) + (g2 + g3), the same value in every group (addition commutes)
#pragma unroll
            for (int msk = GL; msk < AG_WAVE; msk <<= 1) {
                a.x += __shfl_xor(a.x, msk, AG_WAVE);
                a.y += __shfl_xor(a.y, msk, AG_WAVE);
                a.z += __shfl_xor(a.z, msk, AG_WAVE);
                a.w += __shfl_xor(a.w, msk, AG_WAVE);
            }
            if (valid && wl == 0)
                ppr_finish<W>(A, m, row, q, a, seed, err);
        }
    }
    // THREAD and GROUP16 rows, a group each, two rows ahead: while row k is gathered, the
    // first source ids of row k + 1 and the offsets of row k + 2 are in flight
    {
        const uint32_t step = gridDim.x * NG;
        uint32_t row = it < total ? (it - lite0) * NG + gi : lite_rows;
        uint32_t lo = 0, hi = 0, lo1 = 0, hi1 = 0;
        typename Ppr<W>::Ids sl{};
        if (row < lite_rows) {
            lo = G.off[row];
            hi = G.off[row + 1];
            sl = ppr_ids<W>(G, lo, hi, q);
        }
        if (row < lite_rows && row + step < lite_rows) {
            lo1 = G.off[row + step];
            hi1 = G.off[row + step + 1];
        }
        for (; row < lite_rows; row += step) {
            uint32_t lo2 = 0, hi2 = 0;
            if (row + 2 * step < lite_rows) {
                lo2 = G.off[row + 2 * step];
                hi2 = G.off[row + 2 * step + 1];
            }
            const typename Ppr<W>::Ids sl1 = ppr_ids<W>(G, lo1, hi1, q);
            const float4 a = ppr_group_sum<W>(G, A, m, lo, hi, 0, 1, q, sl);
            ppr_finish<W>(A, m, row, q, a, seed, err);
            lo = lo1;
            hi = hi1;
            sl = sl1;
            lo1 = lo2;
            hi1 = hi2;
        }
    }
    ppr_column_errors<W, NG>(err, s_err, s_tot);
    if (tid < W)
        A.part[(size_t)blockIdx.x * W + tid] = s_tot[tid];
}

// Hub rows (their segment partials added in segment order), the column errors of the
// iteration (fixed order) and the stop / refinement decisions. One workgroup.
template <uint32_t W>
__global__ __launch_bounds__(AG_FIN_WG) void ppr_finish_kernel(PullGeom G, PprArgs A)
{
    constexpr uint32_t GL = Ppr<W>::GL, FG = Ppr<W>::FG;
    __shared__ double s_err[FG * W];
    __shared__ double s_tot[W];
    if (*(volatile const uint32_t *)&A.st->done)
        return;
    const PprConf &C = *A.conf;
    const uint32_t iter = *(volatile const uint32_t *)&A.st->iter;
    const Mode m = ppr_mode(A, C.storage, iter);
    const uint32_t tid = threadIdx.x, q = tid % GL, gi = tid / GL;
    uint32_t seed[4];
#pragma unroll
    for (int c = 0; c < 4; c++)
        seed[c] = C.seed[4 * q + c];
    double err[4] = {0.0, 0.0, 0.0, 0.0};
    for (uint32_t hub = gi; hub < G.n_hubs; hub += FG) {
        const uint32_t s0 = G.hub_seg0[hub], s1 = G.hub_seg0[hub + 1];
        float4 t = ((const float4 *)(A.hub_part + (size_t)s0 * W))[q];
        for (uint32_t sg = s0 + 1; sg < s1; sg++)
            add4(t, ((const float4 *)(A.hub_part + (size_t)sg * W))[q]);
        ppr_finish<W>(A, m, G.bin_row[AG_BIN_HUB] + hub, q, t, seed, err);
    }
    ppr_column_errors<W, FG>(err, s_err, s_tot);
    // the iteration kernel's per-workgroup column errors: lane (chunk j, column c) adds the
    // workgroups of chunk j in order (32 loads in flight; 8
    // left this launch at 21 us with 2048 workgroups), then each column adds its hub term
    // and the chunks in chunk order -- a fixed order for any grid
    {
        constexpr uint32_t NCH = AG_FIN_WG / W, U = 32;
        const uint32_t c = tid % W, j = tid / W;
        const uint32_t len = (A.nparts + NCH - 1) / NCH;
        const uint32_t b0 = j * len, b1 = b0 + len < A.nparts ? b0 + len : A.nparts;
        double t = 0.0;
        for (uint32_t b = b0; b < b1; b += U) {
            double v[U];
#pragma unroll
            for (uint32_t u = 0; u < U; u++)
                v[u] = b + u < b1 ? A.part[(size_t)(b + u) * W + c] : 0.0;
#pragma unroll
            for (uint32_t u = 0; u < U; u++)
                t += v[u];
        }
        s_err[j * W + c] = t;   // s_err is free again (ppr_column_errors ends synced)
        __syncthreads();
        if (tid < W) {
            double tot = s_tot[tid];
            for (uint32_t q2 = 0; q2 < NCH; q2++)
                tot += s_err[q2 * W + tid];
            s_tot[tid] = tot;
        }
        __syncthreads();
    }
    if (tid != 0)
        return;
    double E = 0.0;
    bool finite = true;
    for (uint32_t c = 0; c < C.k; c++) {
        A.colerr[c] = s_tot[c];
        E = s_tot[c] > E ? s_tot[c] : E;
        finite = finite && isfinite(s_tot[c]);
    }
    if (!finite)   // a column that overflowed never satisfies the stop rule
        E = INFINITY;
    PrState *st = A.st;
    A.hist[iter] = E;
    bool can_stop = true;
    if (C.storage != AG_STORE_F32) {
        const int32_t ri = st->refine_iter;
        if (ri < 0) {
            refine_decide(*st, iter, E, C.refine_l1);
            can_stop = false;
        } else {
            can_stop = (int32_t)iter >= ri + 1;
        }
    }
    if (can_stop && C.stop_rule == AG_STOP_L1 && E <= C.l1_tol) {
        st->done = 1;
        st->stop_iter = iter;
    }
    st->last_err = E;
    st->iter = iter + 1;
}

// Start of a solve: every rank 1.0, contributions 1 / out_degree (0 for sinks) in the storage
// of the first iteration, and the iteration state reset (thread 0; no other thread reads it
// in this launch).
template <uint32_t W>
__global__ void ppr_init_kernel(PprArgs A)
{
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;  // (vertex, lane)
    if (i == 0) {
        PrState *st = A.st;
        st->iter = 0;
        st->done = 0;
        st->stop_iter = 0;
        st->refine_iter = -1;
        st->last_active = 0;
        st->last_err = 0.0;
        st->best_err = 0.0;
        st->stall = 0;
    }
    if (i >= (uint64_t)A.n * (W / 4u))
        return;
    const uint32_t v = (uint32_t)(i / (W / 4u));
    ((float4 *)A.rank)[i] = make_float4(1.0f, 1.0f, 1.0f, 1.0f);
    const uint32_t od = A.outdeg[v];
    const float c = od ? __fdiv_rn(1.0f, __uint2float_rn(od)) : 0.0f;
    const uint32_t storage = A.conf->storage;
    if (storage == AG_STORE_F32) {
        ((float4 *)A.c32[0])[i] = make_float4(c, c, c, c);
    } else {
        const bool f16 = storage == AG_STORE_F16;
        const float cs = f16 ? ldexpf(c, -A.conf->f16_bias) : c;
        const uint32_t p = pack16(cs, cs, f16);
        ((uint2 *)A.c16[0])[i] = make_uint2(p, p);
    }
}

__global__ void ppr_out_kernel(uint32_t n, uint32_t k, uint32_t W, const float *rank, const uint32_t *d2o,
                               float nf, float *out)
{
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (uint64_t)n * k)
        return;
    const uint32_t v = (uint32_t)(i / k), c = (uint32_t)(i % k);
    out[(size_t)d2o[v] * k + c] = __fdiv_rn(rank[(size_t)v * W + c], nf);
}

} // namespace

// Per-graph PPR workspace, kept between calls (the captured solve holds its pointers).
struct ag_ppr_ws {
    uint32_t n, grid_max, hist_cap;
    uint32_t grid;             // workgroups of this call's iteration kernel (<= grid_max)
    void *c16[2];
    float *c32[2];
    float *rank;
    float *hub_part;
    double *part, *colerr, *hist;
    PrState *st;
    PprConf *conf;
    PrState *st_host;          // pinned [2]
    PprConf *conf_host;        // pinned
    uint32_t *o2d;             // [n] host: device row of every vertex
    // the captured iterations of each column width, kept so that calls of different widths can
    // take turns
    struct {
        hipGraph_t graph;
        hipGraphExec_t exec;
        uint32_t grid;         // its iteration-kernel grid
    } cap[3];
    uint32_t width;            // columns per vertex of this call: 16, 32 or 64
    hipEvent_t ev[2];          // the state copies after the last two replays
};

static void ppr_drop_capture(ag_ppr_ws *w, uint32_t i)
{
    if (w->cap[i].exec)
        (void)hipGraphExecDestroy(w->cap[i].exec);
    if (w->cap[i].graph)
        (void)hipGraphDestroy(w->cap[i].graph);
    w->cap[i].exec = NULL;
    w->cap[i].graph = NULL;
}

void ag_ppr_free_ws(ag_dgraph *g)
{
    ag_ppr_ws *w = g->ppr;
    if (!w)
        return;
    (void)hipStreamSynchronize(g->dev->stream);
    for (uint32_t i = 0; i < 3u; i++)
        ppr_drop_capture(w, i);
    void *ptrs[] = {w->c16[0], w->c16[1], w->c32[0], w->c32[1], w->rank, w->hub_part, w->part,
                    w->colerr, w->hist, w->st, w->conf};
    for (void *p : ptrs)
        if (p)
            (void)hipFree(p);
    if (w->st_host)
        (void)hipHostFree(w->st_host);
    if (w->conf_host)
        (void)hipHostFree(w->conf_host);
    for (hipEvent_t ev : w->ev)
        if (ev)
            (void)hipEventDestroy(ev);
    free(w->o2d);
    free(w);
    g->ppr = NULL;
}

static int ppr_allocate(ag_dgraph *g, ag_ppr_ws *w)
{
    w->o2d = (uint32_t *)malloc((size_t)g->n * sizeof(uint32_t));
    if (!w->o2d)
        return ag_set_error(AG_ERR_OOM, "host allocation failed");
    w->n = g->n;
    for (uint32_t r = 0; r < g->n; r++)
        w->o2d[g->h_d2o[r]] = r;
    // 16-lane groups with up to 16 contribution lines in flight per lane: as many
    // workgroups per CU as fit, up to 8
    w->grid_max = ag_pull_grid(g, AG_WG * 16u + AG_WG * 4u * 8u, 8u);
    if (w->grid_max == 0)
        w->grid_max = 1;
    w->grid = w->grid_max;
    const size_t nv = (size_t)g->n * PPR_W;
    AG_HIP(ag_dev_malloc(g->dev, &w->rank, nv * sizeof(float)));
    AG_HIP(ag_dev_malloc(g->dev, &w->c32[0], nv * sizeof(float)));
    AG_HIP(ag_dev_malloc(g->dev, &w->c32[1], nv * sizeof(float)));
    AG_HIP(ag_dev_malloc(g->dev, &w->c16[0], nv * 2));
    AG_HIP(ag_dev_malloc(g->dev, &w->c16[1], nv * 2));
    AG_HIP(ag_dev_malloc(g->dev, &w->hub_part,
                     (size_t)(g->n_segs ? g->n_segs : 1) * PPR_W * sizeof(float)));
    AG_HIP(ag_dev_malloc(g->dev, &w->part, (size_t)w->grid_max * PPR_W * sizeof(double)));
    AG_HIP(ag_dev_malloc(g->dev, &w->colerr, PPR_W * sizeof(double)));
    AG_HIP(ag_dev_malloc(g->dev, &w->st, sizeof(PrState)));
    AG_HIP(ag_dev_malloc(g->dev, &w->conf, sizeof(PprConf)));
    AG_HIP(hipHostMalloc((void **)&w->st_host, 2 * sizeof(PrState), hipHostMallocDefault));
    for (hipEvent_t &ev : w->ev)
        AG_HIP(hipEventCreateWithFlags(&ev, hipEventDisableTiming));
    AG_HIP(hipHostMalloc((void **)&w->conf_host, sizeof(PprConf), hipHostMallocDefault));
    return AG_OK;
}

// Allocates the workspace on first use (whole, or none); grows the history (dropping the captured
// iterations) when a call asks for more iterations than it holds.
static int ppr_workspace(ag_dgraph *g, uint32_t maxit, ag_ppr_ws **out)
{
    ag_ppr_ws *w = g->ppr;
    if (!w) {
        w = (ag_ppr_ws *)calloc(1, sizeof(ag_ppr_ws));
        if (!w)
            return ag_set_error(AG_ERR_OOM, "host allocation failed");
        g->ppr = w;
        const int st = ppr_allocate(g, w);
        if (st != AG_OK) {
            ag_ppr_free_ws(g);
            return st;
        }
    }
    if (w->hist_cap < maxit) {
        for (uint32_t i = 0; i < 3u; i++)
            ppr_drop_capture(w, i);
        if (w->hist)
            AG_HIP(hipFree(w->hist));
        w->hist = NULL;
        w->hist_cap = 0;
        const uint32_t cap = maxit > 512u ? maxit : 512u;
        AG_HIP(ag_dev_malloc(g->dev, &w->hist, (size_t)cap * sizeof(double)));
        w->hist_cap = cap;
    }
    *out = w;
    return AG_OK;
}

static PprArgs ppr_args(const ag_dgraph *g, const ag_ppr_ws *w)
{
    PprArgs A;
    memset(&A, 0, sizeof(A));
    A.c16[0] = w->c16[0];
    A.c16[1] = w->c16[1];
    A.c32[0] = w->c32[0];
    A.c32[1] = w->c32[1];
    A.rank = w->rank;
    A.outdeg = g->outdeg;
    A.conf = w->conf;
    A.hub_part = w->hub_part;
    A.part = w->part;
    A.colerr = w->colerr;
    A.hist = w->hist;
    A.st = w->st;
    A.nparts = w->grid;
    A.n = g->n;
    A.damp = 0.85f;
    volatile float d = 0.85f;
    A.base = 1.0f - d;
    A.basen = A.base * (float)g->n;
    A.dn = (double)g->n;
    return A;
}

static hipError_t ppr_enqueue_init(const ag_dgraph *g, const ag_ppr_ws *w, const PprArgs &A,
                                   hipStream_t s)
{
    const uint32_t blocks = (uint32_t)(((uint64_t)g->n * (w->width / 4u) + 255u) / 256u);
    switch (w->width) {
    case 16: ppr_init_kernel<16><<<blocks, 256, 0, s>>>(A); break;
    case 32: ppr_init_kernel<32><<<blocks, 256, 0, s>>>(A); break;
    default: ppr_init_kernel<64><<<blocks, 256, 0, s>>>(A); break;
    }
    return hipGetLastError();
}

static hipError_t ppr_enqueue_iterations(const ag_dgraph *g, const ag_ppr_ws *w,
                                         const PprArgs &A, uint32_t count, hipStream_t s)
{
    const PullGeom G = ag_make_geom(g);
    for (uint32_t i = 0; i < count; i++) {
        switch (w->width) {
        case 16:
            ppr_kernel<16><<<w->grid, AG_WG, 0, s>>>(G, A);
            ppr_finish_kernel<16><<<1, AG_FIN_WG, 0, s>>>(G, A);
            break;
        case 32:
            ppr_kernel<32><<<w->grid, AG_WG, 0, s>>>(G, A);
            ppr_finish_kernel<32><<<1, AG_FIN_WG, 0, s>>>(G, A);
            break;
        default:
            ppr_kernel<64><<<w->grid, AG_WG, 0, s>>>(G, A);
            ppr_finish_kernel<64><<<1, AG_FIN_WG, 0, s>>>(G, A);
            break;
        }
    }
    return hipGetLastError();
}

extern "C" void ag_ppr_options_default(ag_ppr_options *o)
{
    memset(o, 0, sizeof(*o));
    o->max_iterations = 100;
    o->stop_rule = AG_STOP_L1;
    o->l1_tolerance = 1e-6;
    o->storage = AG_STORE_BF16;
    o->refine_l1 = 1e-3;
    o->chunk = 0;
    o->use_hip_graph = 1;
}

// A solve is: the init launch, then up to max_iterations x (gather/update, finish); the finish
// launch of the stopping iteration sets a device flag that turns every later launch into a
// no-op. With use_hip_graph, PPR_REPLAY iterations are captured once per graph, width and grid
// and replayed until a replay ends stopped (capturing all max_iterations paid for the no-op
// launches past the stop: 230 of 300 iterations on RMAT-18, 1 of 15 ms); otherwise, and where
// max_iterations is less, the iterations are queued eagerly, `chunk` between polls of the flag.
extern "C" int ag_ppr_pull(ag_dgraph *g, uint32_t k, const uint32_t *seeds,
                           const ag_ppr_options *opts, float *ranks_out, double *col_error,
                           ag_ppr_result *res)
{
    if (!g || k == 0 || k > AG_PPR_MAX_COLS || !seeds || (g->n && !ranks_out) || !res)
        return ag_set_error(AG_ERR_INVALID, "bad argument (k must be in [1, 64])");
    ag_ppr_options o;
    if (opts)
        o = *opts;
    else
        ag_ppr_options_default(&o);
    if (o.stop_rule != AG_STOP_L1 && o.stop_rule != AG_STOP_NONE)
        return ag_set_error(AG_ERR_INVALID, "PPR supports AG_STOP_L1 and AG_STOP_NONE");
    if (o.storage > AG_STORE_F16)
        return ag_set_error(AG_ERR_INVALID, "unknown storage %u", o.storage);
    const uint32_t n = g->n;
    for (uint32_t c = 0; c < k; c++) {
        if (seeds[c] != AG_PPR_UNIFORM && seeds[c] >= n)
            return ag_set_error(AG_ERR_INVALID, "seed %u of column %u out of range", seeds[c], c);
    }
    memset(res, 0, sizeof(*res));
    res->refine_iteration = -1;
    if (n == 0)
        return AG_OK;
    AG_HIP(hipSetDevice(g->dev->ordinal));
    hipStream_t s = g->dev->stream;
    const uint32_t maxit = o.max_iterations ? o.max_iterations : 1;
    ag_ppr_ws *w = NULL;
    int st = ppr_workspace(g, maxit, &w);
    if (st != AG_OK)
        return st;
    st = ag_wait_stream(g->dev);   // the pinned option / state buffers may still feed a copy
    if (st != AG_OK)
        return st;
    // seed vertex -> device row; unused columns run as uniform restarts and are not reported
    PprConf *conf = w->conf_host;
    memset(conf, 0, sizeof(*conf));
    for (uint32_t c = 0; c < PPR_W; c++)
        conf->seed[c] = AG_PPR_UNIFORM;
    for (uint32_t c = 0; c < k; c++)
        if (seeds[c] != AG_PPR_UNIFORM)
            conf->seed[c] = w->o2d[seeds[c]];
    conf->k = k;
    {
        // every scaled rank is at most N (the mass of a column never exceeds N), so a
        // contribution times 2^-bias stays at most 2^15, inside FP16's range
        int32_t bits = 0;
        while (bits < 32 && (1ull << bits) < (uint64_t)n)
            bits++;
        conf->f16_bias = bits > 15 ? bits - 15 : 0;
    }
    conf->storage = o.storage;
    conf->stop_rule = o.stop_rule;
    conf->l1_tol = o.l1_tolerance;
    conf->refine_l1 = o.refine_l1;
    AG_HIP(hipMemcpyAsync(w->conf, conf, sizeof(PprConf), hipMemcpyHostToDevice, s));
    {
        uint32_t grid = w->grid_max;
        if (o.wg_per_cu) {
            const uint64_t want = (uint64_t)g->dev->num_cus * o.wg_per_cu;
            grid = want < grid ? (uint32_t)want : grid;
        }
        w->grid = grid ? grid : 1u;
    }
    w->width = k <= 16u ? 16u : k <= 32u ? 32u : 64u;
    const PprArgs A = ppr_args(g, w);
    hipEvent_t e0 = NULL, e1 = NULL;
    hipError_t e = hipEventCreate(&e0);
    if (e == hipSuccess)
        e = hipEventCreate(&e1);
    if (e == hipSuccess)
        e = hipEventRecord(e0, s);
    if (e == hipSuccess && o.use_hip_graph && maxit >= PPR_REPLAY) {
        const uint32_t ci = w->width == 16u ? 0u : w->width == 32u ? 1u : 2u;
        auto &cap = w->cap[ci];
        if (cap.exec && cap.grid != w->grid)
            ppr_drop_capture(w, ci);
        if (!cap.exec) {
            e = hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal);
            if (e == hipSuccess) {
                const hipError_t qe = ppr_enqueue_iterations(g, w, A, PPR_REPLAY, s);
                const hipError_t ce = hipStreamEndCapture(s, &cap.graph);
                e = qe != hipSuccess ? qe : ce;
            }
            if (e == hipSuccess)
                e = hipGraphInstantiate(&cap.exec, cap.graph, NULL, NULL, 0);
            if (e == hipSuccess)
                cap.grid = w->grid;
            else
                ppr_drop_capture(w, ci);
        }
        if (e == hipSuccess)
            e = ppr_enqueue_init(g, w, A, s);
        // replays, each followed by a copy of the state; the copy before the last is read while
        // the last replay runs, so the device never waits for the host
        bool stopped = false;
        uint32_t done = 0;
        for (uint32_t r = 0; e == hipSuccess && st == AG_OK && !stopped && done < maxit; r++) {
            const uint32_t left = maxit - done;
            if (left >= PPR_REPLAY)
                e = hipGraphLaunch(cap.exec, s);
            else
                e = ppr_enqueue_iterations(g, w, A, left, s);
            done += left < PPR_REPLAY ? left : PPR_REPLAY;
            if (e == hipSuccess)
                e = hipMemcpyAsync(&w->st_host[r & 1u], w->st, sizeof(PrState),
                                   hipMemcpyDeviceToHost, s);
            if (e == hipSuccess)
                e = hipEventRecord(w->ev[r & 1u], s);
            if (e == hipSuccess && r > 0) {
                st = ag_wait_event(g->dev, w->ev[(r & 1u) ^ 1u]);
                stopped = st == AG_OK && w->st_host[(r & 1u) ^ 1u].done;
            }
        }
        if (e == hipSuccess && st == AG_OK)
            e = hipEventRecord(e1, s);
        if (e == hipSuccess && st == AG_OK)
            e = hipMemcpyAsync(w->st_host, w->st, sizeof(PrState), hipMemcpyDeviceToHost, s);
        if (e != hipSuccess)
            st = ag_hip_fail(e, "PPR graph launch", __FILE__, __LINE__);
        else if (st == AG_OK)
            st = ag_wait_stream(g->dev);
    } else if (e == hipSuccess) {
        e = ppr_enqueue_init(g, w, A, s);
        const uint32_t chunk = o.chunk ? o.chunk : 8;
        uint32_t enq = 0;
        while (e == hipSuccess && st == AG_OK && enq < maxit) {
            const uint32_t kk = maxit - enq < chunk ? maxit - enq : chunk;
            e = ppr_enqueue_iterations(g, w, A, kk, s);
            enq += kk;
            if (e == hipSuccess)
                e = hipEventRecord(e1, s);
            if (e == hipSuccess)
                e = hipMemcpyAsync(w->st_host, w->st, sizeof(PrState), hipMemcpyDeviceToHost, s);
            if (e == hipSuccess)
                st = ag_wait_stream(g->dev);
            if (st == AG_OK && e == hipSuccess && w->st_host->done)
                break;
        }
        if (e != hipSuccess)
            st = ag_hip_fail(e, "PPR launch", __FILE__, __LINE__);
    } else {
        st = ag_hip_fail(e, "PPR events", __FILE__, __LINE__);
    }
    if (st == AG_OK) {
        const PrState *sth = w->st_host;
        float ms = 0.0f;
        if (hipEventElapsedTime(&ms, e0, e1) != hipSuccess)
            ms = 0.0f;   // timing is informational; the ranks are already valid
        res->loop_ms = ms;
        res->iterations = sth->done ? sth->stop_iter : sth->iter;
        res->executed = sth->done ? sth->stop_iter + 1 : sth->iter;
        res->max_error = sth->last_err;
        res->refine_iteration = sth->refine_iter;
        // normalised ranks, original order; c32[1] is free as staging once the solve ended
        float *outd = w->c32[1];
        const uint64_t tot = (uint64_t)n * k;
        ppr_out_kernel<<<(uint32_t)((tot + 255) / 256), 256, 0, s>>>(n, k, w->width, w->rank, g->d2o,
                                                                     (float)n, outd);
        e = hipGetLastError();
        const size_t ob = tot * sizeof(float), eb = (size_t)k * sizeof(double);
        st = (e == hipSuccess) ? ag_copy_out(g->dev, ranks_out, outd, ob, ob)
                               : ag_hip_fail(e, "PPR output", __FILE__, __LINE__);
        if (st == AG_OK && col_error)
            st = ag_copy_out(g->dev, col_error, w->colerr, eb, eb);
    }
    if (e0)
        (void)hipEventDestroy(e0);
    if (e1)
        (void)hipEventDestroy(e1);
    return st;
}
