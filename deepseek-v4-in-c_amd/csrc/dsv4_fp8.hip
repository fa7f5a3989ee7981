/* SPDX-License-Identifier: Apache-2.0 */
/* dsv4_fp8.hip - block-scaled FP8 e4m3 GEMV for batch-1 decode on gfx950.
 *
 * What it computes is dsv4_matmul_fp8 (reference src/core/dsv4_matmul.c:
 * 293-318): y[o] = sum over 128-column blocks of (block dot) * scale(o/128,
 * c/128). It replaces the reference's k_mmq_fp8 (src/cuda/dsv4_cuda.cu:
 * 93-129), which gives each row a 128-thread block and reads one byte per
 * lane per step.
 *
 * APPROACH (bandwidth-bound: ~1 multiply-add per weight byte)
 *   - A row is split over TC threads ("row threads", a power of two up to
 *     64 or a multiple of 64 up to 256); thread j owns the 16-byte chunks
 *     j, j+TC, j+2TC, ... of every row it visits (NCH <= 4 of them), so rows
 *     up to 16384 columns take this path. Consecutive lanes read consecutive 16-byte chunks, so one wave
 *     instruction moves 1 KiB of one row -- fully coalesced.
 *   - The thread's slice of x (NCH x 16 floats) is loaded once into VGPRs and
 *     reused for every row the workgroup visits; workgroups are persistent
 *     over a contiguous range of row tiles, so x is fetched ~once per
 *     workgroup, not once per row.
 *   - A thread works on R rows at once: R*NCH independent 16-byte loads in
 *     flight per lane before any arithmetic.
 *   - Decode is v_cvt_pk_f32_fp8 (exact), 16 fp32 FMAs per chunk, then one
 *     FMA applies the chunk's block scale (each 16-column chunk lies in one
 *     128-column block), accumulating per lane in fp32.
 *   - The TC lane partials of a row are summed by a fixed DPP tree inside a
 *     wave and, when a row spans several waves, in wave order through LDS.
 *
 * DETERMINISM. TC, NCH and the reduction tree are functions of `cols` alone
 * (fp8_geom), so a row's result does not depend on R, the grid size or the
 * rows around it; the batched kernel reuses the same per-row arithmetic and
 * is bit-identical to the GEMV per (row, token).
 *
 * NUMERICS. fp32 inside the lane and in the tree (the reference CPU path
 * accumulates in double); measured against it under the vector-scaled
 * relative metric of tests/unit/test_cuda.c:160-167, bound 1e-5.
 */
#include "dsv4_dev.h"
#include "dsv4_internal.h"

#include <algorithm>
#include <stdlib.h>

namespace {

#include "dsv4_bf16_rows.h"
#include "dsv4_prep_rows.h"

struct Fp8Geom {
    int ch;   /* 16-byte chunks per row                       */
    int tc;   /* threads per row (power of two <= 64, or k*64) */
    int nch;  /* chunks per thread (<= 4)                      */
    int wg;   /* workgroup size                                */
    int rg;   /* rows in flight per workgroup per R            */
};

bool fp8_geom(int cols, Fp8Geom *g)
{
    if (cols <= 0 || (cols & 15)) return false;
    const int ch = cols >> 4;
    int tc, nch;
    if (ch <= 64) {
        tc = 1;
        while (tc < ch) tc <<= 1;
        nch = 1;
    } else {
        tc = 64 * ((ch + 255) / 256);
        nch = (ch + tc - 1) / tc;
    }
    if (tc > 256 || nch > 4) return false;     /* cols <= 16384 */
    g->ch = ch;
    g->tc = tc;
    g->nch = nch;
    g->wg = tc * (256 / tc);
    g->rg = g->wg / tc;
    return true;
}

/* A scale as it lies in memory, and its value. A load whose result is decoded
 * where it is needed and not where it is issued does not make the loads
 * issued before it be waited for there. */
template <int SF>
__device__ __forceinline__ uint32_t ld_scale_raw(const void *S, size_t at)
{
    if (SF == 0) return ((const uint8_t *)S)[at];
    return ((const uint32_t *)S)[at];
}
template <int SF>
__device__ __forceinline__ float scale_val(uint32_t raw)
{
    return SF == 0 ? dec_e8m0(raw) : __uint_as_float(raw);
}
template <int SF>
__device__ __forceinline__ float ld_scale(const void *S, size_t at)
{
    return scale_val<SF>(ld_scale_raw<SF>(S, at));
}

/* Dot of 16 decoded weights with 16 activations; 4 interleaved chains. */
/* The chunk's 16 products summed in four chains and a fixed tree, from
 * weights already decoded (dot16f) or from the packed codes (dot16). */
__device__ __forceinline__ float dot16f(const float *w, const float *xr)
{
    float p0 = w[0] * xr[0], p1 = w[1] * xr[1];
    float p2 = w[2] * xr[2], p3 = w[3] * xr[3];
#pragma unroll
    for (int e = 4; e < 16; e += 4) {
        p0 = fmaf(w[e + 0], xr[e + 0], p0);
        p1 = fmaf(w[e + 1], xr[e + 1], p1);
        p2 = fmaf(w[e + 2], xr[e + 2], p2);
        p3 = fmaf(w[e + 3], xr[e + 3], p3);
    }
    return (p0 + p1) + (p2 + p3);
}

__device__ __forceinline__ float dot16(const u32x4 v, const float *xr)
{
    float w[16];
    dec_e4m3x4(v.x, w + 0);
    dec_e4m3x4(v.y, w + 4);
    dec_e4m3x4(v.z, w + 8);
    dec_e4m3x4(v.w, w + 12);
    float p0 = w[0] * xr[0], p1 = w[1] * xr[1];
    float p2 = w[2] * xr[2], p3 = w[3] * xr[3];
#pragma unroll
    for (int e = 4; e < 16; e += 4) {
        p0 = fmaf(w[e + 0], xr[e + 0], p0);
        p1 = fmaf(w[e + 1], xr[e + 1], p1);
        p2 = fmaf(w[e + 2], xr[e + 2], p2);
        p3 = fmaf(w[e + 3], xr[e + 3], p3);
    }
    return (p0 + p1) + (p2 + p3);
}

/* Rows per workgroup are bounded by the LDS that holds the per-wave row
 * partials of rows wider than one wave (at most 4 waves per row). */
constexpr int PART_MAX = 4096;

/* Independent GEMVs of one width in one launch (blockIdx.y = group).
 * Strided: group i reads x + i*x, W + i*w bytes, its scales at S + i*s
 * bytes, and writes y + i*y. Listed (list > 0): group i is matrix Wl[i]
 * (rl[i] rows, scales Sl[i]) into yl[i], all reading the same x. One group
 * with zero strides is the plain GEMV. */
constexpr int FP8_LIST_MAX = 4;
struct Fp8Groups {
    int n = 1;
    long long x = 0, y = 0, w = 0, s = 0;
    int list = 0;
    bool valu = false;                  /* the VALU form even for E8M0 scales */
    const uint8_t *Wl[FP8_LIST_MAX] = {};
    const void *Sl[FP8_LIST_MAX] = {};
    float *yl[FP8_LIST_MAX] = {};
    int rl[FP8_LIST_MAX] = {};
};

/* One step's weights (R rows x NCH chunks) and the block scales of its row
 * block (the R rows of a step lie in one row block: the launcher picks R
 * dividing blk_r, and steps start at multiples of R). Every load is issued
 * unconditionally -- rows past the end read the last row, inactive chunks
 * the last chunk, and their results are discarded -- so no branch stands
 * between the loads and the waits that count them. */
template <int NCH, int R, int SF, bool RAW>
__device__ __forceinline__ void load_step(u32x4 (*wv)[NCH], uint32_t *sv, const uint8_t *W,
                                          const void *S, int rbase, int rend, int cols,
                                          int ch, int j, int tc, const int *cb, int sc,
                                          int blk_r)
{
#pragma unroll
    for (int i = 0; i < R; i++) {
        const int r = min(rbase + i, rend - 1);
#pragma unroll
        for (int n = 0; n < NCH; n++) {
            const int c = min(j + n * tc, ch - 1);
            wv[i][n] = ldg16_stream(W + (size_t)r * cols + (size_t)c * 16);
        }
    }
    const int rb = min(rbase, rend - 1) / blk_r;
#pragma unroll
    for (int n = 0; n < NCH; n++) {
        const uint32_t raw = ld_scale_raw<SF>(S, (size_t)rb * sc + cb[n]);
        sv[n] = RAW ? raw : __float_as_uint(scale_val<SF>(raw));
    }
}

/* Whether a step's scales stay as loaded until they are used (RAW) or are
 * decoded where they are loaded; and whether the first step's loads stand
 * behind a branch (HELD; always taken, a workgroup has rows) that keeps the
 * compiler from mixing them with x's. Neither changes a result. A kernel
 * whose x goes through LDS wants its scales raw and the loads free, so that
 * x does not wait for the first weights; but each form was measured, cold, us:
 *   - E8M0, x from L2: decoded and held (7168x12288 17.67 -> 17.09, 7168x7168
 *     12.12 -> 11.69), but raw for three chunks and one row per step without
 *     prefetch (4096x9216 12.71 -> 11.08, 5120x4608 8.91 -> 7.92) or two rows
 *     with it (3426x8464 10.67 -> 9.67), and raw and free for four chunks and
 *     two rows with prefetch (rows of 192 and 256 threads: 0.98 to 1.00 and
 *     0.97 to 0.99 times);
 *   - fp32, x from L2: held for one row per step (7168x7168 11.84 -> 11.50),
 *     for four, and for three chunks with prefetch (0.98 and 0.99 times), not
 *     for two rows else (16384x12288 35.7 -> 34.2, 1536x12288 8.11 -> 7.90);
 *   - rows of 128 threads through LDS, E8M0, four chunks, two rows per step
 *     without prefetch: decoded and held (10164x7824 16.86 -> 15.78);
 *   - rows of 256 threads through LDS: E8M0 decoded without prefetch
 *     (7168x16384 21.65 -> 20.95), raw with it (4096x16384 14.21 -> 14.05);
 *     fp32 held with prefetch (7168x16384 21.42 -> 20.77, 4096x16384 14.6 ->
 *     14.1), free in one step (256x16384 4.74 -> 4.19). */
template <int NCH, int R, int SF, int PF, int XL>
struct Fp8Form {
    static constexpr bool TWO_PF = R == 2 && PF;
    static constexpr bool X2 = XL == 2 && SF == 0 && NCH == 4 && R == 2 && !PF;
    static constexpr bool RAW = XL == 0 ? (NCH == 3 && R == 1 && !PF) || (NCH >= 3 && TWO_PF)
                                        : (XL != 4 || PF) && !X2;
    static constexpr bool HELD = XL != 0 ? X2 || (XL == 4 && SF == 1 && PF)
                               : SF == 0 ? !(NCH == 4 && TWO_PF)
                                         : R != 2 || (NCH == 3 && PF);
};

/* One workgroup owns the contiguous rows [row0, row0 + rows_per_wg). It walks
 * them in steps of rg*R rows (row group g takes rows g*R .. g*R+R-1 of the
 * step); with PF the next step's weights are in flight while this step's are
 * consumed. Rows that span several waves leave one partial per wave in LDS,
 * summed in wave order after a single barrier at the end. */
/* The GEMV of workgroup (bx, by): rows [bx rows_per_wg, +rows_per_wg) of
 * group or listed matrix by. part: LDS of [waves per row][rows_per_wg]
 * floats, then x (XL), then the norm's weights (NQ). */
template <int NCH, int R, int SF, int PF, int XL, int NQ = 0>
__device__ __forceinline__ void fp8_rows(float *__restrict__ y, const float *__restrict__ x,
                                         const uint8_t *__restrict__ W,
                                         const void *__restrict__ S, int rows, int cols, int sc,
                                         int blk_r, int blk_c, int tc, int rows_per_wg,
                                         const Fp8Groups &gp, int bx, int by, float *part,
                                         const float *__restrict__ nq_w = nullptr,
                                         float nq_eps = 0.0f)
{
    if (gp.list) {
        const int gi = by;
        W = gp.Wl[gi];
        S = gp.Sl[gi];
        y = gp.yl[gi];
        rows = gp.rl[gi];
        if (bx * rows_per_wg >= rows) return;     /* the whole workgroup */
    } else if (gp.n > 1) {
        const size_t gi = by;
        y += gi * gp.y;
        x += gi * gp.x;
        W += gi * gp.w;
        S = (const uint8_t *)S + gi * gp.s;
    }

    constexpr bool RAW = Fp8Form<NCH, R, SF, PF, XL>::RAW;
    constexpr bool HELD = Fp8Form<NCH, R, SF, PF, XL>::HELD;
    const int tid = threadIdx.x;
    const int g = tid / tc;
    const int j = tid - g * tc;
    const int rg = blockDim.x / tc;
    const int ch = cols >> 4;
    const int lane = tid & 63;
    const int row0 = bx * rows_per_wg;
    const int rend = min(rows, row0 + rows_per_wg);
    const int nloc = rend - row0;
    const int step_rows = rg * R;
    const int nsteps = (nloc + step_rows - 1) / step_rows;

    float xr[NCH][16];
    int cb[NCH];
    bool act[NCH];
#pragma unroll
    for (int n = 0; n < NCH; n++) {
        const int c = j + n * tc;
        act[n] = c < ch;
        cb[n] = act[n] ? (c * 16) / blk_c : 0;
    }

    u32x4 wv[R][NCH], wn[R][NCH];
    uint32_t sv[NCH], sn[NCH];
    if (XL) {
        /* x once per workgroup: the whole workgroup requests all of x (four
         * floats per thread per round, all rounds issued together), then the
         * first step's weights; x lands in LDS and each thread reads its
         * slice from there. Without this, every row group of the workgroup
         * would fetch the same x from L2.
         *
         * What is meant to overlap is x's way through LDS (and the norm) with
         * the first weights' latency, so nothing here should wait for those:
         * the scales stay raw (Fp8Form), no branch stands between the loads
         * and the waits that count them (lanes past x's end load and store
         * its last piece), and the rounds are the row's own (XL: the row's
         * waves, 1, 2 or 4). With the scales decoded where loaded and four
         * times the rounds, x was stored only once the weights had arrived
         * (24576x1536 9.26 us, now 8.54). */
        float *xs = part + (size_t)(tc > 64 ? tc / 64 : 0) * rows_per_wg;
        constexpr int XR = XL ? XL * NCH : 1;          /* rounds: cols <= 1024 XR */
        f32x4 xv[XR], nv[NQ ? XR : 1];
        const int nq = cols >> 2;
        /* (NQ: the norm's weights with x, ahead of the weights' requests, and
         * into LDS beside x) */
        float *xw = xs + cols;
#pragma unroll
        for (int q = 0; q < XR; q++) {
            const int i = 4 * min(q * (int)blockDim.x + tid, nq - 1);
            xv[q] = ldf4(x + i);
            if (NQ) nv[q] = ldf4(nq_w + i);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (!HELD || nsteps > 0)
            load_step<NCH, R, SF, RAW>(wv, sv, W, S, row0 + g * R, rend, cols, ch, j, tc, cb,
                                       sc, blk_r);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int q = 0; q < XR; q++) {
            const int i = 4 * min(q * (int)blockDim.x + tid, nq - 1);
            *reinterpret_cast<f32x4 *>(xs + i) = xv[q];
            if (NQ) *reinterpret_cast<f32x4 *>(xw + i) = nv[q];
        }
        __syncthreads();
        if (NQ) {
            /* x = w (x inv), the block's weighted RMSNorm (norm_rope_vec,
             * no RoPE) on the workgroup's copy, with its sum of squares in
             * its order: per thread the elements tid, tid + NR_THREADS, ...
             * in order, then block_sum_d (blockDim.x == NR_THREADS) */
            double sq = 0.0;
            for (int i = tid; i < cols; i += NR_THREADS) {
                const double v = (double)xs[i];
                sq += v * v;
            }
            sq = block_sum_d(sq);
            const float inv = (float)(1.0 / sqrt(sq / (double)cols + (double)nq_eps));
            for (int i = tid; i < cols; i += NR_THREADS) {
                const float v = xs[i] * inv;
                xs[i] = xw[i] * v;
            }
            __syncthreads();
        }
#pragma unroll
        for (int n = 0; n < NCH; n++) {
            const int c = min(j + n * tc, ch - 1);
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const f32x4 v = *reinterpret_cast<const f32x4 *>(xs + c * 16 + q * 4);
                xr[n][q * 4 + 0] = v.x; xr[n][q * 4 + 1] = v.y;
                xr[n][q * 4 + 2] = v.z; xr[n][q * 4 + 3] = v.w;
            }
        }
    } else {
#pragma unroll
        for (int n = 0; n < NCH; n++) {
            const int c = j + n * tc;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const f32x4 v = act[n] ? ldf4(x + c * 16 + q * 4) : f32x4{0, 0, 0, 0};
                xr[n][q * 4 + 0] = v.x; xr[n][q * 4 + 1] = v.y;
                xr[n][q * 4 + 2] = v.z; xr[n][q * 4 + 3] = v.w;
            }
        }
        if (!HELD || nsteps > 0)
            load_step<NCH, R, SF, RAW>(wv, sv, W, S, row0 + g * R, rend, cols, ch, j, tc, cb,
                                       sc, blk_r);
    }

    uint32_t sv0[NCH];
#pragma unroll
    for (int n = 0; n < NCH; n++) sv0[n] = sv[n];
    for (int step = 0; step < nsteps; ++step) {
        const int rbase = row0 + step * step_rows + g * R;
        if (PF && step + 1 < nsteps)
            load_step<NCH, R, SF, RAW>(wn, sn, W, S, rbase + step_rows, rend, cols, ch, j, tc,
                                       cb, sc, blk_r);

        float acc[R];
#pragma unroll
        for (int i = 0; i < R; i++) {
            float a = 0.0f;
#pragma unroll
            for (int n = 0; n < NCH; n++) {
                const float sf = RAW ? scale_val<SF>(sv[n]) : __uint_as_float(sv[n]);
                const float d = fmaf(dot16(wv[i][n], xr[n]), sf, a);
                a = act[n] ? d : a;
            }
            acc[i] = a;
        }

        if (tc <= 64) {
#pragma unroll
            for (int i = 0; i < R; i++) {
                const float v = seg_sum_rt(acc[i], tc);
                if (j == tc - 1 && rbase + i < rend) y[rbase + i] = v;
            }
        } else {
            const int w = j >> 6;                  /* wave within the row */
#pragma unroll
            for (int i = 0; i < R; i++) {
                const float v = seg_sum<64>(acc[i]);
                const int rl = rbase + i - row0;
                if (lane == 63 && rl < nloc) part[w * rows_per_wg + rl] = v;
            }
        }

        if (PF) {
#pragma unroll
            for (int i = 0; i < R; i++)
#pragma unroll
                for (int n = 0; n < NCH; n++) wv[i][n] = wn[i][n];
#pragma unroll
            for (int n = 0; n < NCH; n++) sv[n] = sn[n];
        } else if (step + 1 < nsteps) {
            load_step<NCH, R, SF, RAW>(wv, sv, W, S, rbase + step_rows, rend, cols, ch, j, tc,
                                       cb, sc, blk_r);
        }
    }

    /* A second use of the first step's raw scales, in no instruction. Without
     * it the compiler carries E8M0 scales into the loop as bytes and widens
     * them before it, behind a wait for the first weights that x's reads
     * from LDS then stand behind. */
    if (SF == 0 && XL && RAW) {
#pragma unroll
        for (int n = 0; n < NCH; n++) asm volatile("" ::"v"(sv0[n]));
    }

    if (tc > 64) {
        __syncthreads();
        const int wpr = tc >> 6;
        for (int rl = tid; rl < nloc; rl += blockDim.x) {
            float s = part[rl];
            for (int w = 1; w < wpr; w++) s += part[w * rows_per_wg + rl];
            y[row0 + rl] = s;
        }
    }
}

template <int NCH, int R, int SF, int PF, int XL>
__global__ void __launch_bounds__(256)
k_fp8_gemv(float *__restrict__ y, const float *__restrict__ x,
           const uint8_t *__restrict__ W, const void *__restrict__ S,
           int rows, int cols, int sc, int blk_r, int blk_c, int tc,
           int rows_per_wg, Fp8Groups gp)
{
    extern __shared__ float part[];     /* [waves per row][rows_per_wg], then x (XL) */
    fp8_rows<NCH, R, SF, PF, XL>(y, x, W, S, rows, cols, sc, blk_r, blk_c, tc, rows_per_wg, gp,
                                 (int)blockIdx.x, (int)blockIdx.y, part);
}

/* Batched: the per-(row, token) arithmetic of k_fp8_gemv with R = 1, looped
 * over tokens in blocks of TB with the row's weight chunks held in VGPRs. */
template <int NCH, int SF>
__global__ void __launch_bounds__(256)
k_fp8_gemv_n(float *__restrict__ y, const float *__restrict__ x,
             const uint8_t *__restrict__ W, const void *__restrict__ S,
             int rows, int cols, int sc, int blk_r, int blk_c, int tc, int nt)
{
    constexpr int TB = 8;
    __shared__ float red[4][TB];

    const int tid = threadIdx.x;
    const int g = tid / tc;
    const int j = tid - g * tc;
    const int rg = blockDim.x / tc;
    const int ch = cols >> 4;
    const int wid = tid >> 6, lane = tid & 63;
    const int r = blockIdx.x * rg + g;       /* this row group's row */
    const bool rok = r < rows;

    float wf[NCH][16];                       /* the row's chunks, decoded once */
    float sreg[NCH];
    bool act[NCH];
#pragma unroll
    for (int n = 0; n < NCH; n++) {
        const int c = j + n * tc;
        act[n] = c < ch;
        const u32x4 wv = (act[n] && rok) ? ld16(W + (size_t)r * cols + (size_t)c * 16)
                                         : u32x4{0, 0, 0, 0};
        sreg[n] = (act[n] && rok)
                ? ld_scale<SF>(S, (size_t)(r / blk_r) * sc + (c * 16) / blk_c)
                : 0.0f;
        dec_e4m3x4(wv.x, wf[n] + 0);
        dec_e4m3x4(wv.y, wf[n] + 4);
        dec_e4m3x4(wv.z, wf[n] + 8);
        dec_e4m3x4(wv.w, wf[n] + 12);
    }

    for (int tb = 0; tb < nt; tb += TB) {
        float acc[TB];
#pragma unroll
        for (int t = 0; t < TB; t++) {
            float a = 0.0f;
            if (tb + t < nt) {
                const float *xt = x + (size_t)(tb + t) * cols;
#pragma unroll
                for (int n = 0; n < NCH; n++) {
                    float xr[16];
                    const int c = j + n * tc;
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        const f32x4 v = act[n] ? ldf4(xt + c * 16 + q * 4)
                                               : f32x4{0, 0, 0, 0};
                        xr[q * 4 + 0] = v.x; xr[q * 4 + 1] = v.y;
                        xr[q * 4 + 2] = v.z; xr[q * 4 + 3] = v.w;
                    }
                    a = fmaf(dot16f(wf[n], xr), sreg[n], a);
                }
            }
            acc[t] = a;
        }
        if (tc <= 64) {
#pragma unroll
            for (int t = 0; t < TB; t++) {
                const float v = seg_sum_rt(acc[t], tc);
                if (j == tc - 1 && rok && tb + t < nt)
                    y[(size_t)(tb + t) * rows + r] = v;
            }
        } else {
            const int wpr = tc >> 6;
#pragma unroll
            for (int t = 0; t < TB; t++) {
                const float v = seg_sum<64>(acc[t]);
                if (lane == 63) red[wid][t] = v;
            }
            __syncthreads();
            if (tid < rg * TB) {
                const int gg = tid / TB, tt = tid - gg * TB;
                const int rr = blockIdx.x * rg + gg;
                float s = red[gg * wpr][tt];
                for (int w = 1; w < wpr; w++) s += red[gg * wpr + w][tt];
                if (rr < rows && tb + tt < nt) y[(size_t)(tb + tt) * rows + rr] = s;
            }
            __syncthreads();
        }
    }
}

/* Any shape the chunked kernel does not take (cols not a multiple of 16, or
 * wider than 16384): one wave per row, one element per lane per step. */
template <int SF>
__global__ void __launch_bounds__(256)
k_fp8_gemv_generic(float *__restrict__ y, const float *__restrict__ x,
                   const uint8_t *__restrict__ W, const void *__restrict__ S,
                   int rows, int cols, int sc, int blk_r, int blk_c, int nt)
{
    const int wpb = blockDim.x >> 6;
    const int r = blockIdx.x * wpb + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (r >= rows) return;
    const uint8_t *row = W + (size_t)r * cols;
    for (int t = 0; t < nt; t++) {
        const float *xt = x + (size_t)t * cols;
        float a = 0.0f;
        for (int c = lane; c < cols; c += 64) {
            const float s = ld_scale<SF>(S, (size_t)(r / blk_r) * sc + c / blk_c);
            a = fmaf(dec_e4m3(row[c]) * xt[c], s, a);
        }
        const float v = wave_sum(a);
        if (lane == 0) y[(size_t)t * rows + r] = v;
    }
}

int g_cu_count = 0;

int env_int(const char *name, int dflt)
{
    const char *e = getenv(name);
    return e ? atoi(e) : dflt;
}

int cu_count()
{
    if (!g_cu_count) {
        int dev = 0, n = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
            n <= 0)
            n = 256;
        g_cu_count = n;
    }
    return g_cu_count;
}

/* Launch plan of the VALU form: x through LDS or not, the rows each
 * workgroup owns, the grid along x and the dynamic LDS. */
struct Fp8Plan {
    int xl = 0, rows_per_wg = 0, grid = 0;
    size_t lds = 0;
};

/* Whether a row's x goes through LDS, one fetch per workgroup instead of one
 * per row group (steps: a workgroup's; wgs: the launch's workgroups). Rows of up to 64 threads: always (us,
 * cold, each thread its own x from L2 / through LDS: 4096x4096 5.99 / 5.57,
 * 512x4096 3.73 / 3.28, 32768x4096 25.0 / 23.6, 24576x1536 9.68 / 9.25). Wider
 * rows have fewer row groups to share it, and each group's rounds of 1024
 * columns cost their latency whether x fills them or not (full: it does):
 *   - 128 threads, E8M0: where a step has four rows or the next one is
 *     prefetched (1536x7168 5.71 / 5.56, 2560x4608 6.51 / 5.93), or four
 *     chunks fill the rounds (2048x8192 6.63 / 6.30; 7168x7168 11.7 / 12.0,
 *     8192x4608 9.44 / 9.85, 1024x4608 3.96 / 4.39) or, two rows per step, up to
 *     three workgroups for two CUs (4435x7104 10.05 / 9.67, 5786x6240 9.60 / 10.10);
 *   - 128 threads, fp32: not for one row per step (512x4608 3.58 / 3.79,
 *     5120x4608 7.70 / 8.18), but where four chunks fill the rounds (512x8192
 *     3.95 / 3.77), with prefetch where the rounds are full or there are
 *     four chunks (4096x5120 6.92 / 7.19; 2048x7168 6.03 / 5.93), and for three
 *     chunks without prefetch from four steps on (5823x5200 8.40 / 8.60);
 *   - 256 threads: where a workgroup has several steps or a CU several
 *     workgroups, which then want x at once (4096x13312 14.5 / 12.2, E8M0
 *     936x14400 7.02 / 6.64, 1024x16384 7.4 / 6.8; 199x15664 4.69 / 4.86, fp32
 *     78x15680 4.01 / 4.20, and 3.72 / 4.25 with W in the Infinity Cache).
 * Rows of 192 threads, whose workgroup is not 256, read it from L2. */
bool fp8_xl(const Fp8Geom &g, int R, int pf, int sfmt, int cols, int steps, int wgs)
{
    if (g.wg != 256 || (cols & 3)) return false;
    const int waves = g.tc > 64 ? g.tc / 64 : 1;
    const bool full = cols > 1024 * (waves * g.nch - 1);
    bool xl = true;
    if (waves == 2)
        xl = R == 4 || (g.nch == 4 && full) ||
             (sfmt == 0 ? pf != 0 || (g.nch == 4 && R == 2 && wgs * 2 <= 3 * cu_count())
                        : R == 2 && (g.nch == 4 || (pf ? full : steps >= 4)));
    else if (waves == 4)
        xl = steps > 1 || wgs > cu_count();
    return env_int("DSV4_GPU_FP8_XL", xl) != 0;
}

Fp8Plan fp8_plan(const Fp8Geom &g, int R, int pf, int sfmt, int rows, int cols, int wgs_per_cu,
                 int ngroups, bool lds_x = true)
{
    Fp8Plan p;
    const int step_rows = g.rg * R;
    const int nsteps = (rows + step_rows - 1) / step_rows;
    const int want = (wgs_per_cu * cu_count() + ngroups - 1) / ngroups;
    int spw = (nsteps + want - 1) / want;              /* steps per workgroup */
    const int wpr = g.tc > 64 ? g.tc / 64 : 1;
    const int max_spw = PART_MAX / wpr / step_rows;
    if (spw > max_spw) spw = max_spw;
    if (spw < 1) spw = 1;
    p.rows_per_wg = spw * step_rows;
    p.grid = (rows + p.rows_per_wg - 1) / p.rows_per_wg;
    p.xl = lds_x && fp8_xl(g, R, pf, sfmt, cols, spw, p.grid * ngroups);
    p.lds = (g.tc > 64 ? sizeof(float) * (size_t)wpr * p.rows_per_wg : 0)
          + (p.xl ? sizeof(float) * (size_t)cols : 0);
    return p;
}

template <int NCH, int R, int SF, int PF>
void launch_gemv(const Fp8Geom &g, float *y, const float *x, const uint8_t *W,
                 const void *S, int rows, int cols, int sc, int blk_r,
                 int blk_c, int wgs_per_cu, const Fp8Groups &gp, hipStream_t st)
{
    const Fp8Plan p = fp8_plan(g, R, PF, SF, rows, cols, wgs_per_cu, gp.n);
    auto go = [&](auto kern, bool *opted) {
        if (opted && !*opted) {                     /* x of up to 64 KB + partials */
            (void)dsv4_lds_optin((const void *)kern, dsv4_lds_limit(), "fp8 gemv");
            *opted = true;
        }
        hipLaunchKernelGGL(kern, dim3(p.grid, gp.n), dim3(g.wg), p.lds, st, y, x, W, S, rows,
                           cols, sc, blk_r, blk_c, g.tc, p.rows_per_wg, gp);
    };
    static bool opted[3] = {};
    if (!p.xl) return go(k_fp8_gemv<NCH, R, SF, PF, 0>, nullptr);
    /* fp8_geom: two waves per row have 3 or 4 chunks per thread, four 4 */
    if constexpr (NCH == 4)
        if (g.tc > 128) return go(k_fp8_gemv<NCH, R, SF, PF, 4>, &opted[2]);
    if constexpr (NCH >= 3)
        if (g.tc > 64) return go(k_fp8_gemv<NCH, R, SF, PF, 2>, &opted[1]);
    go(k_fp8_gemv<NCH, R, SF, PF, 1>, &opted[0]);
}

template <int R, int SF, int PF>
void launch_gemv_nch(const Fp8Geom &g, float *y, const float *x,
                     const uint8_t *W, const void *S, int rows, int cols,
                     int sc, int blk_r, int blk_c, int wpc, const Fp8Groups &gp,
                     hipStream_t st)
{
    switch (g.nch) {
    case 1: launch_gemv<1, R, SF, PF>(g, y, x, W, S, rows, cols, sc, blk_r, blk_c, wpc, gp, st); break;
    case 2: launch_gemv<2, R, SF, PF>(g, y, x, W, S, rows, cols, sc, blk_r, blk_c, wpc, gp, st); break;
    case 3: launch_gemv<3, R, SF, PF>(g, y, x, W, S, rows, cols, sc, blk_r, blk_c, wpc, gp, st); break;
    default: launch_gemv<4, R, SF, PF>(g, y, x, W, S, rows, cols, sc, blk_r, blk_c, wpc, gp, st); break;
    }
}

template <int SF, int PF>
void launch_gemv_r(const Fp8Geom &g, int R, float *y, const float *x,
                   const uint8_t *W, const void *S, int rows, int cols, int sc,
                   int blk_r, int blk_c, int wpc, const Fp8Groups &gp, hipStream_t st)
{
    switch (R) {
    case 1: launch_gemv_nch<1, SF, PF>(g, y, x, W, S, rows, cols, sc, blk_r, blk_c, wpc, gp, st); break;
    case 2: launch_gemv_nch<2, SF, PF>(g, y, x, W, S, rows, cols, sc, blk_r, blk_c, wpc, gp, st); break;
    default: launch_gemv_nch<4, SF, PF>(g, y, x, W, S, rows, cols, sc, blk_r, blk_c, wpc, gp, st); break;
    }
}

/* Batched with x through LDS (prefill, nt >= 2): a workgroup of 512 threads
 * (rg = 512 / tc row groups) owns the rows [row0, row0 + rows_per_wg) and
 * walks the tokens in blocks of TB, staged in LDS (TB x cols floats) and
 * read by every row group. A row group takes RR rows per step (rb + g,
 * rb + g + rg, ...), decodes their chunks once for the block, and applies
 * each x piece it reads from LDS to all RR rows. Per (row, token) the
 * arithmetic is k_fp8_gemv's (chunk order, scale fma, segment tree, wave
 * partials in wave order), so every result keeps the GEMV's bits. */
template <int NCH, int SF, int TB, int RR>
__global__ void __launch_bounds__(512)
k_fp8_gemv_nl(float *__restrict__ y, const float *__restrict__ x,
              const uint8_t *__restrict__ W, const void *__restrict__ S, int rows, int cols,
              int sc, int blk_r, int blk_c, int tc, int nt, int rows_per_wg)
{
    /* x of the block as [TB][4 quads][ch chunks] 16-byte pieces: a row
     * group's lanes read consecutive pieces (conflict-free), red after */
    extern __shared__ __attribute__((aligned(16))) float xl[];
    const int tid = threadIdx.x;
    const int g = tid / tc, j = tid - g * tc;
    const int rg = blockDim.x / tc;
    const int ch = cols >> 4;
    const int wid = tid >> 6, lane = tid & 63;
    const int row0 = blockIdx.x * rows_per_wg;
    const int rend = min(rows, row0 + rows_per_wg);
    float *red = xl + (size_t)TB * cols;
    bool act[NCH];
    int cb[NCH];
#pragma unroll
    for (int n = 0; n < NCH; n++) {
        const int c = j + n * tc;
        act[n] = c < ch;
        cb[n] = (min(c, ch - 1) * 16) / blk_c;
    }
    for (int tb = 0; tb < nt; tb += TB) {
        const int ntb = min(TB, nt - tb);
        __syncthreads();                           /* the previous block's reads */
        {
            const int n4 = (ntb * cols) >> 2;
            const float *xs = x + (size_t)tb * cols;
            for (int i0 = 0; i0 < n4; i0 += 8 * (int)blockDim.x) {
                f32x4 v[8];
#pragma unroll
                for (int u = 0; u < 8; u++)
                    v[u] = ldf4(xs + 4 * min(i0 + u * (int)blockDim.x + tid, n4 - 1));
#pragma unroll
                for (int u = 0; u < 8; u++) {
                    const int i = i0 + u * (int)blockDim.x + tid;
                    if (i < n4) {
                        const int t = (4 * i) / cols, e = 4 * i - t * cols;
                        const int c = e >> 4, q = (e >> 2) & 3;
                        *reinterpret_cast<f32x4 *>(xl + (size_t)t * cols + (size_t)q * ch * 4 +
                                                   c * 4) = v[u];
                    }
                }
            }
        }
        __syncthreads();
        for (int rb = row0; rb < rend; rb += RR * rg) {  /* uniform: every group steps */
            int rr[RR];
            bool rok[RR];
            float wf[RR][NCH][16];
            float sreg[RR][NCH];
#pragma unroll
            for (int k = 0; k < RR; k++) {
                const int r = rb + g + k * rg;
                rok[k] = r < rend;
                rr[k] = rok[k] ? r : rend - 1;
#pragma unroll
                for (int n = 0; n < NCH; n++) {
                    const int c = min(j + n * tc, ch - 1);
                    const u32x4 wv = ld16(W + (size_t)rr[k] * cols + (size_t)c * 16);
                    sreg[k][n] = ld_scale<SF>(S, (size_t)(rr[k] / blk_r) * sc + cb[n]);
                    dec_e4m3x4(wv.x, wf[k][n] + 0);
                    dec_e4m3x4(wv.y, wf[k][n] + 4);
                    dec_e4m3x4(wv.z, wf[k][n] + 8);
                    dec_e4m3x4(wv.w, wf[k][n] + 12);
                }
            }
            float acc[RR][TB];
#pragma unroll
            for (int t = 0; t < TB; t++) {
                float a[RR];
#pragma unroll
                for (int k = 0; k < RR; k++) a[k] = 0.0f;
                const float *xt = xl + (size_t)min(t, ntb - 1) * cols;
#pragma unroll
                for (int n = 0; n < NCH; n++) {
                    const int c = min(j + n * tc, ch - 1);
                    float xr[16];
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        const f32x4 v =
                            *reinterpret_cast<const f32x4 *>(xt + (size_t)q * ch * 4 + c * 4);
                        xr[q * 4 + 0] = v.x; xr[q * 4 + 1] = v.y;
                        xr[q * 4 + 2] = v.z; xr[q * 4 + 3] = v.w;
                    }
#pragma unroll
                    for (int k = 0; k < RR; k++) {
                        const float d = fmaf(dot16f(wf[k][n], xr), sreg[k][n], a[k]);
                        a[k] = act[n] ? d : a[k];
                    }
                }
#pragma unroll
                for (int k = 0; k < RR; k++) acc[k][t] = a[k];
            }
            if (tc <= 64) {
#pragma unroll
                for (int k = 0; k < RR; k++)
#pragma unroll
                    for (int t = 0; t < TB; t++) {
                        const float v = seg_sum_rt(acc[k][t], tc);
                        if (j == tc - 1 && rok[k] && t < ntb)
                            y[(size_t)(tb + t) * rows + rb + g + k * rg] = v;
                    }
            } else {
                const int wpr = tc >> 6;
#pragma unroll
                for (int k = 0; k < RR; k++)
#pragma unroll
                    for (int t = 0; t < TB; t++) {
                        const float v = seg_sum<64>(acc[k][t]);
                        if (lane == 63) red[(k * 8 + wid) * TB + t] = v;
                    }
                __syncthreads();
                if (tid < RR * rg * TB) {
                    const int k = tid / (rg * TB), rem = tid - k * (rg * TB);
                    const int gg = rem / TB, tt = rem - gg * TB;
                    const int ro = rb + gg + k * rg;
                    const float *rk = red + (size_t)k * 8 * TB;
                    float s = rk[(gg * wpr) * TB + tt];
                    for (int w = 1; w < wpr; w++) s += rk[(gg * wpr + w) * TB + tt];
                    if (ro < rend && tt < ntb) y[(size_t)(tb + tt) * rows + ro] = s;
                }
                __syncthreads();
            }
        }
    }
}

template <int NCH, int SF, int TB>
void launch_gemv_nl(const Fp8Geom &g, float *y, const float *x, const uint8_t *W,
                    const void *S, int rows, int cols, int sc, int blk_r, int blk_c, int nt,
                    hipStream_t st)
{
    constexpr int RR = 2;
    static bool opted = false;
    if (!opted) {
        (void)dsv4_lds_optin((const void *)k_fp8_gemv_nl<NCH, SF, TB, RR>, dsv4_lds_limit(),
                             "fp8 gemv_n");
        opted = true;
    }
    const int step = RR * (512 / g.tc);
    /* about one workgroup per CU: each stages every token block once */
    const int want = cu_count();
    int rpw = (rows + want - 1) / want;
    rpw = (rpw + step - 1) / step * step;
    const int grid = (rows + rpw - 1) / rpw;
    const size_t lds = sizeof(float) * ((size_t)TB * cols + (size_t)RR * 8 * TB);
    hipLaunchKernelGGL((k_fp8_gemv_nl<NCH, SF, TB, RR>), dim3(grid), dim3(512), lds, st, y,
                       x, W, S, rows, cols, sc, blk_r, blk_c, g.tc, nt, rpw);
}

template <int SF, int TB>
void launch_gemv_nl_nch(const Fp8Geom &g, float *y, const float *x, const uint8_t *W,
                        const void *S, int rows, int cols, int sc, int blk_r, int blk_c,
                        int nt, hipStream_t st)
{
    switch (g.nch) {
    case 1: launch_gemv_nl<1, SF, TB>(g, y, x, W, S, rows, cols, sc, blk_r, blk_c, nt, st); break;
    case 2: launch_gemv_nl<2, SF, TB>(g, y, x, W, S, rows, cols, sc, blk_r, blk_c, nt, st); break;
    case 3: launch_gemv_nl<3, SF, TB>(g, y, x, W, S, rows, cols, sc, blk_r, blk_c, nt, st); break;
    default: launch_gemv_nl<4, SF, TB>(g, y, x, W, S, rows, cols, sc, blk_r, blk_c, nt, st); break;
    }
}

/* ---------------------------------------------- batched on the matrix core
 *
 * The batched GEMV's plan on the f32 matrix core (dsv4_batch_mf.hip, the
 * GEMV's bits): whether it runs, and the workgroups per tile of 16 rows x 16
 * tokens. It takes batches of 5 tokens on: below that its tile is mostly empty
 * columns (us, matrix core / VALU, E8M0: 7168x7168 at 4 tokens 27.4 / 24.0, 6
 * tokens 28.0 / 43.6, 64 tokens 81.5 / 334.7; 1536x7168 at 4 tokens 12.9 /
 * 10.1, at 6 12.9 / 15.9; of 1360 shapes of 16 to 24576 rows and 64 to 16384
 * columns none of 5 tokens or more was slower than before). Rows of 192
 * threads, which k_fp8_gemv_nl does not take: from 8 tokens, few of them from
 * 9 or 11 (64x8208 at 8 tokens 10.5 / 8.2, at 10 10.6 / 10.1; 256x12288 at 9
 * 12.9 / 12.0, at 12 12.9 / 14.6; 512x10240 at 8 13.2 / 12.9); up to 256 rows
 * a token later with fp32 scales, which the VALU loads faster, and another
 * around 10240 columns (fp32 128x8704 at 11 tokens 1.04 times the VALU's, at
 * 12 0.99; 64x10240 at 11 13.0 / 11.5, at 13 13.4 / 12.8; E8M0 128x10240 at
 * 11 1.08 times, at 12 1.02).
 *
 * While the tiles leave CUs idle, rows of 4096 columns on are split
 * over 4, 3 or 2 workgroups (a row's 64-slot blocks, or parts of one) that a
 * second launch joins: a tile's time is its chain down the row, and half of
 * it is worth more than the launch (us, split by 1 / 2 / 4: 1536x7168 at 13
 * tokens 15.4 / 13.4 / -, 576x7168 at 16 14.9 / 12.7 / 9.4, 1024x16384 at 16
 * 29.8 / 21.5 / 15.0, 2048x4096 at 16 11.0 / 10.1 / -; at 512x2048 no gain,
 * 7.1 / 7.1 / 7.1). Rows of 192 threads also while the tiles are a few more
 * than the CUs, up to four thirds: thirds of a tile even out what whole tiles
 * leave to a second round (5120x12288 at 16 tokens 48.8 / 34.6 by 3, 5120x
 * 9216 38.4 / 28.1). DSV4_GPU_MFN_L (slots per wave) takes the form at any
 * batch, unsplit. */
int mf_slots() { return env_int("DSV4_GPU_MFN_L", 0); }

int mf_split(const Fp8Geom &g, int rows, int nt)
{
    const long long tiles = (long long)((rows + 15) / 16) * ((nt + 15) / 16);
    const int cu = cu_count();
    if (mf_slots() != 0 || g.ch < 256 || g.tc < 64) return 1;
    if (g.tc == 192) {
        const long long t = dsv4_batch_mf_tiles(rows, nt, g.tc);
        return tiles * 3 <= cu || (t > cu && t * 3 <= 4 * cu) ? 3 : 1;
    }
    return tiles * 4 <= cu ? 4 : tiles * 2 <= cu ? 2 : 1;
}

/* the most LDS k_fp8_gemv_nl takes for a block of tokens' x */
size_t nl_cap() { return dsv4_lds_limit() - 2048; }

/* From how many tokens. Where tiles would be split but the call has no place for
 * their part sums (a captured one, say), a whole tile's chain is twice or four
 * times as long, and the VALU keeps more tokens (us, whole tiles / VALU):
 *   - 128 threads a row: 512x6144 at 5 tokens 14.8 / 13.2, at 7 14.8 / 14.2;
 *     where k_fp8_gemv_nl holds eight tokens of x, 512x4112 at 8 1.16 times
 *     the VALU's, at 9 0.77;
 *   - 192: 64x10240 at 12 21.2 / 13.4, 512x12288 at 12 24.7 / 22.7, at 16
 *     25.2 / 27.9, 1024x12288 at 8 24.6 / 30.3;
 *   - 256: 512x14336 at 8 27.2 / 24.9, at 9 27.6 / 28.9; 512x16384 at 9 30.8
 *     / 29.9; of 1360 rows on from 5. */
int mf_from(const Fp8Geom &g, int sfmt, int rows, int cols, bool whole)
{
    if (g.tc == 192) {
        if (whole) return rows <= 256 ? 21 : rows <= 512 ? 15 : rows <= 768 ? 10 : 8;
        if (rows <= 256) return 11 + (sfmt != 0) + (cols > 9856 && cols <= 10496);
        return rows <= 512 ? 9 : 8;
    }
    if (whole && g.tc == 128) return 8 * sizeof(float) * (size_t)cols <= nl_cap() ? 9 : 7;
    if (whole && g.tc == 256 && rows <= 1024) return cols > 15360 ? 10 : 9;
    return 5;
}

bool mf_takes(const Fp8Geom &g, int sfmt, int rows, int cols, int blk_r, int nt, bool whole)
{
    return env_int("DSV4_GPU_FP8_MFN", 1) != 0 && nt >= 2 && g.tc >= 4 && (blk_r & 15) == 0 &&
           (mf_slots() != 0 || nt >= mf_from(g, sfmt, rows, cols, whole));
}

/* 0; -1 where the f32 matrix-core form's launch failed, whose error it has
 * taken (a failed launch of the others is still there for the caller to get) */
template <int SF>
int launch_gemv_n(const Fp8Geom &g, float *y, const float *x, const uint8_t *W,
                  const void *S, int rows, int cols, int sc, int blk_r,
                  int blk_c, int nt, hipStream_t st, void *scratch)
{
    const int split = mf_split(g, rows, nt);
    if (mf_takes(g, SF, rows, cols, blk_r, nt, split > 1 && !scratch)) {
        Dsv4BatchMf b;
        b.fmt = SF; b.y = y; b.x = x; b.W = W; b.S = S;
        b.rows = rows; b.cols = cols; b.nt = nt;
        b.tc = g.tc; b.sc = sc; b.blk_r = blk_r; b.blk_c = blk_c;
        b.slots = mf_slots();
        b.split = split;
        b.part = (float *)scratch;
        const int rc = dsv4_batch_mf_launch(b, st);
        if (rc <= 0) return rc;
    }
    /* two or more tokens: x through LDS, the largest token block that fits
     * and the tokens fill (8 x 4096, 4 x 7168, 2 x 16384 columns); three
     * tokens take one block of four rather than two of two (us, 7168x7168 31.9
     * -> 24.0, 1536x7168 11.3 -> 10.1) */
    const size_t cap = nl_cap();
    if (nt >= 2 && (((uintptr_t)x) & 15) == 0 && g.tc <= 256 && 512 % g.tc == 0) {
        const size_t row4 = sizeof(float) * (size_t)cols;
        if (nt >= 8 && 8 * row4 <= cap) { launch_gemv_nl_nch<SF, 8>(g, y, x, W, S, rows, cols, sc, blk_r, blk_c, nt, st); return 0; }
        if (nt >= 3 && 4 * row4 <= cap) { launch_gemv_nl_nch<SF, 4>(g, y, x, W, S, rows, cols, sc, blk_r, blk_c, nt, st); return 0; }
        if (2 * row4 <= cap) { launch_gemv_nl_nch<SF, 2>(g, y, x, W, S, rows, cols, sc, blk_r, blk_c, nt, st); return 0; }
    }
    const int grid = (rows + g.rg - 1) / g.rg;
    switch (g.nch) {
    case 1: hipLaunchKernelGGL((k_fp8_gemv_n<1, SF>), dim3(grid), dim3(g.wg), 0, st, y, x, W, S, rows, cols, sc, blk_r, blk_c, g.tc, nt); break;
    case 2: hipLaunchKernelGGL((k_fp8_gemv_n<2, SF>), dim3(grid), dim3(g.wg), 0, st, y, x, W, S, rows, cols, sc, blk_r, blk_c, g.tc, nt); break;
    case 3: hipLaunchKernelGGL((k_fp8_gemv_n<3, SF>), dim3(grid), dim3(g.wg), 0, st, y, x, W, S, rows, cols, sc, blk_r, blk_c, g.tc, nt); break;
    default: hipLaunchKernelGGL((k_fp8_gemv_n<4, SF>), dim3(grid), dim3(g.wg), 0, st, y, x, W, S, rows, cols, sc, blk_r, blk_c, g.tc, nt); break;
    }
    return 0;
}

bool blocking_ok(int blk_r, int blk_c)
{
    return blk_r >= 1 && blk_c >= 16 && (blk_c & 15) == 0;
}

/* Which arithmetic a matrix gets, by its format and shape alone (never by the
 * batch size or by where x lies, so the single-token and batched calls agree
 * bit for bit):
 *   - by default every matrix takes the VALU form of this file, the faster
 *     one at batch 1 on every shape measured (E8M0, cold, us, VALU against
 *     matrix core: 576x7168 4.41 / 8.07, 1536x7168 6.04 / 8.44, 24576x1536
 *     10.03 / 11.27, 7168x7168 11.90 / 12.92, 7168x16384 21.58 / 23.85, LM
 *     head 140.4 / 142.2, 2048x4096 4.77 / 6.68, 4096x2048 5.05 / 6.40);
 *   - DSV4_GPU_FP8_MX=1 sends E8M0-scaled matrices the matrix-core form
 *     (dsv4_fp8_mx.hip), single token and batched alike: slower at batch 1,
 *     much faster batched (7168x7168 at 64 tokens 63.9 against 335.2 us),
 *     for prefill-heavy work;
 *   - shapes neither chunked kernel takes run the generic kernel.
 * The chunked forms need x and W 16-byte aligned; a call that breaks that
 * is refused rather than sent to another arithmetic (chunked_ok). */
bool mx_form(int sfmt, int cols, int blk_r, int blk_c)
{
    return env_int("DSV4_GPU_FP8_MX", 0) != 0 && dsv4_fp8_mx_ok(sfmt, cols, blk_r, blk_c);
}

/* x and W of a chunked-form call are 16-byte aligned; else -1 with a
 * message (the host-buffer entry points stage x aligned, and the
 * residency keeps W as allocated, so only a caller's device pointer can
 * break this). */
int chunked_ok(const float *x, const uint8_t *W, const char *what)
{
    if ((((uintptr_t)x | (uintptr_t)W) & 15) == 0) return 0;
    DSV4_ERR("%s: x (%p) and W (%p) must be 16-byte aligned", what, (const void *)x,
             (const void *)W);
    return -1;
}

/* The VALU form's launch parameters for a matrix of rows x cols: R rows per
 * thread per step (at most blk_r's largest power-of-two divisor up to 4),
 * the next step prefetched or not, workgroups per CU. None of these changes
 * a row's arithmetic, and the environment can override each. The rule, from
 * sweeps over the C1/C2 and attention-block shapes on MI355X (R in 1, 2, 4;
 * prefetch on/off; x through LDS or not; 1-8 workgroups per CU; cold, us):
 *   - two workgroups per CU (four when rows are narrow, cols < 4096);
 *   - rows of 16384 columns with fp32 scales: one row per step with the
 *     next, if there is one, prefetched (7168x16384: 21.7-22.2 -> 21.1-21.3);
 *     with E8M0
 *     scales the base below (21.2-21.4 against 22.4-22.5 for one row);
 *   - more than 4096 rows: two rows per step without prefetch, unless that
 *     grid leaves its last round of workgroups short, so that some CUs get
 *     fewer than others, while one row per step fills it (7168x7168: 448
 *     workgroups at two rows, 512 at one; 12.0 -> 11.5). The LM head keeps
 *     two (505 workgroups; one row per step measured 147 against 137.5);
 *   - at most 4096 rows of at least 4096 columns: one row per step without
 *     prefetch where that grid is one round of workgroups (1024x4096 4.4 ->
 *     3.8, 512x4096 4.2 -> 3.6, either scale format), or, with E8M0 scales,
 *     where its rounds are full (4096x8192 9.9 -> 9.1, 4096x4096 6.2 ->
 *     6.1; with fp32 scales, whose step loads four bytes of scale per
 *     chunk, 9.5 either way and 6.1 against 6.2 for two rows);
 *     else four rows per step without prefetch where only that grid is
 *     full (1536x7168: 384 workgroups at two rows, 192 at four; 5.9 ->
 *     5.7); otherwise, and for narrower rows, two rows per step with the
 *     next prefetched (576x7168: 4.3 at two rows, 4.6 at one, whose 288
 *     workgroups spill onto 32 CUs).
 * tuned = false keeps the base rule (two rows; prefetch where rows <= 4096)
 * for the attention block's combined launches, which are built for it. */
struct Fp8Valu {
    int R, pf, wpc;
};

Fp8Valu fp8_valu(int rows, int cols, int blk_r, int sfmt, bool tuned = true)
{
    Fp8Valu v;
    v.wpc = env_int("DSV4_GPU_FP8_WPC", cols >= 4096 ? 2 : 4);
    if (v.wpc <= 0) v.wpc = 2;
    int R = 2, pf = rows <= 4096 ? 1 : 0;
    Fp8Geom g;
    if (tuned && fp8_geom(cols, &g)) {
        const int cu = cu_count();
        /* every round of workgroups but the last is full; the last at least
         * 15/16 full, or the grid is a single round */
        auto grid = [&](int r) { return fp8_plan(g, r, 0, sfmt, rows, cols, v.wpc, 1, false).grid; };
        auto full = [&](int r) {
            const int n = grid(r), last = n % cu;
            return n <= cu || last == 0 || last * 16 >= cu * 15;
        };
        if (g.tc == 256) {
            if (sfmt != 0) {
                const Fp8Plan p = fp8_plan(g, 1, 0, sfmt, rows, cols, v.wpc, 1, false);
                R = 1;
                pf = p.rows_per_wg > g.rg;
            }
        } else if (rows > 4096) {
            if (!full(2) && full(1)) R = 1;
        } else if (cols >= 4096) {
            if (sfmt == 0 ? full(1) : grid(1) <= cu) {
                R = 1;
                pf = 0;
            } else if (!full(2) && full(4)) {
                R = 4;
                pf = 0;
            }
        }
    }
    R = env_int("DSV4_GPU_FP8_R", R);
    R = R >= 4 ? 4 : R >= 2 ? 2 : 1;
    while (blk_r % R) R >>= 1;                   /* a step stays in one row block */
    v.R = R;
    v.pf = env_int("DSV4_GPU_FP8_PF", pf);
    return v;
}

int fp8_gemv(float *y, const float *x, const uint8_t *W, const void *S, int sfmt,
             int rows, int cols, int blk_r, int blk_c, const Fp8Groups &gp,
             hipStream_t st)
{
    if (rows <= 0 || cols <= 0 || blk_r <= 0 || blk_c <= 0 || gp.n <= 0 || gp.n > 65535) {
        DSV4_ERR("fp8 gemv: bad shape %dx%d blk %dx%d", rows, cols, blk_r, blk_c);
        return -1;
    }
    const int sc = (cols + blk_c - 1) / blk_c;
    Fp8Geom g;
    if (!gp.valu && mx_form(sfmt, cols, blk_r, blk_c)) {
        if (chunked_ok(x, W, "fp8 gemv") != 0) return -1;
        Dsv4Fp8Mx a;
        a.y = y; a.x = x; a.w = W; a.s = (const uint8_t *)S;
        a.rows = rows; a.cols = cols; a.sc = sc; a.blk_r = blk_r; a.blk_c = blk_c;
        a.n = gp.n;
        a.x_stride = gp.x; a.y_stride = gp.y; a.w_stride = gp.w; a.s_stride = gp.s;
        a.list = gp.list;
        for (int i = 0; gp.list && i < gp.n; i++) {
            a.wl[i] = gp.Wl[i]; a.sl[i] = (const uint8_t *)gp.Sl[i];
            a.yl[i] = gp.yl[i]; a.rl[i] = gp.rl[i];
        }
        return dsv4_fp8_mx_launch(a, st);
    }
    if (fp8_geom(cols, &g) && blocking_ok(blk_r, blk_c)) {
        if (chunked_ok(x, W, "fp8 gemv") != 0) return -1;
        /* launch shape (fp8_valu): none of it changes a row's arithmetic */
        const Fp8Valu v = fp8_valu(rows, cols, blk_r, sfmt);
        const int R = v.R, pf = v.pf, wpc = v.wpc;
        if (sfmt == 0) {
            if (pf) launch_gemv_r<0, 1>(g, R, y, x, W, S, rows, cols, sc, blk_r, blk_c, wpc, gp, st);
            else    launch_gemv_r<0, 0>(g, R, y, x, W, S, rows, cols, sc, blk_r, blk_c, wpc, gp, st);
        } else {
            if (pf) launch_gemv_r<1, 1>(g, R, y, x, W, S, rows, cols, sc, blk_r, blk_c, wpc, gp, st);
            else    launch_gemv_r<1, 0>(g, R, y, x, W, S, rows, cols, sc, blk_r, blk_c, wpc, gp, st);
        }
    } else {
        const int grid = (rows + 3) / 4;
        for (int i = 0; i < gp.n; i++) {
            float *yi = y + i * gp.y;
            const float *xi = x + i * gp.x;
            const uint8_t *Wi = W + i * gp.w;
            const void *Si = (const uint8_t *)S + i * gp.s;
            if (sfmt == 0)
                hipLaunchKernelGGL((k_fp8_gemv_generic<0>), dim3(grid), dim3(256), 0, st,
                                   yi, xi, Wi, Si, rows, cols, sc, blk_r, blk_c, 1);
            else
                hipLaunchKernelGGL((k_fp8_gemv_generic<1>), dim3(grid), dim3(256), 0, st,
                                   yi, xi, Wi, Si, rows, cols, sc, blk_r, blk_c, 1);
        }
    }
    HIP_OK(hipGetLastError(), "fp8 gemv launch");
    return 0;
}

/* The attention block's x projections in one launch: its listed FP8
 * matrices (blockIdx.y < gp.n) run k_fp8_gemv's body, its listed BF16
 * matrices the BF16 GEMV's (dsv4_bf16_rows.h); all read the same x. Each
 * part keeps its own launch plan, so every row has the bits of its own
 * GEMV; workgroups past a part's grid leave at once. */
struct XProj {
    const float *x = nullptr;
    int cols = 0;
    Fp8Groups gp;                                  /* FP8: list of gp.n */
    int rows8 = 0, sc = 0, blk_r = 0, blk_c = 0, tc8 = 0, rpw8 = 0, grid8 = 0;
    B16List ls;                                    /* BF16: list of ls.n */
    int tc16 = 0, rpw16 = 0, grid16 = 0;
};

template <int NCH, int R, int SF, int PF, int BNCH, int BR>
__global__ void __launch_bounds__(256)
k_xproj(XProj a)
{
    extern __shared__ float part[];
    const int bx = blockIdx.x, by = blockIdx.y;
    if (by < a.gp.n) {
        if (bx >= a.grid8) return;
        /* (the list supplies each matrix's W, S, y and rows) */
        fp8_rows<NCH, R, SF, PF, 0>(a.gp.yl[0], a.x, a.gp.Wl[0], a.gp.Sl[0], a.rows8, a.cols,
                                    a.sc, a.blk_r, a.blk_c, a.tc8, a.rpw8, a.gp, bx, by, part);
    } else {
        if (bx >= a.grid16) return;
        b16_rows<BNCH, BR>(a.ls.y[0], a.x, a.ls.W[0], a.ls.rows[0], a.cols, a.tc16, a.rpw16,
                           a.ls, bx, by - a.gp.n, part);
    }
}

/* The attention block's q GEMVs and the rest of its prep step in one
 * launch: its listed FP8 matrices (blockIdx.y < gp.n; wq_b and the indexer's
 * wq_b) read qr and normalise their workgroup's copy of it themselves (the
 * prep step's q job, same arithmetic and order: NQ), and the workgroups of
 * row gp.n run the prep step's other jobs (the ring slot's norm and RoPE,
 * the compressor's slot), which nothing in this launch reads. */
struct QProj {
    const float *x = nullptr, *nw = nullptr;
    int cols = 0;
    float eps = 0.0f;
    Fp8Groups gp;
    int rows8 = 0, sc = 0, blk_r = 0, blk_c = 0, tc8 = 0, rpw8 = 0, grid8 = 0;
    Dsv4Prep prep{};
    int nprep = 0;
};

template <int NCH, int R, int SF>
__global__ void __launch_bounds__(256)
k_qproj(QProj a)
{
    extern __shared__ float part[];
    const int bx = blockIdx.x, by = blockIdx.y;
    if (by < a.gp.n) {
        if (bx >= a.grid8) return;
        fp8_rows<NCH, R, SF, 0, 1, 1>(a.gp.yl[0], a.x, a.gp.Wl[0], a.gp.Sl[0], a.rows8, a.cols,
                                      a.sc, a.blk_r, a.blk_c, a.tc8, a.rpw8, a.gp, bx, by, part,
                                      a.nw, a.eps);
    } else {
        if (bx >= a.nprep) return;
        prep_rows(a.prep, bx);
    }
}

} // namespace

int dsv4_fp8_gemv_launch(float *y, const float *x, const uint8_t *W,
                         const void *S, int sfmt, int rows, int cols,
                         int blk_r, int blk_c, hipStream_t st, bool valu)
{
    Fp8Groups gp;
    gp.valu = valu;
    return fp8_gemv(y, x, W, S, sfmt, rows, cols, blk_r, blk_c, gp, st);
}

int dsv4_fp8_gemv_list_launch(const float *x, int cols, int sfmt, int blk_r, int blk_c,
                              int n, const uint8_t *const *W, const void *const *S,
                              float *const *y, const int *rows, hipStream_t st, bool valu)
{
    if (n < 1 || n > FP8_LIST_MAX) {
        DSV4_ERR("fp8 gemv list: %d matrices (1 .. %d)", n, FP8_LIST_MAX);
        return -1;
    }
    Fp8Groups gp;
    gp.n = n;
    gp.list = 1;
    gp.valu = valu;
    int rmax = 0;
    for (int i = 0; i < n; i++) {
        if (rows[i] <= 0 || (((uintptr_t)W[i]) & 15)) {
            DSV4_ERR("fp8 gemv list: matrix %d (%d rows) empty or unaligned", i, rows[i]);
            return -1;
        }
        gp.Wl[i] = W[i]; gp.Sl[i] = S[i]; gp.yl[i] = y[i]; gp.rl[i] = rows[i];
        rmax = rows[i] > rmax ? rows[i] : rmax;
    }
    Fp8Geom g;
    if (!fp8_geom(cols, &g) || !blocking_ok(blk_r, blk_c) || (((uintptr_t)x) & 15)) {
        for (int i = 0; i < n; i++)
            if (dsv4_fp8_gemv_launch(y[i], x, W[i], S[i], sfmt, rows[i], cols, blk_r, blk_c,
                                     st, valu) != 0)
                return -1;
        return 0;
    }
    return fp8_gemv(y[0], x, W[0], S[0], sfmt, rmax, cols, blk_r, blk_c, gp, st);
}

int dsv4_fp8_gemv_groups_launch(float *y, const float *x, const uint8_t *W,
                                const void *S, int sfmt, int rows, int cols, int blk_r,
                                int blk_c, int groups, long long y_stride,
                                long long x_stride, long long w_stride,
                                long long s_stride, hipStream_t st, bool valu)
{
    Fp8Groups gp;
    gp.n = groups;
    gp.valu = valu;
    gp.y = y_stride; gp.x = x_stride; gp.w = w_stride; gp.s = s_stride;
    if (groups > 1 && (((uintptr_t)(x_stride * 4) | (uintptr_t)w_stride) & 15)) {
        DSV4_ERR("fp8 gemv groups: strides break 16-byte alignment");
        return -1;
    }
    return fp8_gemv(y, x, W, S, sfmt, rows, cols, blk_r, blk_c, gp, st);
}

bool dsv4_fp8_mx_form(int sfmt, int cols, int blk_r, int blk_c)
{
    return mx_form(sfmt, cols, blk_r, blk_c);
}

/* The split tiles' block sums (mf_split): on 256 CUs at most 128 tiles of 256
 * results, 4 sums of each, or of rows of 192 threads 336 tiles, 3 of each. */
size_t dsv4_fp8_n_split_bytes(int rows, int cols, int nt)
{
    Fp8Geom g;
    if (rows <= 0 || nt < 2 || !fp8_geom(cols, &g)) return 0;
    const int z = mf_split(g, rows, nt);
    return z == 1 ? 0 : sizeof(float) * (size_t)std::max(z, g.tc / 64) * nt * rows;
}

size_t dsv4_fp8_n_scratch_bytes(int rows, int cols, int nt)
{
    return std::max(dsv4_fp8_mxn_scratch_bytes(cols, nt), dsv4_fp8_n_split_bytes(rows, cols, nt));
}

int dsv4_fp8_gemv_n_launch(float *y, const float *x, const uint8_t *W,
                           const void *S, int sfmt, int rows, int cols,
                           int blk_r, int blk_c, int nt, hipStream_t st, void *xscratch)
{
    if (rows <= 0 || cols <= 0 || nt <= 0 || blk_r <= 0 || blk_c <= 0) {
        DSV4_ERR("fp8 gemv_n: bad shape %dx%d nt %d", rows, cols, nt);
        return -1;
    }
    if (nt == 1)                       /* the GEMV itself: same bits, its launch shape */
        return fp8_gemv(y, x, W, S, sfmt, rows, cols, blk_r, blk_c, Fp8Groups{}, st);
    if (mx_form(sfmt, cols, blk_r, blk_c)) {
        if (chunked_ok(x, W, "fp8 gemv_n") != 0) return -1;
        return dsv4_fp8_mxn_launch(y, x, W, (const uint8_t *)S, rows, cols, blk_r, blk_c, nt,
                                   st, xscratch);
    }
    const int sc = (cols + blk_c - 1) / blk_c;
    Fp8Geom g;
    if (fp8_geom(cols, &g) && blocking_ok(blk_r, blk_c)) {
        if (chunked_ok(x, W, "fp8 gemv_n") != 0) return -1;
        if ((sfmt == 0 ? launch_gemv_n<0>(g, y, x, W, S, rows, cols, sc, blk_r, blk_c, nt, st,
                                          xscratch)
                       : launch_gemv_n<1>(g, y, x, W, S, rows, cols, sc, blk_r, blk_c, nt, st,
                                          xscratch)) != 0)
            return -1;
    } else {
        const int grid = (rows + 3) / 4;
        if (sfmt == 0)
            hipLaunchKernelGGL((k_fp8_gemv_generic<0>), dim3(grid), dim3(256), 0, st,
                               y, x, W, S, rows, cols, sc, blk_r, blk_c, nt);
        else
            hipLaunchKernelGGL((k_fp8_gemv_generic<1>), dim3(grid), dim3(256), 0, st,
                               y, x, W, S, rows, cols, sc, blk_r, blk_c, nt);
    }
    HIP_OK(hipGetLastError(), "fp8 gemv_n launch");
    return 0;
}

int dsv4_xproj_launch(const float *x, int cols, int sfmt, int blk_r, int blk_c, int nf,
                      const uint8_t *const *Wf, const void *const *Sf, float *const *yf,
                      const int *rf, int nb, const uint16_t *const *Wb, float *const *yb,
                      const int *rb, hipStream_t st)
{
    auto two = [&]() -> int {
        if (nf > 0 &&
            dsv4_fp8_gemv_list_launch(x, cols, sfmt, blk_r, blk_c, nf, Wf, Sf, yf, rf, st,
                                      true) != 0)
            return -1;
        if (nb > 0 && dsv4_bf16_gemv_list_launch(x, cols, nb, Wb, yb, rb, st) != 0) return -1;
        return 0;
    };
    if (nf < 1 || nb < 1 || nf > FP8_LIST_MAX || nb > B16_LIST_MAX ||
        (sfmt != 0 && sfmt != 1) || env_int("DSV4_GPU_XPROJ", 1) == 0)
        return two();
    Fp8Geom g;
    B16Geom gb;
    bool ok = fp8_geom(cols, &g) && blocking_ok(blk_r, blk_c) && b16_geom(cols, &gb) &&
              (((uintptr_t)x) & 15) == 0;
    int rmf = 0, rmb = 0;
    for (int i = 0; i < nf; i++) {
        ok = ok && rf[i] > 0 && (((uintptr_t)Wf[i]) & 15) == 0;
        rmf = rf[i] > rmf ? rf[i] : rmf;
    }
    for (int i = 0; i < nb; i++) {
        ok = ok && rb[i] > 0 && (((uintptr_t)Wb[i]) & 15) == 0;
        rmb = rb[i] > rmb ? rb[i] : rmb;
    }
    if (!ok) return two();
    const Fp8Valu v = fp8_valu(rmf, cols, blk_r, sfmt, false);
    const Fp8Plan pf = fp8_plan(g, v.R, v.pf, sfmt, rmf, cols, v.wpc, nf, false);
    /* the BF16 part within the FP8 part's grid (DSV4_GPU_XPROJ_CAP=0: its own
     * plan): a wider x grid only adds workgroups of one step each */
    const B16Plan pb = b16_plan(gb, rmb, nb, env_int("DSV4_GPU_XPROJ_CAP", 1) ? pf.grid : 0);
    /* the one combination built: FP8 with 4 chunks per thread, 2 rows per
     * step, prefetch, x in registers (through LDS the step measured slower:
     * ratio 128 at 2200 positions 48.9 / 49.5 us, ratio 4 71.9 / 72.0; the
     * second step's weights are then requested only after the first's
     * arrive); BF16 with 8 chunks per thread, 1 row (hidden 4096 and 7168,
     * the Flash and full shapes) */
    if (g.nch < 4 || v.R != 2 || !v.pf || cols >= 16384 || gb.nch <= 4 || pb.R != 1 ||
        g.wg != 256 || gb.wg != 256)
        return two();
    XProj a;
    a.x = x;
    a.cols = cols;
    a.gp.n = nf;
    a.gp.list = 1;
    a.gp.valu = true;
    for (int i = 0; i < nf; i++) {
        a.gp.Wl[i] = Wf[i]; a.gp.Sl[i] = Sf[i]; a.gp.yl[i] = yf[i]; a.gp.rl[i] = rf[i];
    }
    a.rows8 = rmf; a.sc = (cols + blk_c - 1) / blk_c; a.blk_r = blk_r; a.blk_c = blk_c;
    a.tc8 = g.tc; a.rpw8 = pf.rows_per_wg; a.grid8 = pf.grid;
    a.ls.n = nb;
    for (int i = 0; i < nb; i++) {
        a.ls.W[i] = Wb[i]; a.ls.y[i] = yb[i]; a.ls.rows[i] = rb[i];
    }
    a.tc16 = gb.tc; a.rpw16 = pb.rows_per_wg; a.grid16 = pb.grid;
    const dim3 grid(pf.grid > pb.grid ? pf.grid : pb.grid, nf + nb);
    const size_t lds = pf.lds > pb.lds ? pf.lds : pb.lds;
    if (sfmt == 0)
        hipLaunchKernelGGL((k_xproj<4, 2, 0, 1, 8, 1>), grid, dim3(256), lds, st, a);
    else
        hipLaunchKernelGGL((k_xproj<4, 2, 1, 1, 8, 1>), grid, dim3(256), lds, st, a);
    HIP_OK(hipGetLastError(), "x projections launch");
    return 0;
}

int dsv4_qproj_launch(const float *qr, int cols, const float *nw, float eps, int sfmt,
                      int blk_r, int blk_c, int nf, const uint8_t *const *Wf,
                      const void *const *Sf, float *const *yf, const int *rf,
                      const Dsv4Prep *prep, hipStream_t st)
{
    if (!prep || prep->nj > 1 || nf < 1 || nf > FP8_LIST_MAX) {
        DSV4_ERR("q projections: bad arguments (%d matrices)", nf);
        return -1;
    }
    /* the separate form: the prep step with the q job first, then the list */
    auto two = [&]() -> int {
        Dsv4Prep p = *prep;
        if (p.nj == 1) p.job[1] = p.job[0];
        p.job[0] = Dsv4NormJob{const_cast<float *>(qr), qr, nw, cols, 0};
        p.nj = prep->nj + 1;
        if (dsv4_block_prep_launch(&p, st) != 0) return -1;
        return dsv4_fp8_gemv_list_launch(qr, cols, sfmt, blk_r, blk_c, nf, Wf, Sf, yf, rf, st,
                                         true);
    };
    Fp8Geom g;
    bool ok = env_int("DSV4_GPU_QPROJ", 1) != 0 && (sfmt == 0 || sfmt == 1) && nw &&
              fp8_geom(cols, &g) && blocking_ok(blk_r, blk_c) && (((uintptr_t)qr) & 15) == 0;
    int rm = 0;
    for (int i = 0; i < nf; i++) {
        ok = ok && rf[i] > 0 && (((uintptr_t)Wf[i]) & 15) == 0;
        rm = rf[i] > rm ? rf[i] : rm;
    }
    if (!ok) return two();
    const Fp8Valu v = fp8_valu(rm, cols, blk_r, sfmt, false);
    /* rows per step: 4 (a step stays in one row block), or 2. Four measured
     * faster for the block's q GEMVs (wq_b 32768x1024 and the indexer's
     * 8192x1024 with the prep step: 77.1 -> 74.9 us per CSA step); one row
     * with no prefetch in the x launch measured slower (78.7), so that
     * launch keeps two rows with prefetch. */
    const int qrr = env_int("DSV4_GPU_QPROJ_R", 4) >= 4 && blk_r % 4 == 0 ? 4 : 2;
    /* each matrix the grid it would have alone, not a share of one: each
     * workgroup's norm stands between its first weights and the rest, and
     * the more of them there are the more weights are in flight meanwhile
     * (the CSA step above 75.6 -> 73.8 us). */
    const Fp8Plan pf = fp8_plan(g, qrr, 0, sfmt, rm, cols, v.wpc, 1);
    /* the combinations built: x through LDS, 1 or 2 chunks
     * per thread, 2 or 4 rows per step, no prefetch (wq_b's rows), 256
     * threads */
    if (!pf.xl || g.wg != 256 || g.nch > 2 || v.R != 2 || v.pf) return two();
    QProj a;
    a.x = qr; a.nw = nw; a.cols = cols; a.eps = eps;
    a.gp.n = nf; a.gp.list = 1; a.gp.valu = true;
    for (int i = 0; i < nf; i++) {
        a.gp.Wl[i] = Wf[i]; a.gp.Sl[i] = Sf[i]; a.gp.yl[i] = yf[i]; a.gp.rl[i] = rf[i];
    }
    a.rows8 = rm; a.sc = (cols + blk_c - 1) / blk_c; a.blk_r = blk_r; a.blk_c = blk_c;
    a.tc8 = g.tc; a.rpw8 = pf.rows_per_wg; a.grid8 = pf.grid;
    a.prep = *prep;
    a.nprep = prep_wgs(*prep);
    const dim3 grid(pf.grid > a.nprep ? pf.grid : a.nprep, nf + (a.nprep ? 1 : 0));
    static bool opted = false;
    const size_t lds = pf.lds + sizeof(float) * (size_t)cols;   /* + the norm's weights */
    if (!opted) {
        const size_t cap = dsv4_lds_limit();
        const void *fns[] = {(const void *)k_qproj<1, 2, 0>, (const void *)k_qproj<2, 2, 0>,
                             (const void *)k_qproj<1, 2, 1>, (const void *)k_qproj<2, 2, 1>,
                             (const void *)k_qproj<1, 4, 0>, (const void *)k_qproj<2, 4, 0>,
                             (const void *)k_qproj<1, 4, 1>, (const void *)k_qproj<2, 4, 1>};
        for (const void *f : fns) (void)dsv4_lds_optin(f, cap, "q projections");
        opted = true;
    }
#define DSV4_QP(NCH, R, SF) hipLaunchKernelGGL((k_qproj<NCH, R, SF>), grid, dim3(256), lds, st, a)
    if (qrr == 4) {
        if (sfmt == 0) { if (g.nch == 1) DSV4_QP(1, 4, 0); else DSV4_QP(2, 4, 0); }
        else           { if (g.nch == 1) DSV4_QP(1, 4, 1); else DSV4_QP(2, 4, 1); }
    } else {
        if (sfmt == 0) { if (g.nch == 1) DSV4_QP(1, 2, 0); else DSV4_QP(2, 2, 0); }
        else           { if (g.nch == 1) DSV4_QP(1, 2, 1); else DSV4_QP(2, 2, 1); }
    }
#undef DSV4_QP
    HIP_OK(hipGetLastError(), "q projections launch");
    return 0;
}
