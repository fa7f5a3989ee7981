/* SPDX-License-Identifier: Apache-2.0 */
/* dsv4_batch_mf.hip - the batched GEMVs (prefill: y[nt][rows] for x[nt][cols])
 * of FP8, BF16 and MXFP4 matrices on gfx950's f32 matrix core, each (row,
 * token) with the bits of the single-token GEMV of its format
 * (dsv4_fp8.hip, dsv4_bf16.hip, dsv4_fp4.hip).
 *
 * HOW THE BITS ARE KEPT. A single-token GEMV gives each of a row's tc threads
 * ("slots") the 16-byte chunks j, j + tc, ...; a chunk's elements are dotted
 * in a few interleaved f32 chains (a product, then fmaf), the chains are
 * added in a fixed tree, the chunk joins the slot's sum, and the slots meet
 * in a balanced tree within 64 and in order across the 64s. Measured on the
 * device (2^21 outputs with normal, wide-exponent, cancelling and subnormal
 * operands and -0.0 addends), v_mfma_f32_16x16x4f32 computes each output as
 * the sequential fmaf chain over its four k in ascending order from C,
 * without flushing subnormals. So four consecutive terms of a chain are one
 * MFMA (A[row][k] = w, B[k][token] = x; C = -0.0 for a chain's start, since
 * fmaf(a, b, -0.0) is a * b), and the VALU does the adds in the GEMV's order:
 *   FP8   chunk of 16: 4 chains (elements c, c+4, c+8, c+12), one MFMA each;
 *         (p0 + p1) + (p2 + p3), fmaf with the chunk's scale into the slot.
 *   BF16  chunk of 8: 2 chains (even, odd elements), one MFMA each; p0 + p1
 *         added into the slot.
 *   FP4   chunk of 32: 4 chains of 8, two MFMAs each; joined as FP8's.
 *
 * WHAT BOUNDS IT. The f32 matrix core and the VALU share the SIMD's FP32
 * pipes: a compute-only loop takes 32.4 cycles (2.4 GHz) per MFMA, and 43.4
 * with FP8's or BF16's 4 VALU operations per MFMA beside it (2 or more waves
 * per SIMD; 54 with one). At 7168x7168 and 64 tokens that is 57 us, of 81.5
 * measured (122 with the same chains staged through registers and a workgroup
 * barrier per step): the rest is the operands' decode and the starts and ends
 * of 7 workgroups per CU. A grid of one workgroup per CU that walks its tiles
 * without emptying its stages measured slower (99 us): two waves per SIMD do
 * not cover each other's waits. Batches of few tiles are bound by one tile's
 * chain, about 3.6 us + 1.6 ns per column (2048x7168 FP4 at 24 tokens 102 ->
 * 16.4 us, 1024x4096 BF16 at 48 tokens 66 -> 10.9).
 *
 * LAYOUT. A workgroup is P waves for one tile of 16 rows and 16 tokens; wave p
 * walks the row's slots [p L, p L + L), L = tc / P, four at a time. Splitting
 * the slots over the waves keeps the GEMV's tree: a wave forms its aligned
 * block's subtree, and the P subtrees meet in LDS after one barrier, in the
 * tree's order. A step is four consecutive slots at one n: 64 bytes of each
 * row and the 16 tokens' x of those chunks, copied by direct-to-LDS loads into
 * the wave's own ring of two stages, so no wave waits for another. (Operand
 * loads in the matrix core's order, straight into registers, ran 7168x7168 at
 * 120 us: four neighbouring lanes then read four different rows, one cache
 * line each per cycle.) A step's operands are read from LDS into one register
 * set while the step before, in the other, is computed. Lane (row r, k group
 * g) reads chunk g of its row whole; four v_permlane swaps hand every lane
 * its group's piece of each chunk. */
#include "dsv4_dev.h"
#include "dsv4_internal.h"

namespace {

#include "dsv4_batch_walk.h"

enum { MF_E8M0 = 0, MF_F32S = 1, MF_BF16 = 2, MF_FP4 = 3 };

struct MfArgs {
    float *y;
    const float *x;
    const uint8_t *W;
    const void *S;
    int rows, cols, nt;
    int ch, tc, nch, L;          /* the GEMV's geometry; slots per wave       */
    uint32_t nch_m;              /* ceil(2^16 / nch)                          */
    int sc, blk_r, blk_c;        /* scale grid (not BF16)                     */
    int P, Z;                    /* waves per workgroup, workgroups per tile  */
    float *part;                 /* Z > 1: the workgroups' block sums         */
    uint32_t bc_m;               /* ceil(2^32 / blk_c): a column's block is a multiply */
};

template <int FMT> constexpr int mf_elems() { return FMT == MF_BF16 ? 8 : FMT == MF_FP4 ? 32 : 16; }

__device__ __forceinline__ void swap32(uint32_t &a, uint32_t &b)
{
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = r[0];
    b = r[1];
}
__device__ __forceinline__ void swap16(uint32_t &a, uint32_t &b)
{
    const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    a = r[0];
    b = r[1];
}

/* Lane group g holds chunk g's four dwords. FP8, BF16: o[q] = dword g of
 * chunk q. FP4: o[q] = the dword that holds its elements 4g..4g+3, o[4 + q]
 * the one that holds 16+4g..16+4g+3 (in the low or, for odd g, high half). */
template <int FMT>
__device__ __forceinline__ void spread(const u32x4 v, uint32_t *o)
{
    uint32_t a = v.x, b = v.y, c = v.z, d = v.w;
    if (FMT == MF_FP4) {
        swap32(a, b);
        swap32(c, d);
        o[0] = a; o[1] = a; o[2] = b; o[3] = b;
        o[4] = c; o[5] = c; o[6] = d; o[7] = d;
        swap16(o[0], o[1]);
        swap16(o[2], o[3]);
        swap16(o[4], o[5]);
        swap16(o[6], o[7]);
        return;
    }
    swap32(a, c);
    swap32(b, d);
    swap16(a, b);
    swap16(c, d);
    o[0] = a; o[1] = b; o[2] = c; o[3] = d;
}

/* The balanced sum of N waves' values of one result. */
template <int N>
__device__ __forceinline__ float tree(const float *v)
{
    if constexpr (N == 1) return v[0];
    else return tree<N / 2>(v) + tree<N / 2>(v + N / 2 * 256);
}

typedef __attribute__((address_space(3))) void lds_void;

/* The instructions that copy one part's x of a step (1 KiB each). */
template <int FMT> constexpr int mf_nxi() { return FMT == MF_BF16 ? 2 : FMT == MF_FP4 ? 8 : 4; }

/* 16 bytes per lane from base + off + soff (inside its `bytes`) to dst + 16
 * lane in LDS, without passing through registers. */
__device__ __forceinline__ void copy16(const void *base, uint32_t bytes, unsigned char *dst,
                                       int off, int soff)
{
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, (int)bytes, 0x00020000),
        (lds_void *)dst, 16, off, soff, 0, 0);
}

template <int N>
__device__ __forceinline__ void vm_wait()
{
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

/* FMT; SC1: a step's four chunks share one scale (FP8,
 * blk_c a multiple of 64) or, FP4, their scale bytes are one aligned dword of
 * each row (1x32 blocks, cols a multiple of 128); FULL: ch % 4 == 0, so a step
 * is wholly inside the row. */
template <int FMT, bool SC1, bool FULL>
__global__ void __launch_bounds__(FMT == MF_FP4 ? 512 : 1024)
k_batch_mf(const MfArgs a)
{
    constexpr int CE = mf_elems<FMT>(), NXI = mf_nxi<FMT>();
    constexpr int NX = FMT == MF_FP4 ? 2 : 1;              /* x pieces per chunk and lane */
    constexpr bool F8 = FMT == MF_E8M0 || FMT == MF_F32S;
    constexpr int DP = 2;                                  /* stages in the ring */
    constexpr int DPW = NXI + 1;                           /* copies per step */
    constexpr int SB = DPW * 1024;                         /* bytes per stage */
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const int lane = threadIdx.x & 63;
    const int p = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int P = a.P;
    const int r = lane & 15, g = lane >> 4;
    /* grid (8 Z, token tiles, row tiles / 8): the token tiles of a row tile
     * are 8 Z workgroups apart, so on one XCD and at about the same time */
    const int z = (int)blockIdx.x >> 3;
    const int t0 = (int)blockIdx.y * 16;
    const int row0 = (int)(blockIdx.z * 8 + (blockIdx.x & 7)) * 16;
    if (row0 >= a.rows) return;                            /* the whole workgroup */
    const int ch = a.ch, tc = a.tc, nch = a.nch;
    const int j0 = (z * P + p) * a.L;                      /* this wave's slots */
    unsigned char *const ring = lds + p * (DP * SB);       /* its own stages */

    /* the copies: lane -> (row lane / 4, slot lane % 4) of the weights' 64
     * bytes per row, (token, slot) of x; the piece in a slot is XORed with
     * the row or token so that the operand reads below fall in distinct
     * banks. Buffer loads: a lane offset formed once, the step's column as
     * the scalar offset; the descriptors end with the matrix and with x. */
    const size_t rowb = (size_t)ch * 16;
    const uint8_t *const Wt = a.W + (size_t)row0 * rowb;
    const float *const Xt = a.x + (size_t)t0 * a.cols;
    const uint32_t wbytes = (uint32_t)min((size_t)(a.rows - row0) * rowb, (size_t)0xFFFFFFFFu);
    const uint32_t xbytes = (uint32_t)(a.nt - t0) * (uint32_t)a.cols * 4u;
    const int wrow = lane >> 2, wpc = (lane & 3) ^ ((lane >> 4) & 3);
    const int wo = min(wrow, a.rows - 1 - row0) * (int)rowb + (FULL ? wpc * 16 : 0);
    constexpr int LPT = 4 * NXI;                           /* lanes per token */
    int xo[NXI], xe[NXI];
#pragma unroll
    for (int k = 0; k < NXI; k++) {
        const int t = k * (64 / LPT) + lane / LPT, sl = lane % LPT;
        const int pc = sl ^ (FMT == MF_BF16 ? (t >> 1) & 7 : t);
        xe[k] = 16 * pc;
        xo[k] = min(t, a.nt - 1 - t0) * a.cols * 4 + (FULL ? 16 * pc : 0);
    }
    auto issue = [&](int c, int slot) {
        unsigned char *st = ring + slot * SB;
        copy16(Wt, wbytes, st + NXI * 1024,
               FULL ? wo : wo + min(c + wpc, ch - 1) * 16, FULL ? c * 16 : 0);
#pragma unroll
        for (int k = 0; k < NXI; k++)
            copy16(Xt, xbytes, st + 1024 * k,
                   FULL ? xo[k] : xo[k] + min(c * CE * 4 + xe[k], a.cols * 4 - 16),
                   FULL ? c * CE * 4 : 0);
    };

    /* a wave's steps (dsv4_batch_walk.h) */
    const int U = a.L >> 2, steps = mf_steps(j0, a.L, tc, ch, nch);

    /* (the chunk and ring slot of the next copy, of the next step) */
    int cu = 0, cc = j0, cs = 0, ci = 0;
    auto request = [&]() {
        issue(cc, cs);
        cs = cs + 1 == DP ? 0 : cs + 1;
        if (cc + tc < ch) cc += tc;
        else cc = j0 + 4 * ++cu;
        ci++;
    };
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < DP; s++)
        if (ci < steps) request();
    __builtin_amdgcn_sched_barrier(0);

    /* the scales. FP8: lane i holds those of the wave's group i = u nch + n
     * (the tile's rows share theirs: blk_r % 16 == 0), read by readlane.
     * FP4: bf16 (exact for a power of two) in LDS, [group][k group g][chunk]
     * [row 4g + e], so a lane's 16 of a step are 32 consecutive bytes. */
    const int groups = U * nch;                            /* <= 64 for FP8 */
    constexpr int NS = SC1 ? 1 : 4;
    uint32_t sr[NS];
    unsigned char *const sl4 = lds + P * (DP * SB) + p * groups * 128;
    auto chunk_of = [&](int i) {                           /* group i's first chunk */
        const int u = (int)(((uint32_t)i * a.nch_m) >> 16);
        return j0 + 4 * u + (i - u * nch) * tc;
    };
    if (F8) {
        const uint32_t so = (uint32_t)(row0 / a.blk_r) * (uint32_t)a.sc;
        const int c = chunk_of(min(lane, groups - 1));
#pragma unroll
        for (int q = 0; q < NS; q++) {
            const uint32_t at = so + __umulhi((uint32_t)(min(c + q, ch - 1) * 16), a.bc_m);
            sr[q] = FMT == MF_E8M0 ? __float_as_uint(dec_e8m0(((const uint8_t *)a.S)[at]))
                                   : ((const uint32_t *)a.S)[at];
        }
    } else if (FMT == MF_FP4) {
        const uint8_t *S = (const uint8_t *)a.S;
        const size_t so = (size_t)(min(row0 + r, a.rows - 1) / a.blk_r) * (size_t)a.sc;
        for (int i = lane >> 4; i < groups; i += 4) {      /* row r, group i */
            const int c = min(chunk_of(i), ch - 1);
            uint32_t b[4];
            if (SC1) {
                const uint32_t v = *reinterpret_cast<const uint32_t *>(S + so + (c & ~3));
#pragma unroll
                for (int q = 0; q < 4; q++) b[q] = (v >> (8 * q)) & 0xFF;
            } else {
#pragma unroll
                for (int q = 0; q < 4; q++)
                    b[q] = S[so + __umulhi((uint32_t)(min(c + q, ch - 1) * 32), a.bc_m)];
            }
#pragma unroll
            for (int q = 0; q < 4; q++)
                *reinterpret_cast<uint16_t *>(sl4 + i * 128 + (r >> 2) * 32 + q * 8 + (r & 3) * 2) =
                    (uint16_t)(__float_as_uint(dec_e8m0(b[q])) >> 16);
        }
    }

    /* the operand reads: lane (row or token r, k group g) */
    int xa[4 * NX];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        if (FMT == MF_BF16)
            xa[q] = r * 128 + (((2 * q + (g >> 1)) ^ (r >> 1)) & 7) * 16 + 8 * (g & 1);
        else
#pragma unroll
            for (int k = 0; k < NX; k++)
                xa[q * NX + k] = r * (64 * NXI) + ((4 * (NX * q + k) + g) ^ r) * 16;
    }
    const int wa = NXI * 1024 + r * 64 + ((g ^ (r >> 2)) & 3) * 16;

    const f32x4 negz = {-0.0f, -0.0f, -0.0f, -0.0f};
    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    f32x4 A[4], h[4], res;
    /* a group's four slots summed, then a binary counter over the groups:
     * after the last group res is the wave's subtree */
    auto join = [&](int u) {
        f32x4 v = (A[0] + A[1]) + (A[2] + A[3]);
        if (!(u & 1)) h[0] = v;
        else {
            v = h[0] + v;
            if (!(u & 2)) h[1] = v;
            else {
                v = h[1] + v;
                if (!(u & 4)) h[2] = v;
                else {
                    v = h[2] + v;
                    if (!(u & 8)) h[3] = v;
                    else v = h[3] + v;
                }
            }
        }
        res = v;
#pragma unroll
        for (int q = 0; q < 4; q++) A[q] = zero;
    };
#pragma unroll
    for (int q = 0; q < 4; q++) A[q] = zero;

    /* A step's operands are read into one register set while the step before
     * it, in the other, is computed; its slot is then free for the copies
     * of the step DP ahead. */
    struct Ops {
        u32x4 w, s4[2];
        f32x4 x[4][NX];
    } fe, fo;
    MfWalk rd(j0);                                         /* the next step to read */
    int rs = 0, ri = 0;
    auto fetch = [&](Ops &f) {
        /* its copies have arrived; those of the steps after it may be in
         * flight (past the last step: a read of what lies there, so that
         * every pass makes the same reads and the waits count them) */
        if (steps - 1 - ri >= 1) vm_wait<DPW>();
        else vm_wait<0>();
        const unsigned char *st = ring + rs * SB;
        f.w = *reinterpret_cast<const u32x4 *>(st + wa);
#pragma unroll
        for (int q = 0; q < 4; q++) {
            if (FMT == MF_BF16) {
                typedef float f32x2 __attribute__((ext_vector_type(2)));
                const f32x2 t = *reinterpret_cast<const f32x2 *>(st + xa[q]);
                f.x[q][0].x = t.x;
                f.x[q][0].y = t.y;
            } else {
#pragma unroll
                for (int k = 0; k < NX; k++)
                    f.x[q][k] = *reinterpret_cast<const f32x4 *>(st + xa[q * NX + k]);
            }
        }
        if (FMT == MF_FP4) {
            const unsigned char *const s4 = sl4 + rd.entry(nch, groups) * 128 + g * 32;
            f.s4[0] = *reinterpret_cast<const u32x4 *>(s4);
            f.s4[1] = *reinterpret_cast<const u32x4 *>(s4 + 16);
        }
        rs = rs + 1 == DP ? 0 : rs + 1;
        ri++;
        rd.next(j0, tc, ch);
    };

    int u = 0, n = 0, c0 = j0;
    auto step = [&](Ops &f, Ops &nx) {
        /* f is here, so its slot is free */
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (ci < steps) request();
        fetch(nx);
        float sf[NS];
        if (F8) {
#pragma unroll
            for (int q = 0; q < NS; q++)
                sf[q] = __uint_as_float(__builtin_amdgcn_readlane(sr[q], u * nch + n));
        }
        uint32_t d[FMT == MF_FP4 ? 8 : 4];
        spread<FMT>(f.w, d);
        /* chunk q's chains on the matrix core */
        auto mm = [&](int q, f32x4 *o) {
            if (FMT == MF_BF16) {
                o[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(d[q] << 16),
                                                            f.x[q][0].x, negz, 0, 0, 0);
                o[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(d[q] & 0xFFFF0000u),
                                                            f.x[q][0].y, negz, 0, 0, 0);
            } else {
                float wf[8];
                if (F8) {
                    dec_e4m3x4(d[q], wf);
                } else {
                    const uint32_t v = d[q] >> (16 * (g & 1));
                    const uint32_t v2 = d[(FMT == MF_FP4 ? 4 : 0) + q] >> (16 * (g & 1));
                    dec_fp4x2<0>(v, wf);
                    dec_fp4x2<1>(v, wf + 2);
                    dec_fp4x2<0>(v2, wf + 4);
                    dec_fp4x2<1>(v2, wf + 6);
                }
#pragma unroll
                for (int k = 0; k < 4; k++)
                    o[k] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[k], f.x[q][0][k], negz, 0, 0, 0);
                if (FMT == MF_FP4) {
#pragma unroll
                    for (int k = 0; k < 4; k++)
                        o[k] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[4 + k], f.x[q][NX - 1][k],
                                                                    o[k], 0, 0, 0);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        /* chunk q's chains into its slot */
        auto va = [&](int q, const f32x4 *o) {
            if (!FULL && c0 + q >= ch) return;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                if (FMT == MF_BF16) {
                    A[q][e] = A[q][e] + (o[0][e] + o[1][e]);
                } else {
                    const float dt = (o[0][e] + o[1][e]) + (o[2][e] + o[3][e]);
                    float sc;
                    if (F8) {
                        sc = sf[SC1 ? 0 : q];
                    } else {
                        const uint32_t v = f.s4[q >> 1][2 * (q & 1) + (e >> 1)];
                        sc = __uint_as_float(e & 1 ? v & 0xFFFF0000u : v << 16);
                    }
                    A[q][e] = fmaf(dt, sc, A[q][e]);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        /* a chunk's chains issued ahead of the additions of the chunk before
         * it, whose results they give time to arrive */
        f32x4 oe[4], oo[4];
        mm(0, oe);
        mm(1, oo);
        va(0, oe);
        mm(2, oe);
        va(1, oo);
        mm(3, oo);
        va(2, oe);
        va(3, oo);
        n++;
        c0 += tc;
        if (c0 >= ch) {
            join(u);
            u++;
            n = 0;
            c0 = j0 + 4 * u;
        }
    };
    fetch(fe);
    for (int s = 0; s < (steps >> 1); s++) {
        step(fe, fo);
        step(fo, fe);
    }
    if (steps & 1) step(fe, fo);
    for (; u < U; u++) join(u);                            /* groups past the row: zeros */

    /* result (row 4g + e, token r) of the tile at 64 e + lane, in the ring */
    __syncthreads();
    float *const red = reinterpret_cast<float *>(lds);
#pragma unroll
    for (int e = 0; e < 4; e++) red[(p * 4 + e) * 64 + lane] = res[e];
    __syncthreads();
    const int pb = min(P, 64 / a.L);                       /* waves per 64-slot block */
    for (int i = threadIdx.x; i < 256; i += (int)blockDim.x) {
        /* thread -> (token, row): neighbours write neighbouring rows */
        const int rr = i & 15, t = i >> 4;
        const float *v = red + (rr & 3) * 64 + (rr >> 2) * 16 + t;
        const int row = row0 + rr, tok = t0 + t;
        const bool in = row < a.rows && tok < a.nt;
        float out = 0.0f;
        for (int k = 0; k < P; k += pb) {
            const float *vk = v + k * 256;
            const float b = pb == 1 ? vk[0] : pb == 2 ? tree<2>(vk) : pb == 4 ? tree<4>(vk)
                          : pb == 8 ? tree<8>(vk) : tree<16>(vk);
            out = k == 0 ? b : out + b;
            if (a.Z > 1 && in)
                a.part[((size_t)(z * (P / pb) + k / pb) * a.nt + tok) * a.rows + row] = b;
        }
        if (a.Z == 1 && in) a.y[(size_t)tok * a.rows + row] = out;
    }
}

/* The rest of the slot tree per (row, token) from the n sums of `slots`
 * aligned slots each: within each 64-slot block the balanced tree, then the
 * blocks in order. */
__global__ void __launch_bounds__(256)
k_batch_mf_join(float *__restrict__ y, const float *__restrict__ part, int count, int n, int slots)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= count) return;
    const int pb = min(n, 64 / slots);
    float out = 0.0f;
    for (int k0 = 0; k0 < n; k0 += pb) {
        const float *v = part + (size_t)k0 * count + i;
        float b = v[0];
        if (pb == 2) b = v[0] + v[count];
        else if (pb == 4) b = (v[0] + v[count]) + (v[2 * (size_t)count] + v[3 * (size_t)count]);
        out = k0 == 0 ? b : out + b;
    }
    y[i] = out;
}

template <int FMT, bool SC1, bool FULL>
int mf_go(const MfArgs &a, dim3 grid, size_t lds, hipStream_t st)
{
    static bool opted = false;
    if (!opted) {
        (void)dsv4_lds_optin((const void *)k_batch_mf<FMT, SC1, FULL>, dsv4_lds_limit(),
                             "batched gemv");
        opted = true;
    }
    hipLaunchKernelGGL((k_batch_mf<FMT, SC1, FULL>), grid, dim3(64 * a.P), lds, st, a);
    HIP_OK(hipGetLastError(), "batched gemv (matrix core) launch");
    return 0;
}

template <int FMT>
int mf_fmt(MfArgs &a, bool sc1, bool full, hipStream_t st)
{
    constexpr int NXI = mf_nxi<FMT>();
    const dim3 grid(8 * a.Z, (a.nt + 15) / 16, ((a.rows + 15) / 16 + 7) / 8);
    if (grid.z > 65535) return 1;
    const size_t lds = 2 * (size_t)a.P * (NXI + 1) * 1024 +
                       (FMT == MF_FP4 ? (size_t)a.P * (a.L / 4) * a.nch * 128 : 0);
    if (lds > dsv4_lds_limit()) return 1;
    if constexpr (FMT != MF_BF16)
        if (!sc1) return mf_go<FMT, false, false>(a, grid, lds, st);
    return full ? mf_go<FMT, true, true>(a, grid, lds, st)
                : mf_go<FMT, true, false>(a, grid, lds, st);
}

/* The waves a row tile's slots are split over. While every tile has a CU to
 * itself the most (16; 8 for FP4, whose two register sets take 173 to 185
 * VGPRs, too many for two such workgroups on a CU): a tile's time is its own
 * chain (us, P 16 / 8: FP8 2048x4096 at 16 tokens 11.1 / 11.4, BF16 1024x4096
 * at 48 10.9 / 12.2, 1024x7168 16.6 / 18.9). With more tiles, fewer, so that
 * several workgroups share a CU's LDS and one starts while another ends (FP8
 * 7168x7168 at 64 tokens P 16 / 8 / 4: 100.6 / 81.5 / 84.2, 24576x1536 at 64
 * 116.5 / 71.3 / 67.5; BF16 16384x4096 at 64 162.2 / 123.9 / 117.4; FP4 P 8 /
 * 4: 8192x8192 at 64 129.7 / 108.9).
 * 192 slots divide into 12, 6 or 3 waves, of which 6 leave the LDS of half a
 * CU unused: 12 up to three rounds of tiles, then 3 (us, P 12 / 6 / 3: 3072x
 * 12288 at 48 tokens, 576 tiles, 70.7 / 79.5 / 84.3; 4096x12288 at 64, 1024
 * tiles, 94.7 / 123.6 / 85.6); rows whose chunks do not end on a step (!full)
 * keep 6 in the third round (12288x8208 at 16 59.6 / 57.4). Split over three
 * workgroups (mf_split in dsv4_fp8.hip) with more tiles than CUs, 4 each
 * (5120x12288 at 16 tokens P 16 / 8 / 4 / 2: 45.6 / 36.1 / 34.6 / 37.3). */
int mf_waves(int fmt, int tc, bool full, bool split, long long tiles)
{
    if (tiles <= 256) return fmt == MF_FP4 ? 8 : 16;
    if (fmt == MF_FP4) return 4;
    if (fmt == MF_BF16) return tiles <= 512 ? 8 : 4;
    if (tc == 192) return split ? 4 : tiles <= (full ? 800 : 512) ? 12 : tiles <= 800 ? 8 : 3;
    return tc < 64 || (tc == 64 && tiles > 2048) ? 4 : 8;
}

} // namespace

/* Rows of 192 slots: with the row tiles rounded up to the grid's eight per
 * XCD, as one more than an XCD's CUs is a second round there (1360x12288 at 33
 * tokens, 255 tiles: 45.6 us unsplit). */
long long dsv4_batch_mf_tiles(int rows, int nt, int tc)
{
    const long long rt = ((long long)rows + 15) / 16;
    return (tc == 192 ? (rt + 7) / 8 * 8 : rt) * ((nt + 15) / 16);
}

int dsv4_batch_mf_launch(const Dsv4BatchMf &b, hipStream_t st)
{
    const int ce = b.fmt == MF_BF16 ? 8 : b.fmt == MF_FP4 ? 32 : 16;
    if (b.cols % ce || b.tc < 4 || (b.tc & 3) || (((uintptr_t)b.x | (uintptr_t)b.W) & 15) ||
        b.rows <= 0 || b.nt <= 0 || b.tc > 256 ||
        (b.tc < 64 ? (b.tc & (b.tc - 1)) != 0 : b.tc % 64 != 0))
        return 1;
    MfArgs a;
    a.y = b.y; a.x = b.x; a.W = (const uint8_t *)b.W; a.S = b.S;
    a.rows = b.rows; a.cols = b.cols; a.nt = b.nt;
    a.ch = b.cols / ce; a.tc = b.tc;
    a.nch = (a.ch + a.tc - 1) / a.tc;
    a.nch_m = (65536u + a.nch - 1) / a.nch;
    a.sc = b.sc; a.blk_r = b.blk_r; a.blk_c = b.blk_c;
    const bool f8 = b.fmt == MF_E8M0 || b.fmt == MF_F32S;
    if (f8 && (b.blk_r & 15)) return 1;
    /* P waves per row tile (mf_waves): the smallest part of at least 4 slots,
     * at most the 64 of one block of the tree */
    const int Z = b.split > 1 && b.part ? b.split : 1;
    const bool full = a.ch % 4 == 0;
    const int want = mf_waves(b.fmt, a.tc, full, Z > 1, dsv4_batch_mf_tiles(b.rows, b.nt, a.tc));
    int L = 4;
    while (a.tc / L / Z > want && 2 * L <= 64 && 2 * L <= a.tc) L *= 2;
    if (b.slots) L = b.slots;
    if (L < 4 || L > 64 || L > a.tc || (L & (L - 1)) || a.tc % L) return 1;
    /* a workgroup's slots (of a split tile: whole 64-slot blocks of the
     * tree, or an aligned part of one) */
    const int sw = a.tc / Z, P = sw / L;
    if (P < 1 || P * L * Z != a.tc || (Z > 1 && sw % 64 != 0 && (sw < 16 || 64 % sw != 0)))
        return 1;
    if (P > (b.fmt == MF_FP4 ? 8 : 16) || (f8 && L / 4 * a.nch > 64)) return 1;
    a.L = L;
    a.P = P; a.Z = Z;
    a.part = b.part;
    a.bc_m = b.blk_c > 0 ? (uint32_t)(((1ull << 32) + b.blk_c - 1) / b.blk_c) : 0;
    const bool sc1 = b.fmt == MF_BF16 ||
                     (f8 ? b.blk_c % 64 == 0
                         : full && b.blk_r == 1 && b.blk_c == 32 && (((uintptr_t)b.S) & 3) == 0);
    int rc;
    switch (b.fmt) {
    case MF_E8M0: rc = mf_fmt<MF_E8M0>(a, sc1, full, st); break;
    case MF_F32S: rc = mf_fmt<MF_F32S>(a, sc1, full, st); break;
    case MF_BF16: rc = mf_fmt<MF_BF16>(a, sc1, full, st); break;
    default: rc = mf_fmt<MF_FP4>(a, sc1, full, st); break;
    }
    if (rc != 0 || Z == 1) return rc;
    const int n = sw >= 64 ? b.tc / 64 : Z, count = b.nt * b.rows;   /* sums, of tc / n slots */
    hipLaunchKernelGGL(k_batch_mf_join, dim3((count + 255) / 256), dim3(256), 0, st, b.y, b.part,
                       count, n, b.tc / n);
    HIP_OK(hipGetLastError(), "batched gemv join launch");
    return 0;
}
