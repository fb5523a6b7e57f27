/* SPDX-License-Identifier: Unlicense
 *
 * Exact-path (fp32 operand) GEMM on gfx950:
 *   C = act(alpha * A * op(B) + bias) + R     (sam3_kernels.cl:57-69)
 * with float A and C and float or half B: large products on the bf16 matrix
 * cores from split operands (k_gemm_frag, k_gemm_split), small ones on the
 * f32 MFMA with K spread over waves (k_gemm_small_f32). launch_gemm_split
 * chooses; what it does not take (unaligned or bf16 operands, bf16 C) stays
 * with k_gemm_f32.
 *
 * The split. The f32 MFMA peaks at 157 TFLOP/s, the bf16 MFMA at sixteen
 * times that. A float x in bf16 pieces: x0 the rounding of x to bf16, x1 that
 * of x - x0, x2 what is left, 8 + 8 + 8 mantissa bits: |x1| <= 2^-8 |x|, |x2| <=
 * 2^-16 |x|, roundings to nearest, so the pieces' signs are unbiased. bf16
 * has the float's exponents, so the lowest piece of a float below 2^-109 would
 * fall out of its range: floats are scaled by 2^24 first (SPLIT_SCALE),
 * which leaves every bit of every float, subnormals too, at 2^-125 or above,
 * and the sums are scaled back. So three pieces are exactly the float for
 * every |x| < 2^103; larger ones overflow (below). Of the nine products of
 * two split values the six of order 2^-16 and above are formed on the bf16
 * MFMA with f32 accumulation; the three dropped ones are below 2^-24 of the
 * product (2^-27 in the mean), less than the rounding of one f32 fused
 * multiply-add. A half is exactly two pieces (five products), unscaled.
 * Rounding the accumulator six times per 16 k instead of once per two, the
 * result is no further from the 64-bit product than the f32 MFMA's in
 * k_gemm_f32: relative error 1.1e-7 against 1.4e-7 at K = 64, 2.4e-7 against
 * 2.9e-7 at 256, 4.9e-7 against 5.7e-7 at 1024, 1.0e-6 against 1.15e-6 at
 * 4096; the small kernel's split sums 1.5e-7 (256) and 2.9e-7 (2048, 8.1e-7
 * before).
 *
 * A non-finite operand, or one past 2^103, makes its pieces, and so every
 * output it enters, NaN; a sum past 2^80 overflows. A 32 x 32 block with a
 * non-finite output is formed again from the float operands by the f32 MFMA
 * (block_f32) and those outputs taken from there, so infinities and NaN
 * travel as in k_gemm_f32 and a product full of NaN costs what the f32 unit
 * costs, not a serial sum per output.
 *
 * LDS holds MFMA fragments: per 32 rows, 16 k and piece 1 KiB of 64 chunks
 * of 16 bytes (8 k of one row), chunk 32 (k half) + row, so that a fragment
 * read is linear in the lane.
 */
#include "k_common.h"

#include <type_traits>

#define GS_K 16   /* K per step */
/* Steps of a packed operand: K rounded up to 64 (zeros). */
#define GS_STEPS(K) (((K) + 63) / 64 * 4)
#define GS_NXCD 8 /* XCDs (L2 domains) of an MI355X */
#define GS_BAND 8 /* tile rows walked together */
#define GS_XCD_TILES 64 /* fewest tiles dealt to the XCDs in ranges */

/* LDS byte offset, in its piece's 1 KiB, of k quad q (4 k, 0..3) of row r
 * of a 32-row block. */
__device__ __forceinline__ int frag_off(int r, int q)
{
    const int h = q >> 1;

    return 16 * (32 * h + (r ^ (4 * h))) + 8 * (q & 1);
}

/* A 32 x 32 block of the product by the f32 MFMA from the float operands:
 * lane l's row of A and column of B are l % 32 of the block's; a lane half
 * takes four consecutive k of every eight (K % 4 == 0: in or out together). */
template <int BDT>
__device__ __noinline__ f32x16 block_f32(const float *a, const void *b, long bstep, int K)
{
    const int h = (threadIdx.x & 63) >> 5;
    f32x16 acc = {};

#pragma unroll 1
    for (int k0 = 0; k0 < K; k0 += 8) {
        const int k = k0 + 4 * h;
        f32x4 x = {}, y = {};

        if (k < K) {
            x = *(const f32x4 *)(a + k);
            for (int e = 0; e < 4; e++)
                y[e] = BDT == DT_F32 ? ((const float *)b)[(k + e) * bstep]
                                     : h2f(((const uint16_t *)b)[(k + e) * bstep]);
        }
#pragma unroll
        for (int e = 0; e < 4; e++)
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(x[e], y[e], acc, 0, 0, 0);
    }
    return acc;
}

/* Epilogue (store_one, sam3_kernels.cl:306-319) of a wave's 32 NA x 32 NB
 * part of C from (m0, n0), 32 lanes to 128 contiguous bytes of a row: act(alpha
 * v + bias) + R of the sums scaled back, the non-finite v taken from
 * block_f32. arow(m), bcol(n): row
 * m of A, column n of B; C and R at the matrix's element 0. */
template <int BDT, int NA, int NB, class ROW, class COL>
__device__ __forceinline__ void store_blocks(const gemm_desc &d, f32x16 (&acc)[NA][NB], int m0,
                                             int n0, float *C, const float *R, ROW arow, COL bcol)
{
    const int l = threadIdx.x & 63, h = l >> 5, l32 = l & 31;

#pragma unroll
    for (int j = 0; j < NB; j++) {
        const int n = n0 + 32 * j + l32;
        float bn = d.bias && n < d.N ? d.bias[n] : 0.0f;

        /* The load is waited for here, once: at its first use, in a branch
         * per result, the wait came back in every branch and took in the
         * store of the one before (1 us per tile). */
        asm volatile("" : "+v"(bn));
#pragma unroll
        for (int i = 0; i < NA; i++) {
            const int mb = m0 + 32 * i;
            unsigned long long bad = 0;
            float alpha = d.alpha * split_unscale<BDT>;

#pragma unroll
            for (int r = 0; r < 16; r++)
                bad |= __ballot(!(fabsf(acc[i][j][r]) < __builtin_inff()));
            if (bad) {
                const f32x16 x = block_f32<BDT>(arow(min(mb + l32, d.M - 1)),
                                                bcol(min(n, d.N - 1)), d.transb ? 1L : d.ldb, d.K);

#pragma unroll
                for (int r = 0; r < 16; r++)
                    acc[i][j][r] = fabsf(acc[i][j][r]) < __builtin_inff()
                                       ? acc[i][j][r] * split_unscale<BDT>
                                       : x[r];
                alpha = d.alpha;
            }
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int m = mb + 8 * (r >> 2) + 4 * h + (r & 3);
                float v = acc[i][j][r];

                if (m >= d.M || n >= d.N)
                    continue;
                v = act_k(alpha * v + bn, d.act);
                if (R)
                    v += R[(long)m * d.ldc + n];
                C[(long)m * d.ldc + n] = v;
            }
        }
    }
}

/* Operands split while they are staged: a workgroup owns a BM x BN tile of
 * C, each wave WM x WN of it as 32 x 32 accumulators. K moves in steps of
 * 16: beside a step's MFMAs from one LDS slot, the next step's floats,
 * loaded into registers a step earlier, are split and written to the other
 * slot (k half 1's chunks at row ^ 4, which keeps the staging writes, 4 rows
 * x 16 k per 16 lanes, off each other's banks), and the loads of the step
 * after go out: one barrier per step.
 *
 * Bound by issue: a split costs 22 VALU instructions per four floats, and on
 * this chip VALU and MFMA time add up rather than overlap (165888 x 128 x
 * 256: 40 % and 30 % of the SIMD cycles, the rest waits), so it is used where
 * a float meets few columns and splitting it in a pass of its own would cost
 * more: the decoder's image tokens, 331776 x 128 x 256, 189 us against 254 by
 * k_gemm_f32; 165888 rows 87 us, 168 with the pass. */
template <int BM, int BN, int WM, int WN, int BDT, bool TRANSB>
__global__ __launch_bounds__((BM / WM) * (BN / WN) * 64, 1) void k_gemm_split(gemm_desc d)
{
    constexpr int NW = (BM / WM) * (BN / WN), T = NW * 64;
    constexpr int NA = WM / 32, NB = WN / 32;
    constexpr int NPB = BDT == DT_F32 ? 3 : 2; /* pieces of B */
    constexpr int ABYTES = BM / 32 * 3 * 1024, BBYTES = BN / 32 * NPB * 1024;
    constexpr int SLOT = ABYTES + BBYTES;
    constexpr int LA = BM * 4 / T, LB = BN * 4 / T; /* k quads per thread */
    static_assert(BM * 4 % T == 0 && BN * 4 % T == 0, "staging split");
    __shared__ __attribute__((aligned(16))) char S[2 * SLOT];
    const int t = threadIdx.x, l = t & 63, w = t >> 6, h = l >> 5, l32 = l & 31;
    const int wm = w / (BN / WN), wn = w % (BN / WN);
    const int tn = (d.N + BN - 1) / BN, tm = (d.M + BM - 1) / BM;
    const int total = tn * tm, per = (total + GS_NXCD - 1) / GS_NXCD;
    /* Workgroup g runs on XCD g % 8: contiguous tiles per XCD, in bands of
     * GS_BAND tile rows, so that its L2 serves a window of A and B rows. Few
     * tiles (of each of a batch) are taken as they come: rounding their
     * number up to the XCDs would launch mostly empty workgroups (1000
     * products of 16 x 16 x 16: 33 us against 10). */
    const int tile = total < GS_XCD_TILES
                         ? (int)blockIdx.x
                         : (int)(blockIdx.x % GS_NXCD) * per + blockIdx.x / GS_NXCD;

    if (tile >= total)
        return;
    const int band = tile / (GS_BAND * tn), rem = tile - band * GS_BAND * tn;
    const int brows = min(GS_BAND, tm - band * GS_BAND);
    const int m0 = (band * GS_BAND + rem % brows) * BM, n0 = rem / brows * BN;
    const long z0 = blockIdx.z / d.nb1, z1 = blockIdx.z % d.nb1;
    const long abase = d.aoff + z0 * d.sa0 + z1 * d.sa1;
    const long bbase = d.boff + z0 * d.sb0 + z1 * d.sb1;
    const int nk = (d.K + GS_K - 1) / GS_K;
    f32x16 acc[NA][NB];
    f32x4 ra[LA], rb[LB];
    u32x2 hb[LB]; /* B's quads as loaded (half N x K operand) */
    const float *pa[LA];
    long ob[LB];

#pragma unroll
    for (int i = 0; i < NA; i++)
#pragma unroll
        for (int j = 0; j < NB; j++)
            acc[i][j] = (f32x16){};
    /* Quad i of thread t: row (t + T i) / 4, k quad t % 4; four lanes read a
     * row's 64 bytes. Rows past M or N read the last one (never stored). A
     * K x N B is read with lanes along n: column (t + T i) % BN, quad
     * (t + T i) / BN. */
#pragma unroll
    for (int i = 0; i < LA; i++)
        pa[i] = (const float *)d.A + abase + (long)min(m0 + (t + T * i) / 4, d.M - 1) * d.lda +
                4 * (t & 3);
#pragma unroll
    for (int i = 0; i < LB; i++)
        ob[i] = TRANSB ? bbase + (long)min(n0 + (t + T * i) / 4, d.N - 1) * d.ldb + 4 * (t & 3)
                       : bbase + min(n0 + (t + T * i) % BN, d.N - 1);

    /* The floats of step ks; `last` (a constant): the step may be partial,
     * its k past K are zero. */
    auto load = [&](int ks, auto last) {
        const int k0 = ks * GS_K;
        const bool in = !decltype(last)::value || k0 + 4 * (t & 3) < d.K;

#pragma unroll
        for (int i = 0; i < LA; i++)
            ra[i] = in ? *(const f32x4 *)(pa[i] + k0) : (f32x4){};
#pragma unroll
        for (int i = 0; i < LB; i++) {
            if constexpr (TRANSB) {
                if constexpr (BDT == DT_F32)
                    rb[i] = in ? *(const f32x4 *)((const float *)d.B + ob[i] + k0) : (f32x4){};
                else
                    hb[i] = in ? *(const u32x2 *)((const uint16_t *)d.B + ob[i] + k0) : (u32x2){};
            }
            else {
                const int q = (t + T * i) / BN;

                for (int e = 0; e < 4; e++) {
                    const int k = k0 + 4 * q + e;
                    const bool kin = !decltype(last)::value || k < d.K;
                    const long bi = ob[i] + (long)(kin ? k : 0) * d.ldb;
                    const float v = BDT == DT_F32 ? ((const float *)d.B)[bi]
                                                  : h2f(((const uint16_t *)d.B)[bi]);

                    rb[i][e] = kin ? v : 0.0f;
                }
            }
        }
    };
    auto stage = [&](int slot) {
        char *s = S + slot * SLOT;

#pragma unroll
        for (int i = 0; i < LA; i++) {
            const int row = (t + T * i) / 4;
            char *p = s + (row >> 5) * 3072 + frag_off(row & 31, t & 3);
            u32x2 v[3];

            split4<3>(ra[i] * SPLIT_SCALE, v);
            for (int e = 0; e < 3; e++)
                *(u32x2 *)(p + 1024 * e) = v[e];
        }
#pragma unroll
        for (int i = 0; i < LB; i++) {
            const int row = TRANSB ? (t + T * i) / 4 : (t + T * i) % BN;
            const int q = TRANSB ? t & 3 : (t + T * i) / BN;
            char *p = s + ABYTES + (row >> 5) * NPB * 1024 + frag_off(row & 31, q);
            u32x2 v[NPB];

            /* Converted here, not where they are loaded: there the compiler
             * may convert at once and wait for the load (37 against 47 us,
             * 4298 x 321 x 888). */
            if constexpr (TRANSB && BDT == DT_F16)
                for (int e = 0; e < 4; e++)
                    rb[i][e] = h2f((uint16_t)(hb[i][e >> 1] >> (16 * (e & 1))));
            split4<NPB>(BDT == DT_F32 ? rb[i] * SPLIT_SCALE : rb[i], v);
            for (int e = 0; e < NPB; e++)
                *(u32x2 *)(p + 1024 * e) = v[e];
        }
    };
    const int fo = 16 * (32 * h + (l32 ^ (4 * h)));
    auto products = [&](int slot) {
        const char *sa = S + slot * SLOT + wm * NA * 3072 + fo;
        const char *sb = S + slot * SLOT + ABYTES + wn * NB * NPB * 1024 + fo;
        bf16x8 a[NA][3], b[NB][NPB];

#pragma unroll
        for (int i = 0; i < NA; i++)
#pragma unroll
            for (int e = 0; e < 3; e++)
                a[i][e] = *(const bf16x8 *)(sa + 3072 * i + 1024 * e);
#pragma unroll
        for (int j = 0; j < NB; j++)
#pragma unroll
            for (int e = 0; e < NPB; e++)
                b[j][e] = *(const bf16x8 *)(sb + NPB * 1024 * j + 1024 * e);
        /* Piece pairs (a, b) with a + b <= 2, in k_gemm_frag's order: the
         * two kernels give the same bits. */
        constexpr int pairs[6][2] = {{2, 0}, {1, 1}, {1, 0}, {0, 2}, {0, 1}, {0, 0}};

#pragma unroll
        for (int p = 0; p < 6; p++) {
            if (pairs[p][1] >= NPB)
                continue;
#pragma unroll
            for (int i = 0; i < NA; i++)
#pragma unroll
                for (int j = 0; j < NB; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                        a[i][pairs[p][0]], b[j][pairs[p][1]], acc[i][j], 0, 0, 0);
        }
    };

    const std::false_type whole;
    const std::true_type last;
    /* Step ks from slot ks % 2 beside the staging of step ks + 1 and the
     * loads of step ks + 2, in one basic block. */
    auto step = [&](int ks, auto slot) {
        constexpr int s = decltype(slot)::value;

        __syncthreads();
        /* Nothing of the staging moves up between the products of the step
         * before: its wait for the loads would come with it (344 x 2919 x
         * 1732: 70 -> 63 us, half B 56 -> 47). Not with a K x N half B, whose
         * single-element loads gain by moving (50 x 3179 x 3232: 124 -> 112). */
        if constexpr (BDT == DT_F32 || TRANSB)
            __builtin_amdgcn_sched_barrier(0);
        stage(s ^ 1);
        load(ks + 2, whole);
        products(s);
    };

    if (nk > 1)
        load(0, whole);
    else
        load(0, last);
    stage(0);
    if (nk > 2)
        load(1, whole);
    else if (nk > 1)
        load(1, last);
    int ks = 0;

    for (; ks + 4 < nk; ks += 2) {
        step(ks, std::integral_constant<int, 0>());
        step(ks + 1, std::integral_constant<int, 1>());
    }
    for (; ks < nk; ks++) {
        __syncthreads();
        if (ks + 1 < nk) {
            stage((ks + 1) & 1);
            if (ks + 2 < nk)
                load(ks + 2, last);
        }
        products(ks & 1);
    }

    store_blocks<BDT, NA, NB>(
        d, acc, m0 + wm * WM, n0 + wn * WN, (float *)d.C + d.coff + z0 * d.sc0 + z1 * d.sc1,
        d.R ? (const float *)d.R + d.roff + z0 * d.sc0 + z1 * d.sc1 : nullptr,
        [&](int m) { return (const float *)d.A + abase + (long)m * d.lda; },
        [&](int n) {
            return (const char *)d.B +
                   (BDT == DT_F32 ? 4 : 2) * (bbase + n * (TRANSB ? (long)d.ldb : 1L));
        });
}

/* ------------------------------------------------------------ packed */

/* Large products split their operands in a pass of their own (k_split_pack:
 * 10 bytes moved per element, 12-40 us for the trunk's), so that the K loop
 * is MFMAs, fragment reads and asynchronous copies only (k_gemm_frag). At
 * 5184 rows, pass included, against k_gemm_f32 and against the split while
 * staging: 1024 -> 3072 158 us, 301, 215 (206 TFLOP/s); 1024 -> 4096 232, 446,
 * 289; 4096 -> 1024 280, 672, 310; 1024 -> 1024 78, 180, 85; half weights 135,
 * 190, 237 and 68 us. What bounds it is the MFMA rate under its own power: the
 * MFMA unit is busy 70 % of the cycles, 225 TFLOP/s of six products are 1350
 * TFLOP/s of bf16, 93 % of what the platform's 8192^3 bf16 product reaches.
 */

/* An operand split once into MFMA fragments: [32-row block][16-k step]
 * [piece][64 chunks of 16 bytes], chunk 32 (k half) + row % 32; rows and k
 * past the matrix are zero. */
struct frag_src {
    const void *src; /* element 0 of the operand */
    long ld;
    int rows, K, kmajor; /* kmajor: element (r, k) at k ld + r, else r ld + k */
    char *dst;
    int win_H, win_ws, win_nwx, win_m0; /* gemm_desc's (A only; win_ws 0: rows as they lie) */
};

/* Window-partition position of grid token t (k_window_unpartition_add's). */
__device__ __forceinline__ long win_row(int t, int H, int ws, int nwx)
{
    const int y = t / H, x = t - y * H, wy = y / ws, wx = x / ws;

    return ((long)wy * nwx + wx) * ws * ws + (y - wy * ws) * ws + (x - wx * ws);
}

/* 32 rows x 64 k per 256-thread workgroup: eight lanes read 256 contiguous
 * bytes of a row (or, k-major, 32 lanes 128 contiguous bytes of a k), the
 * pieces go through LDS (chunk position xored with the k octet against bank
 * conflicts) and leave as contiguous fragments. */
template <int DT, int NP, bool WIN>
__device__ __forceinline__ void pack_block(const frag_src &f, int blk, char *S)
{
    const int t = threadIdx.x, nks = GS_STEPS(f.K), nkc = nks / 4;
    const int rb = blk / nkc, kc = blk % nkc;
    const int r = f.kmajor ? t & 31 : t >> 3, k8 = f.kmajor ? t >> 5 : t & 7;
    const int row = rb * 32 + r, k0 = kc * 64 + k8 * 8;
    f32x4 x[2] = {};

    if (row < f.rows) {
        const long srow =
            WIN ? win_row(f.win_m0 + row, f.win_H, f.win_ws, f.win_nwx) : row;
        const long i0 = f.kmajor ? (long)k0 * f.ld + row : srow * f.ld + k0;

        if (!f.kmajor && k0 + 8 <= f.K) {
            if constexpr (DT == DT_F32) {
                x[0] = ((const f32x4 *)((const float *)f.src + i0))[0];
                x[1] = ((const f32x4 *)((const float *)f.src + i0))[1];
            }
            else {
                const u32x2 *v = (const u32x2 *)((const uint16_t *)f.src + i0);

                for (int j = 0; j < 2; j++)
                    for (int e = 0; e < 4; e++)
                        x[j][e] = h2f((uint16_t)(v[j][e >> 1] >> (16 * (e & 1))));
            }
        }
        else
            for (int e = 0; e < 8; e++)
                if (k0 + e < f.K) {
                    const long i = i0 + (f.kmajor ? e * f.ld : e);

                    x[e >> 2][e & 3] = DT == DT_F32 ? ((const float *)f.src)[i]
                                                    : h2f(((const uint16_t *)f.src)[i]);
                }
    }
    u32x2 lo[NP], hi[NP];
    const float scale = DT == DT_F32 ? SPLIT_SCALE : 1.0f;

    split4<NP>(x[0] * scale, lo);
    split4<NP>(x[1] * scale, hi);
    for (int p = 0; p < NP; p++) {
        const int c = (32 * (k8 & 1) + r) ^ k8;

        *(u32x4 *)(S + ((k8 >> 1) * NP + p) * 1024 + 16 * c) =
            (u32x4){lo[p].x, lo[p].y, hi[p].x, hi[p].y};
    }
    __syncthreads();
    const int frags = NP * 4;
    char *dst = f.dst + ((long)rb * nks + 4 * kc) * NP * 1024;

    for (int i = t; i < frags * 64; i += 256) {
        const int fr = i >> 6, c = i & 63, k = 2 * (fr / NP) + (c >> 5);

        *(u32x4 *)(dst + 16L * i) = *(const u32x4 *)(S + fr * 1024 + 16 * (c ^ k));
    }
}

/* WIN: A's rows are taken from their windows. */
template <int BDT, bool WIN>
__global__ __launch_bounds__(256) void k_split_pack(frag_src a, frag_src b, int ablocks)
{
    __shared__ __attribute__((aligned(16))) char S[4 * 3 * 1024];

    if ((int)blockIdx.x < ablocks)
        pack_block<DT_F32, 3, WIN>(a, blockIdx.x, S);
    else
        pack_block<BDT, BDT == DT_F32 ? 3 : 2, false>(b, blockIdx.x - ablocks, S);
}

__device__ __forceinline__ void gs_vmwait0()
{
    asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
}

/* A workgroup owns a BM x BN tile, each wave WM x WN; per step of 16 k the
 * fragments of the tile's rows and columns go HBM -> LDS asynchronously into
 * one of two slots, a step ahead. The loop is one basic block (the step count
 * is even; copies past the end repeat the last step into a slot that no one
 * reads): with a branch in it the compiler kept a second copy of the
 * accumulators, 128 moves per step (145 against 180 TFLOP/s). Registers are
 * kept to what two 256 x 128 workgroups on a CU leave (5184 x 4096 x 1024 with
 * GELU: 250 us, 259 with one). */
template <int BM, int BN, int WM, int WN, int BDT, bool WIN>
__global__ __launch_bounds__((BM / WM) * (BN / WN) * 64, BM * BN >= 256 * 128 ? 4 : 1) void
k_gemm_frag(gemm_desc d, const char *pa, const char *pb)
{
    constexpr int NW = (BM / WM) * (BN / WN), NSLOT = 2;
    constexpr int NA = WM / 32, NB = WN / 32;
    constexpr int NPB = BDT == DT_F32 ? 3 : 2;
    constexpr int AFR = BM / 32 * 3, FR = AFR + BN / 32 * NPB; /* fragments per step */
    constexpr int CPW = (FR + NW - 1) / NW;                    /* copies per wave */
    constexpr int SLOT = FR * 1024;
    __shared__ __attribute__((aligned(16))) char S[NSLOT * SLOT];
    const int t = threadIdx.x, l = t & 63;
    const int wu = __builtin_amdgcn_readfirstlane(t >> 6);
    const int wm = wu / (BN / WN), wn = wu % (BN / WN);
    const int tn = (d.N + BN - 1) / BN, tm = (d.M + BM - 1) / BM;
    const int total = tn * tm, per = (total + GS_NXCD - 1) / GS_NXCD;
    const int tile = (int)(blockIdx.x % GS_NXCD) * per + blockIdx.x / GS_NXCD;

    if (tile >= total)
        return;
    constexpr int GR = 4;
    const int band = tile / (GR * tn), rem = tile - band * GR * tn;
    const int brows = min(GR, tm - band * GR);
    const int m0 = (band * GR + rem % brows) * BM, n0 = rem / brows * BN;
    const int nk = GS_STEPS(d.K);
    const int amax = (d.M - 1) / 32, bmax = (d.N - 1) / 32;
    const char *src[CPW];
    unsigned step[CPW], lds[CPW];

    /* Copy i of wave w: fragment w + NW i of the step (the last ones may
     * repeat fragment FR - 1); row blocks past the matrix read the last
     * (never stored). */
#pragma unroll
    for (int i = 0; i < CPW; i++) {
        const int f = min(wu + NW * i, FR - 1);
        const bool isa = f < AFR;
        const int np = isa ? 3 : NPB, g = isa ? f : f - AFR;
        const int rb = isa ? min(m0 / 32 + g / 3, amax) : min(n0 / 32 + g / NPB, bmax);

        src[i] = (isa ? pa : pb) + ((long)rb * nk * np + g % np) * 1024;
        step[i] = np * 1024u;
        lds[i] = (unsigned)(uintptr_t)S + 1024u * f;
    }
    const unsigned voff = 16u * l;
    /* Copies of step ks (past the last: the last again, into a slot that no
     * one reads any more, so that the loop has no branch). */
    auto load = [&](int ks, int slot) {
        const long kc = min(ks, nk - 1);

#pragma unroll
        for (int i = 0; i < CPW; i++)
            g2lds16(src[i] + kc * step[i], voff, lds[i] + (unsigned)SLOT * slot);
    };
    f32x16 acc[NA][NB];
#pragma unroll
    for (int i = 0; i < NA; i++)
#pragma unroll
        for (int j = 0; j < NB; j++)
            acc[i][j] = (f32x16){};
    const char *sa = S + wm * NA * 3072 + 16 * l;
    const char *sb = S + AFR * 1024 + wn * NB * NPB * 1024 + 16 * l;
    bf16x8 a[3][NA], b[NPB][NB];
    auto rda = [&](int slot, int p) {
#pragma unroll
        for (int i = 0; i < NA; i++)
            a[p][i] = *(const bf16x8 *)(sa + SLOT * slot + 3072 * i + 1024 * p);
    };
    auto rdb = [&](int slot, int p) {
#pragma unroll
        for (int j = 0; j < NB; j++)
            b[p][j] = *(const bf16x8 *)(sb + SLOT * slot + NPB * 1024 * j + 1024 * p);
    };
    auto mm = [&](int p, int q) {
#pragma unroll
        for (int i = 0; i < NA; i++)
#pragma unroll
            for (int j = 0; j < NB; j++)
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[p][i], b[q][j], acc[i][j],
                                                                    0, 0, 0);
    };

    /* Step ks from slot `sl`: its first fragments (a[2], b[0]) are in
     * registers. Once the others are too, the slot goes to the copies of
     * step ks + 2 and the next step's first fragments are read under the
     * last products. */
    auto body = [&](int ks, auto slot) {
        constexpr int sl = decltype(slot)::value, sn = (sl + 1) % NSLOT;

        rda(sl, 1);
        rdb(sl, 1);
        mm(2, 0);
        rda(sl, 0);
        if constexpr (NPB == 3)
            rdb(sl, 2);
        mm(1, 1);
        mm(1, 0);
        if constexpr (NPB == 3)
            mm(0, 2);
        mm(0, 1);
        gs_vmwait0();
        __syncthreads();
        load(ks + NSLOT, sl);
        rda(sn, 2);
        mm(0, 0);
        rdb(sn, 0);
    };

    load(0, 0);
    gs_vmwait0();
    __syncthreads();
    load(1, 1);
    rda(0, 2);
    rdb(0, 0);
    for (int ks = 0; ks < nk; ks += NSLOT) {
        body(ks, std::integral_constant<int, 0>());
        body(ks + 1, std::integral_constant<int, 1>());
    }
    /* No copy may land after the workgroup's LDS is given back. */
    gs_vmwait0();
    store_blocks<BDT, NA, NB>(
        d, acc, m0 + wm * WM, n0 + wn * WN, (float *)d.C + d.coff,
        d.R ? (const float *)d.R + d.roff : nullptr,
        [&](int m) {
            return (const float *)d.A + d.aoff +
                   (WIN ? win_row(d.win_m0 + m, d.win_H, d.win_ws, d.win_nwx) : (long)m) * d.lda;
        },
        [&](int n) {
            return (const char *)d.B +
                   (BDT == DT_F32 ? 4 : 2) * (d.boff + n * (d.transb ? (long)d.ldb : 1L));
        });
}

/* ------------------------------------------------------------ small */

/* Small GEMMs of the exact path : a workgroup per tile of
 * 16 MT rows x 16 columns whose NW waves split K; no operand staging: each
 * lane loads four consecutive k of its row of A and its row of B (the Linear
 * weight, float or half) straight from memory, 16 k of 16 rows per load, as
 * the operands of four v_mfma_f32_16x16x4_f32, and the partial tiles are
 * summed through LDS in wave order.
 *
 * Bound by latency: a 128 x 128 tile of k_gemm_f32 walks K in steps of 16
 * with the loads of each exposed (32 x 4096 x 1024: 112 us on 32 of 256
 * CUs). Here a wave's loads for SMALLF_BATCH steps are in flight at once and
 * K is spread over the waves: that product 8.4 us, the decoder's token
 * products 3.1 us (8 x 256 x 256) to 7.9 us (8 x 256 x 2048).
 *
 * MFMA 16x16x4 lane layouts: A lane l holds A[l % 16][l / 16], B lane l
 * B[l / 16][l % 16], D register r of lane l D[4 (l / 16) + r][l % 16]. The
 * k a lane half holds may be any permutation as long as A and B agree. */
#define SMALLF_BATCH 4

template <int BDT, int MT, int NW>
__global__ __launch_bounds__(64 * NW) void k_gemm_small_f32(gemm_desc d)
{
    __shared__ float red[NW][MT][4][64];
    const int t = threadIdx.x, l = t & 63, w = t >> 6, q = l >> 4, l16 = l & 15;
    const int m0 = blockIdx.y * 16 * MT, n0 = blockIdx.x * 16;
    const long z0 = blockIdx.z / d.nb1, z1 = blockIdx.z % d.nb1;
    const long cz = z0 * d.sc0 + z1 * d.sc1;
    const int ksteps = (d.K + 15) / 16, per = (ksteps + NW - 1) / NW;
    const int s0 = w * per, s1 = min(s0 + per, ksteps);
    const int n = min(n0 + l16, d.N - 1);
    const float *pa[MT];
    const long ao = d.aoff + z0 * d.sa0 + z1 * d.sa1 + 4 * q;
    const long bo = d.boff + z0 * d.sb0 + z1 * d.sb1 + (long)n * d.ldb + 4 * q;
    f32x4 acc[MT];

    for (int i = 0; i < MT; i++) {
        pa[i] = (const float *)d.A + ao + (long)min(m0 + 16 * i + l16, d.M - 1) * d.lda;
        acc[i] = (f32x4){};
    }
    for (int s = s0; s < s1; s += SMALLF_BATCH) {
        f32x4 a[SMALLF_BATCH][MT], b[SMALLF_BATCH];

#pragma unroll
        for (int u = 0; u < SMALLF_BATCH; u++) {
            /* K % 4 == 0: a lane's four k are in or out together. */
            const int k = 16 * (s + u);
            const bool in = s + u < s1 && k + 4 * q < d.K;

            for (int i = 0; i < MT; i++)
                a[u][i] = in ? *(const f32x4 *)(pa[i] + k) : (f32x4){};
            if constexpr (BDT == DT_F32)
                b[u] = in ? *(const f32x4 *)((const float *)d.B + bo + k) : (f32x4){};
            else {
                const uint2 v = in ? *(const uint2 *)((const uint16_t *)d.B + bo + k)
                                   : make_uint2(0, 0);

                b[u][0] = h2f((uint16_t)(v.x & 0xffffu));
                b[u][1] = h2f((uint16_t)(v.x >> 16));
                b[u][2] = h2f((uint16_t)(v.y & 0xffffu));
                b[u][3] = h2f((uint16_t)(v.y >> 16));
            }
        }
#pragma unroll
        for (int u = 0; u < SMALLF_BATCH; u++)
#pragma unroll
            for (int e = 0; e < 4; e++)
#pragma unroll
                for (int i = 0; i < MT; i++)
                    acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u][i][e], b[u][e], acc[i], 0,
                                                                  0, 0);
    }
    for (int i = 0; i < MT; i++)
        for (int r = 0; r < 4; r++)
            red[w][i][r][l] = acc[i][r];
    __syncthreads();
    for (int x = t; x < MT * 256; x += 64 * NW) {
        const int i = x >> 8, r = (x >> 6) & 3, ll = x & 63;
        const int mr = m0 + 16 * i + 4 * (ll >> 4) + r, nc = n0 + (ll & 15);
        const long idx = (long)mr * d.ldc + nc;
        float v = red[0][i][r][ll];

        for (int p = 1; p < NW; p++)
            v += red[p][i][r][ll];
        if (mr >= d.M || nc >= d.N)
            continue;
        v = act_k(d.alpha * v + (d.bias ? d.bias[nc] : 0.0f), d.act);
        if (d.R)
            v += ((const float *)d.R)[d.roff + cz + idx];
        ((float *)d.C)[d.coff + cz + idx] = v;
    }
}

/* ------------------------------------------------------------ launch */

static int gs_aligned(const gemm_desc *d)
{
    const long a = d->aoff | d->sa0 | d->sa1 | d->lda, b = d->boff | d->sb0 | d->sb1 | d->ldb;

    /* alpha carries the scale of the pieces (2^-48) and stays normal. */
    if (d->alpha != 0.0f && !(fabsf(d->alpha) >= 0x1p-60f))
        return 0;
    if (d->mode != MODE_F32 || d->adt != DT_F32 || d->cdt != DT_F32 || d->bdt == DT_BF16 ||
        d->unpart_ws > 0 || d->pack_N > 0 || d->K < 4 || d->K % 4 || a % 4 ||
        ((uintptr_t)d->A & 15))
        return 0;
    /* A K x N operand is read element by element. */
    return !d->transb || (b % 4 == 0 && ((uintptr_t)d->B & 15) == 0);
}

static long gs_tiles(const gemm_desc *d, int bm, int bn)
{
    return (long)((d->M + bm - 1) / bm) * ((d->N + bn - 1) / bn);
}

/* Small: at most one 64 x 64 tile per two CUs, where a staged tile's K loop
 * is all latency (400 x 1024 x 1024, 112 tiles: 27 us against 28; 1000 x 1024
 * x 1024, 256 tiles: 49 against 30; 1000 x 300 x 4096, 80 tiles: 75 against
 * 117). Of a batch only products of up to three tiles or 32 rows or columns:
 * above that a batch fills the chip and the small kernel, which reads its
 * operands once per 16 columns, is bound by the caches (576 x 576 x 64: 16
 * products 34 us against 15, 144 272 against 80; 64 products of 256 x 256 x
 * 128 40 against 21). A batch is told by its strides, not by how many
 * products the call holds, so that a call's bits do not depend on that. */
static int gs_small(const gemm_desc *d)
{
    const long tiles = gs_tiles(d, 64, 64);
    const int batch = (d->sa0 | d->sa1 | d->sb0 | d->sb1 | d->sc0 | d->sc1) != 0;

    return d->transb && tiles * 2 <= dev_cu_count() &&
           !(batch && tiles > 3 && d->M > 32 && d->N > 32);
}

/* Rows of A per packed chunk: at most 512 MiB of pieces. */
static int gs_chunk(const gemm_desc *d)
{
    const long row = GS_STEPS((long)d->K) * 96, rows = (512L << 20) / row / 256 * 256;

    return rows < 256 ? 256 : rows < d->M ? (int)rows : d->M;
}

/* Packing pays when what it saves, about 4.6e-15 s per product (125 against
 * 175 TFLOP/s), exceeds its 2.2e-12 s per element and a launch: 1000 x 1024 x
 * 1024 30 us staged, 37 packed; 1400 rows 42 and 44; 5184 rows 85 and 78. A
 * product over the tokens of windows replaces one over all window rows, so
 * it is packed where that was. */
extern "C" size_t gemm_split_ws(const gemm_desc *d)
{
    const double wr = (double)d->win_nwx * d->win_ws, M = d->win_ws > 0 ? wr * wr : d->M, N = d->N, K = d->K;

    if (!gs_aligned(d) || d->nb != 1 || gs_small(d) ||
        (M + N) * K * 2.2e-12 + 4e-6 > M * N * K * 4.6e-15)
        return 0;
    return (size_t)GS_STEPS((long)d->K) * 1024 *
           (((size_t)gs_chunk(d) + 31) / 32 * 3 +
            ((size_t)d->N + 31) / 32 * (d->bdt == DT_F32 ? 3 : 2));
}

/* Tile shape of k_gemm_frag. With every CU busy the chip runs at its power:
 * a 64 x 64 unit of C costs 1.0 (256 x 256 tiles) to 1.17 (64 x 64, more
 * operand traffic); a last round that fills only some CUs runs each of its
 * tiles at the higher clock, `alone` per unit, unless the power is used up
 * all the same. Measured (11 us per unit at K = 1024, 5184 x 1024 .. 4096 and
 * 2500 x 1024); the model picks within 3 % of the best of the five. */
static const struct {
    int bm, bn;
    double full, alone;
} gs_cfg[5] = {{256, 256, 1.0, 0.62}, {256, 128, 1.05, 0.85}, {128, 128, 1.06, 0.95},
               {128, 64, 1.13, 0.9}, {64, 64, 1.17, 1.0}};

static int gs_pick(const gemm_desc *d)
{
    const long cus = dev_cu_count();
    double best = 0.0;
    int pick = 0;

    for (int c = 0; c < 5; c++) {
        const long tiles = gs_tiles(d, gs_cfg[c].bm, gs_cfg[c].bn), rem = tiles % cus;
        const double unit = gs_cfg[c].bm * gs_cfg[c].bn / 4096.0;
        const double part = gs_cfg[c].full * rem / cus;
        const double cost = unit * (tiles / cus * gs_cfg[c].full +
                                    (rem == 0 ? 0.0
                                              : part > gs_cfg[c].alone ? part : gs_cfg[c].alone));

        if (c == 0 || cost < best) {
            best = cost;
            pick = c;
        }
    }
    return pick;
}

template <int BDT>
static int launch_packed(const gemm_desc *d, void *ws, hipStream_t s)
{
    constexpr int NPB = BDT == DT_F32 ? 3 : 2;
    const long nks = GS_STEPS((long)d->K);
    const int chunk = gs_chunk(d), bblocks = (int)((d->N + 31L) / 32 * (nks / 4));
    char *pb = (char *)ws, *pa = pb + (d->N + 31L) / 32 * nks * NPB * 1024;
    const frag_src fb = {(const char *)d->B + (BDT == DT_F32 ? 4 : 2) * d->boff, d->ldb, d->N,
                         d->K, !d->transb, pb, 0, 0, 0, 0};

    for (int m0 = 0; m0 < d->M; m0 += chunk) {
        gemm_desc c = *d;

        c.M = d->M - m0 < chunk ? d->M - m0 : chunk;
        c.win_m0 = m0;
        if (d->win_ws == 0)
            c.aoff += (long)m0 * d->lda;
        c.coff += (long)m0 * d->ldc;
        c.roff += (long)m0 * d->ldc;
        const frag_src fa = {(const float *)d->A + c.aoff, d->lda, c.M, d->K, 0, pa,
                             c.win_H, c.win_ws, c.win_nwx, c.win_m0};
        const long ablocks = (c.M + 31L) / 32 * (nks / 4);
        const int cfg = gs_pick(&c);
        const long grid = (gs_tiles(&c, gs_cfg[cfg].bm, gs_cfg[cfg].bn) + GS_NXCD - 1) /
                          GS_NXCD * GS_NXCD;

        if (ablocks + bblocks > 0x7fffffffL || grid > 0x7fffffffL)
            return hipErrorInvalidConfiguration;
        /* The weights are split once, with the first chunk. */
        const dim3 pgrid((unsigned)(ablocks + (m0 ? 0 : bblocks)));

        if (d->win_ws > 0)
            hipLaunchKernelGGL((k_split_pack<BDT, true>), pgrid, dim3(256), 0, s, fa, fb,
                               (int)ablocks);
        else
            hipLaunchKernelGGL((k_split_pack<BDT, false>), pgrid, dim3(256), 0, s, fa, fb,
                               (int)ablocks);
#define GS_FRAG(I, BM, BN, WM, WN)                                                              \
    if (cfg == I && d->win_ws > 0)                                                             \
        hipLaunchKernelGGL((k_gemm_frag<BM, BN, WM, WN, BDT, true>), dim3((unsigned)grid),     \
                           dim3((BM / WM) * (BN / WN) * 64), 0, s, c, pa, pb);                 \
    else if (cfg == I)                                                                         \
        hipLaunchKernelGGL((k_gemm_frag<BM, BN, WM, WN, BDT, false>), dim3((unsigned)grid),    \
                           dim3((BM / WM) * (BN / WN) * 64), 0, s, c, pa, pb)
        GS_FRAG(0, 256, 256, 64, 64);
        GS_FRAG(1, 256, 128, 64, 64);
        GS_FRAG(2, 128, 128, 64, 32);
        GS_FRAG(3, 128, 64, 64, 32);
        GS_FRAG(4, 64, 64, 32, 32);
#undef GS_FRAG
    }
    return hipGetLastError();
}

template <int BDT, bool TRANSB>
static int launch_staged(const gemm_desc *d, hipStream_t s)
{
    /* 128 x 64 tiles when they give every CU two (331776 x 128 x 256: 189 us
     * against 202; 165888 rows 87 against 90), else 64 x 64 (5184 x 128 x 256:
     * 11 us against 16). */
    const bool big = gs_tiles(d, 128, 64) * d->nb >= 2L * dev_cu_count();
    const long tiles = big ? gs_tiles(d, 128, 64) : gs_tiles(d, 64, 64);
    const long grid =
        tiles < GS_XCD_TILES ? tiles : (tiles + GS_NXCD - 1) / GS_NXCD * GS_NXCD;

    if (grid > 0x7fffffffL)
        return hipErrorInvalidConfiguration;
    if (big)
        hipLaunchKernelGGL((k_gemm_split<128, 64, 64, 32, BDT, TRANSB>),
                           dim3((unsigned)grid, 1, d->nb), dim3(256), 0, s, *d);
    else
        hipLaunchKernelGGL((k_gemm_split<64, 64, 32, 32, BDT, TRANSB>),
                           dim3((unsigned)grid, 1, d->nb), dim3(256), 0, s, *d);
    return hipGetLastError();
}

template <int BDT> static int launch_small(const gemm_desc *d, hipStream_t s)
{
    /* Two row tiles per workgroup once single ones would give every CU two;
     * four waves' loads cover K <= 512, eight beyond. */
    const long t16 = gs_tiles(d, 16, 16);
    const int mt = t16 >= 2L * dev_cu_count() ? 2 : 1;
    const dim3 grid((d->N + 15) / 16, (d->M + 16 * mt - 1) / (16 * mt), d->nb);

    if (mt == 2 && d->K > 512)
        hipLaunchKernelGGL((k_gemm_small_f32<BDT, 2, 8>), grid, dim3(512), 0, s, *d);
    else if (mt == 2)
        hipLaunchKernelGGL((k_gemm_small_f32<BDT, 2, 4>), grid, dim3(256), 0, s, *d);
    else if (d->K > 512)
        hipLaunchKernelGGL((k_gemm_small_f32<BDT, 1, 8>), grid, dim3(512), 0, s, *d);
    else
        hipLaunchKernelGGL((k_gemm_small_f32<BDT, 1, 4>), grid, dim3(256), 0, s, *d);
    return hipGetLastError();
}

extern "C" int launch_gemm_split(const gemm_desc *d, void *ws, size_t ws_bytes, void *stream)
{
    hipStream_t s = (hipStream_t)stream;
    const size_t need = gemm_split_ws(d);

    if (!gs_aligned(d))
        return -1;
    if (d->win_ws > 0 && !(need && ws && ws_bytes >= need))
        return -1; /* row map: packed operands only */
    if (gs_small(d))
        return d->bdt == DT_F32 ? launch_small<DT_F32>(d, s) : launch_small<DT_F16>(d, s);
    if (need && ws && ws_bytes >= need)
        return d->bdt == DT_F32 ? launch_packed<DT_F32>(d, ws, s)
                                : launch_packed<DT_F16>(d, ws, s);
    if (d->bdt == DT_F32)
        return d->transb ? launch_staged<DT_F32, true>(d, s) : launch_staged<DT_F32, false>(d, s);
    return d->transb ? launch_staged<DT_F16, true>(d, s) : launch_staged<DT_F16, false>(d, s);
}
