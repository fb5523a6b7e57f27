/* SPDX-License-Identifier: Unlicense
 *
 * Mask decoder output kernels on gfx950: the scatter of the 2x2 /
 * stride-2 transposed convolutions of the output upscaling
 * (sam3_kernels.cl:762-786), the low-resolution mask logits
 * (sam3_kernels.cl:789-805) and the postprocessing resize with its
 * per-mask statistics (sam3_kernels.cl:807-883).
 */
#include "k_common.h"

/* One thread per (prompt, input pixel, output channel co): the four GEMM
 * columns co 4 + dy 2 + dx are one float4 (coalesced across co), and each
 * lands at output pixel (2y + dy, 2x + dx) of the P x 2H x 2W x Co map as
 * act(G + bias[co] (+ add)), consecutive co again consecutive. The add map
 * (2H x 2W x Co) is shared by the prompts. */
__global__ __launch_bounds__(256) void k_convt_scatter(const float *__restrict__ G,
                                                       float *__restrict__ out,
                                                       const float *__restrict__ bias,
                                                       const float *__restrict__ add,
                                                       int H, int W, int Co,
                                                       long total, int act)
{
    const long gid = (long)blockIdx.x * 256 + threadIdx.x;

    if (gid >= total)
        return;
    const int co = (int)(gid % Co);
    const long pix = gid / Co;
    const int x = (int)(pix % W);
    const long rest = pix / W;
    const int y = (int)(rest % H);
    const long p = rest / H;
    const f32x4 v = *(const f32x4 *)(G + 4 * gid);
    const float bc = bias[co];

    for (int dy = 0; dy < 2; dy++)
        for (int dx = 0; dx < 2; dx++) {
            const long o = ((2 * y + dy) * 2L * W + 2 * x + dx) * Co + co;
            float u = v[2 * dy + dx] + bc;

            if (add)
                u += add[o];
            out[p * 4L * H * W * Co + o] = act_k(u, act);
        }
}

extern "C" int launch_convt_scatter(const float *G, float *out,
                                    const float *bias, const float *add,
                                    int P, int H, int W, int Co, int act,
                                    void *stream)
{
    const long total = (long)P * H * W * Co;

    if (total <= 0)
        return hipSuccess;
    if ((total + 255) / 256 > 0x7fffffffL || ((uintptr_t)G & 15))
        return hipErrorInvalidConfiguration;
    hipLaunchKernelGGL(k_convt_scatter, dim3((unsigned)((total + 255) / 256)),
                       dim3(256), 0, (hipStream_t)stream, G, out, bias, add,
                       H, W, Co, total, act);
    return hipGetLastError();
}

/* The reference's float4 dot as a chain of fused multiply-adds and its
 * dot16 of four quarters summed left to right. */
__device__ __forceinline__ float dot4f(f32x4 a, f32x4 b)
{
    return fmaf(a.w, b.w, fmaf(a.z, b.z, fmaf(a.y, b.y, a.x * b.x)));
}

/* Low-resolution logits: one thread per (prompt, pixel); the pixel's 32
 * channels are 8 float4 loads, the prompt's 96 hypernetwork weights are
 * read through the cache. out [P][3][npix]. */
__global__ __launch_bounds__(256) void k_mask_logits(const float *__restrict__ U,
                                                     const float *__restrict__ hyper,
                                                     float *__restrict__ out,
                                                     int npix, long total)
{
    const long gid = (long)blockIdx.x * 256 + threadIdx.x;

    if (gid >= total)
        return;
    const long p = gid / npix, pix = gid - p * npix;
    const f32x4 *u = (const f32x4 *)(U + gid * 32);
    const f32x4 *h = (const f32x4 *)(hyper + p * 96);
    f32x4 uv[8];

    for (int i = 0; i < 8; i++)
        uv[i] = u[i];
    for (int k = 0; k < 3; k++) {
        const f32x4 *hk = h + 8 * k;
        const float d0 = ((dot4f(uv[0], hk[0]) + dot4f(uv[1], hk[1])) + dot4f(uv[2], hk[2])) +
                         dot4f(uv[3], hk[3]);
        const float d1 = ((dot4f(uv[4], hk[4]) + dot4f(uv[5], hk[5])) + dot4f(uv[6], hk[6])) +
                         dot4f(uv[7], hk[7]);

        out[(p * 3 + k) * npix + pix] = d0 + d1;
    }
}

extern "C" int launch_mask_logits(const float *U, const float *hyper,
                                  float *out, int P, int npix, void *stream)
{
    const long total = (long)P * npix;

    if (total <= 0)
        return hipSuccess;
    if (((uintptr_t)U | (uintptr_t)hyper) & 15)
        return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_mask_logits, dim3((unsigned)((total + 255) / 256)),
                       dim3(256), 0, (hipStream_t)stream, U, hyper, out, npix,
                       total);
    return hipGetLastError();
}

/* PyTorch bilinear source coordinate, align_corners = False. */
__device__ __forceinline__ float src_coord(float scale, int dst)
{
    const float s = scale * ((float)dst + 0.5f) - 0.5f;

    return s < 0.0f ? 0.0f : s;
}

/* Columns per wave (4 per lane), most rows per wave (a lane holds the
 * coordinates of one) and waves per workgroup of k_mask_post. */
#define MP_COLS 256
#define MP_ROWS 64
#define MP_WAVES 4

/* Postprocessing of mask k = blockIdx.z (plane sel[k] of lowres): bilinear
 * value, binary mask byte, the counts (v > offset, v > -offset) and the
 * bounding box of v > 0 of the out_h x out_w crop.
 *
 * Bound by VALU issue and the mask stores about equally, so everything that
 * does not change per pixel is taken out of the pixel: a lane owns four
 * columns (their x0, x1, lx formed once) and walks MP_ROWS rows; the two
 * horizontally interpolated source rows (top, bot) are kept while the output
 * rows stay between them (a wave-uniform test; when upscaling they last
 * out_h / L rows, and the next pair's top is this one's bot), the counts are
 * lane sums reduced once, the box is one flag word per lane and a scalar row
 * range, and the four mask bytes go out as one dword (at any byte
 * alignment). The value of a pixel is formed by the same operations in the
 * same order as one pixel at a time would be. 64 planes of 288^2 to 1080 x
 * 1440: 61 us against 813 us with a pixel's coordinates, gathers, byte
 * store and minima formed per pixel. */
__global__ __launch_bounds__(64 * MP_WAVES) void
k_mask_post(const float *__restrict__ lowres, const int *__restrict__ sel, int L,
            int out_h, int out_w, int wrows, float offset,
            unsigned char *__restrict__ mask, int *__restrict__ stats)
{
    __shared__ int red[MP_WAVES][6];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int oy0 = (blockIdx.y * MP_WAVES + w) * wrows;
    const int ox0 = blockIdx.x * MP_COLS + 4 * lane;
    const int k = blockIdx.z, rows = min(wrows, out_h - oy0);
    const float *lr = lowres + (long)sel[k] * L * L;
    const int ncol = min(4, out_w - ox0); /* <= 0: the lane has no column */
    const float scx = (float)L / out_w;
    int x0[4], x1[4];
    float lx[4], top[4] = {}, bot[4] = {};
    unsigned cols = 0; /* byte e: column ox0 + e holds a pixel with v > 0 */
    int inter = 0, uni = 0, ymin = 0x7fffffff, ymax = -1, cy0 = -1, cy1 = -1;
    /* Lane i holds row i's source coordinate. */
    const float syl = src_coord((float)L / out_h, oy0 + lane);
    const int y0l = (int)syl;
    const float lyl = syl - y0l;

    for (int e = 0; e < 4; e++) {
        const float sx = src_coord(scx, min(ox0 + e, out_w - 1));

        x0[e] = (int)sx;
        x1[e] = x0[e] + (x0[e] < L - 1);
        /* Columns past the edge interpolate to NaN, which no test counts. */
        lx[e] = e < ncol ? sx - x0[e] : __builtin_nanf("");
    }
    for (int i = 0; i < rows; i++) {
        const int oy = oy0 + i;
        /* The row is the wave's: its source rows in scalar registers. */
        const int y0 = __builtin_amdgcn_readlane(y0l, i), y1 = y0 + (y0 < L - 1);
        const float ly = __builtin_bit_cast(
            float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, lyl), i));
        const float hy = 1.0f - ly;
        unsigned bytes = 0;

        if (y0 != cy0 || y1 != cy1) {
            const float *r0 = lr + (long)y0 * L, *r1 = lr + (long)y1 * L;
            const bool shift = y0 == cy1;

            for (int e = 0; e < 4; e++) {
                top[e] = shift ? bot[e]
                               : fmaf(lx[e], r0[x1[e]], (1.0f - lx[e]) * r0[x0[e]]);
                bot[e] = fmaf(lx[e], r1[x1[e]], (1.0f - lx[e]) * r1[x0[e]]);
            }
            cy0 = y0;
            cy1 = y1;
        }
        for (int e = 0; e < 4; e++) {
            const float v = fmaf(ly, bot[e], hy * top[e]);

            bytes |= v > 0.0f ? 1u << (8 * e) : 0u;
            inter += v > offset;
            uni += v > -offset;
        }
        if (ncol == 4) {
            unsigned char *p = mask + ((long)k * out_h + oy) * out_w + ox0;

            __builtin_memcpy(p, &bytes, 4);
        }
        else
            for (int e = 0; e < ncol; e++)
                mask[((long)k * out_h + oy) * out_w + ox0 + e] =
                    (unsigned char)(bytes >> (8 * e));
        cols |= bytes;
        if (__ballot(bytes != 0)) {
            ymin = min(ymin, oy);
            ymax = oy;
        }
    }
    for (int s = 32; s >= 1; s >>= 1) {
        inter += __shfl_xor(inter, s, 64);
        uni += __shfl_xor(uni, s, 64);
    }
    {
        int x0m = 0x7fffffff, x1m = -1;

        for (int e = 0; e < 4; e++) {
            const unsigned long long b = __ballot(cols >> (8 * e) & 1);

            if (b) {
                const int base = blockIdx.x * MP_COLS + e;

                x0m = min(x0m, base + 4 * (__ffsll(b) - 1));
                x1m = max(x1m, base + 4 * (63 - __clzll(b)));
            }
        }
        if (lane == 0) {
            red[w][0] = inter;
            red[w][1] = uni;
            red[w][2] = x0m;
            red[w][3] = ymin;
            red[w][4] = x1m;
            red[w][5] = ymax;
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        int s[6];

        for (int j = 0; j < 6; j++)
            s[j] = red[0][j];
        for (int i = 1; i < MP_WAVES; i++) {
            s[0] += red[i][0];
            s[1] += red[i][1];
            s[2] = min(s[2], red[i][2]);
            s[3] = min(s[3], red[i][3]);
            s[4] = max(s[4], red[i][4]);
            s[5] = max(s[5], red[i][5]);
        }
        int *st = stats + 6 * k;

        if (s[0])
            atomicAdd(&st[0], s[0]);
        if (s[1])
            atomicAdd(&st[1], s[1]);
        if (s[4] >= 0) {
            atomicMin(&st[2], s[2]);
            atomicMin(&st[3], s[3]);
            atomicMax(&st[4], s[4]);
            atomicMax(&st[5], s[5]);
        }
    }
}

/* Up to 256 plane numbers by value, so that they travel with the launch. */
struct mask_sel {
    int v[256];
};

/* sel[i0 + i] and the empty statistics of masks i0 .. i0 + n - 1. */
__global__ __launch_bounds__(256) void k_mask_init(mask_sel s, int n, int i0,
                                                   int *__restrict__ sel,
                                                   int *__restrict__ stats)
{
    const int i = threadIdx.x;

    if (i >= n)
        return;
    int *st = stats + 6 * (i0 + i);

    sel[i0 + i] = s.v[i];
    st[0] = st[1] = 0;
    st[2] = st[3] = 0x7fffffff;
    st[4] = st[5] = -1;
}

/* The masks' plane numbers (host) and empty statistics into device memory,
 * without a transfer that the host would wait for (about 10 us each). */
extern "C" int launch_mask_init(const int *hsel, int n, int *sel, int *stats, void *stream)
{
    for (int i0 = 0; i0 < n; i0 += 256) {
        const int c = n - i0 < 256 ? n - i0 : 256;
        mask_sel s;

        for (int i = 0; i < c; i++)
            s.v[i] = hsel[i0 + i];
        for (int i = c; i < 256; i++)
            s.v[i] = 0;
        hipLaunchKernelGGL(k_mask_init, dim3(1), dim3(256), 0, (hipStream_t)stream, s, c, i0, sel,
                           stats);
    }
    return hipGetLastError();
}

extern "C" int launch_mask_post(const float *lowres, const int *sel, int n,
                                int L, int out_h, int out_w, float offset,
                                unsigned char *mask, int *stats, void *stream)
{
    if (n <= 0 || out_h <= 0 || out_w <= 0)
        return hipSuccess;
    if (n > 65535 || (out_h + 15) / 16 > 65535)
        return hipErrorInvalidConfiguration;
    /* Rows per wave: as many as leave about sixteen waves per CU (each
     * workgroup ends in up to six atomics on a few cache lines, which cost
     * more than its pixels when the workgroups are small: 85 us at 16 rows,
     * 65 at 64), from 4 to 64, then the same for every wave. */
    const long cols = (out_w + MP_COLS - 1) / MP_COLS;
    const long fill = cols * out_h * n / (16L * dev_cu_count());
    const int most = MP_WAVES * (fill < 4 ? 4 : fill > MP_ROWS ? MP_ROWS : (int)fill);
    const int ny = (out_h + most - 1) / most;
    const int wrows = (out_h + ny * MP_WAVES - 1) / (ny * MP_WAVES);

    hipLaunchKernelGGL(k_mask_post,
                       dim3((unsigned)cols, ny, n),
                       dim3(64 * MP_WAVES), 0, (hipStream_t)stream, lowres, sel, L,
                       out_h, out_w, wrows, offset, mask, stats);
    return hipGetLastError();
}
