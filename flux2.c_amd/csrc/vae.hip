/*
 * vae.hip - the memory-bound kernels of the VAE decoder and encoder (reference: flux_vae_decode,
 * flux_vae.c:690-837; flux_vae_encode, flux_vae.c:320-443); their convolutions and attention
 * products run as MFMA GEMMs (gemm.hip).
 *
 * Images are channels-last with a one-pixel zero border: position p = y * Wp + x over the
 * (H+2) x (W+2) grid, channels contiguous. That makes a 3x3 convolution one GEMM whose K steps
 * read the same rows shifted by a constant (flux_hip_conv), and every kernel here keeps the
 * border at zero so that the next convolution sees its padding. The residual stream is fp32;
 * what feeds an MFMA is bf16.
 */
#include "common.h"
#include "../../include/flux_hip.h"
#include <math.h>

#define LAUNCH_OK(what)                                                                         \
    do {                                                                                        \
        hipError_t e_ = hipGetLastError();                                                      \
        if (e_ != hipSuccess) return flux_hip_fail("%s launch failed: %s", what, hipGetErrorString(e_)); \
    } while (0)

__device__ __forceinline__ bool interior(int p, int hp, int wp) {
    const int y = p / wp, x = p - y * wp;
    return y >= 1 && y < hp - 1 && x >= 1 && x < wp - 1;
}

/* latent [128, h, w] fp32 -> x * sqrt(var + eps) + mean per latent channel (flux_vae.c:718-728),
 * 2x2 unpatchify to 32 channels at (2h, 2w) (flux_kernels.c:1067-1097), 1x1 post-quant
 * convolution 32 -> 32 (flux_vae.c:739-741); written as bf16 [Hp*Wp, 64] with channels 32..63
 * zero (the first 3x3 convolution wants a multiple of 64 input channels). 32 lanes a position: a lane scales one of its input channels,
 * takes the others' from their lanes and makes one output channel, eight positions at a time per workgroup. (A lane that scaled all 32 itself,
 * one load after the other, for one position per wave: 12.1 us at 32 x 32 positions and 27.6 at 128 x 128, now 6.0 and 12.8.) */
#define LATENT_TRIPS 2
__global__ __launch_bounds__(256) void vae_latent_kernel(bf16 *__restrict__ out, const float *__restrict__ latent,
                                                         const float *__restrict__ bn_mean, const float *__restrict__ bn_var,
                                                         const float *__restrict__ pq_w, const float *__restrict__ pq_b,
                                                         int h, int w, float eps) {
    const int hp = 2 * h + 2, wp = 2 * w + 2, c = threadIdx.x & 31;
    float wc[32];
#pragma unroll
    for (int ci = 0; ci < 32; ci++) wc[ci] = pq_w[c * 32 + ci];
    const float bias = pq_b[c];
    for (int t = 0; t < LATENT_TRIPS; t++) {
        const int p = (blockIdx.x * LATENT_TRIPS + t) * 8 + (threadIdx.x >> 5);
        const int y = p / wp, x = p - y * wp, cy = min(max(y - 1, 0), 2 * h - 1), cx = min(max(x - 1, 0), 2 * w - 1);
        const int lc = c * 4 + (cy & 1) * 2 + (cx & 1);
        const float z = latent[((size_t)lc * h + (cy >> 1)) * w + (cx >> 1)] * sqrtf(bn_var[lc] + eps) + bn_mean[lc];
        float v = bias;
#pragma unroll
        for (int ci = 0; ci < 32; ci++) v += wc[ci] * __shfl(z, ci, 32);
        if (p < hp * wp) {
            out[(size_t)p * 64 + c] = (bf16)(interior(p, hp, wp) ? v : 0.0f);
            out[(size_t)p * 64 + 32 + c] = (bf16)0.0f;
        }
    }
}

/* ---- group norm (flux_group_norm, flux_kernels.c:511-553): 32 groups of C/32 adjacent channels,
 * statistics over the whole image. Three kernels: per-block partial sums, their combination in
 * double precision, and the normalisation itself. Border positions hold zeros and add nothing
 * to the sums; the element count is the interior's. ---- */
#define GN_ROWS 256 /* positions per workgroup */

/* p / wp for p < 2^22, wp < 2^12 through a multiplication: magic = ceil(2^40 / wp) */
__device__ __forceinline__ int div_wp(int p, unsigned long long magic) { return (int)(((unsigned long long)p * magic) >> 40); }

__device__ __forceinline__ f32x4 load_quad(const float *p) { return *(const f32x4 *)p; }
__device__ __forceinline__ f32x4 load_quad(const bf16 *p) {
    const bf16x4 v = *(const bf16x4 *)p;
    f32x4 o;
#pragma unroll
    for (int e = 0; e < 4; e++) o[e] = (float)v[e];
    return o;
}

/* A workgroup covers GN_ROWS positions: thread (r0, q) walks rows r0, r0 + rpi, ... of quad q
 * (4 adjacent channels, always inside one group), four rows per trip so that four loads are in
 * flight. */
template <typename T>
__global__ __launch_bounds__(256) void gn_partial_kernel(float *__restrict__ partial, const T *__restrict__ x, int rows, int C) {
    __shared__ float sh[256][2];
    const int quads = C >> 2, rpi = 256 / quads; /* C is 128, 256 or 512: 32, 64 or 128 quads */
    const int q = threadIdx.x % quads, r0 = threadIdx.x / quads;
    const int row_begin = blockIdx.x * GN_ROWS, row_end = min(rows, row_begin + GN_ROWS);
    float s = 0.0f, ss = 0.0f;
    const T *src = x + q * 4;
    int r = row_begin + r0;
    for (; r + 3 * rpi < row_end; r += 4 * rpi) {
        f32x4 v[4];
#pragma unroll
        for (int k = 0; k < 4; k++) v[k] = load_quad(src + (size_t)(r + k * rpi) * C);
#pragma unroll
        for (int k = 0; k < 4; k++)
#pragma unroll
            for (int e = 0; e < 4; e++) { s += v[k][e]; ss += v[k][e] * v[k][e]; }
    }
    for (; r < row_end; r += rpi) {
        const f32x4 v = load_quad(src + (size_t)r * C);
#pragma unroll
        for (int e = 0; e < 4; e++) { s += v[e]; ss += v[e] * v[e]; }
    }
    sh[threadIdx.x][0] = s;
    sh[threadIdx.x][1] = ss;
    __syncthreads();
    if (threadIdx.x < 32) {
        /* group g owns quads [g * qpg, (g+1) * qpg) of every thread row; fixed summation order */
        const int g = threadIdx.x, qpg = quads >> 5;
        float a = 0.0f, b = 0.0f;
        for (int rr = 0; rr < rpi; rr++)
            for (int k = 0; k < qpg; k++) {
                a += sh[rr * quads + g * qpg + k][0];
                b += sh[rr * quads + g * qpg + k][1];
            }
        partial[((size_t)blockIdx.x * 32 + g) * 2 + 0] = a;
        partial[((size_t)blockIdx.x * 32 + g) * 2 + 1] = b;
    }
}

/* one workgroup per group: mean and 1/sqrt(var + eps) with the biased variance */
__global__ __launch_bounds__(256) void gn_finalize_kernel(float *__restrict__ stats, const float *__restrict__ partial, int nblocks,
                                                          double count, float eps) {
    __shared__ double sh[256][2];
    const int g = blockIdx.x;
    double a = 0.0, b = 0.0;
    for (int i = threadIdx.x; i < nblocks; i += 256) {
        a += (double)partial[((size_t)i * 32 + g) * 2 + 0];
        b += (double)partial[((size_t)i * 32 + g) * 2 + 1];
    }
    sh[threadIdx.x][0] = a;
    sh[threadIdx.x][1] = b;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s) {
            sh[threadIdx.x][0] += sh[threadIdx.x + s][0];
            sh[threadIdx.x][1] += sh[threadIdx.x + s][1];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const double mean = sh[0][0] / count;
        double var = sh[0][1] / count - mean * mean;
        if (var < 0.0) var = 0.0;
        stats[g * 2 + 0] = (float)mean;
        stats[g * 2 + 1] = (float)(1.0 / sqrt(var + (double)eps));
    }
}

/* First stage when the sums come from convolution epilogues (flux_hip_conv_stats): conv
 * [prows][C/4][2] holds one (sum, sum of squares) per row-tile half and 4-channel quad. Each
 * workgroup folds a contiguous range of those rows into per-group sums, in the layout the
 * finalize kernel reads. Same thread-to-quad map as the partial-sum pass: coalesced reads. */
__global__ __launch_bounds__(256) void gn_fold_quads_kernel(float *__restrict__ partial, const float *__restrict__ conv, int prows, int C) {
    __shared__ float sh[256][2];
    const int quads = C >> 2, rpi = 256 / quads;
    const int q = threadIdx.x % quads, r0 = threadIdx.x / quads;
    const int per = (prows + gridDim.x - 1) / gridDim.x;
    const int row_begin = blockIdx.x * per, row_end = min(prows, row_begin + per);
    float s = 0.0f, ss = 0.0f;
    for (int r = row_begin + r0; r < row_end; r += rpi) {
        const f32x2 v = *(const f32x2 *)(conv + ((size_t)r * quads + q) * 2);
        s += v[0];
        ss += v[1];
    }
    sh[threadIdx.x][0] = s;
    sh[threadIdx.x][1] = ss;
    __syncthreads();
    if (threadIdx.x < 32) {
        const int g = threadIdx.x, qpg = quads >> 5;
        float a = 0.0f, b = 0.0f;
        for (int rr = 0; rr < rpi; rr++)
            for (int k = 0; k < qpg; k++) {
                a += sh[rr * quads + g * qpg + k][0];
                b += sh[rr * quads + g * qpg + k][1];
            }
        partial[((size_t)blockIdx.x * 32 + g) * 2 + 0] = a;
        partial[((size_t)blockIdx.x * 32 + g) * 2 + 1] = b;
    }
}

/* Both stages in one launch, for images whose convolutions leave few partial rows: a workgroup owns one group and sums its
 * quads over every row in double precision. Up to 2048 rows (512 x 512 positions) that is one launch of 5 us instead of
 * two of 4.7; beyond, the strided 8- to 32-byte reads of 32 workgroups take longer than the two coalesced passes
 * (16448 rows, 1024 x 1024 positions: 6.4 + 4.8 us). */
#define GN_ONE_PASS_ROWS 2048
__global__ __launch_bounds__(256) void gn_stats_kernel(float *__restrict__ stats, const float *__restrict__ conv, int prows, int C, double count,
                                                       float eps) {
    __shared__ double sh[4][2];
    const int g = blockIdx.x, quads = C >> 2, qpg = quads >> 5, sub = threadIdx.x & (qpg - 1), step = 256 / qpg; /* qpg = 1, 2 or 4 */
    double a = 0.0, b = 0.0;
#pragma unroll 4
    for (int r = threadIdx.x / qpg; r < prows; r += step) {
        const f32x2 v = *(const f32x2 *)(conv + ((size_t)r * quads + g * qpg + sub) * 2);
        a += (double)v[0];
        b += (double)v[1];
    }
    for (int o = 32; o > 0; o >>= 1) {
        a += __shfl_xor(a, o);
        b += __shfl_xor(b, o);
    }
    if ((threadIdx.x & 63) == 0) {
        sh[threadIdx.x >> 6][0] = a;
        sh[threadIdx.x >> 6][1] = b;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        const double mean = ((sh[0][0] + sh[1][0]) + (sh[2][0] + sh[3][0])) / count;
        double var = ((sh[0][1] + sh[1][1]) + (sh[2][1] + sh[3][1])) / count - mean * mean;
        if (var < 0.0) var = 0.0;
        stats[g * 2 + 0] = (float)mean;
        stats[g * 2 + 1] = (float)(1.0 / sqrt(var + (double)eps));
    }
}

/* out bf16 = [swish](gamma * (x - mean) * rstd + beta), zeros on the border; raw (optional)
 * receives x itself as bf16, the input of a residual block's 1x1 shortcut convolution. Same
 * thread-to-data map as the partial-sum pass, over `span` positions per workgroup: with 256 of them a 32 x 32 image of 512
 * channels was five workgroups and 32 us, with 8 it is 145 and a few; images that give every compute unit several
 * workgroups either way keep 256. */
template <typename T>
__global__ __launch_bounds__(256) void gn_apply_kernel(bf16 *__restrict__ out, bf16 *__restrict__ raw, const T *__restrict__ x,
                                                       const float *__restrict__ stats, const float *__restrict__ gamma,
                                                       const float *__restrict__ beta, int rows, int C, int hp, int wp,
                                                       unsigned long long magic, int swish, int span) {
    const int quads = C >> 2, rpi = 256 / quads;
    const int q = threadIdx.x % quads, r0 = threadIdx.x / quads;
    const int row_begin = blockIdx.x * span, row_end = min(rows, row_begin + span);
    const int g = (q * 4) / (C >> 5);
    const float mean = stats[g * 2], rstd = stats[g * 2 + 1];
    const f32x4 gm = *(const f32x4 *)(gamma + q * 4), bt = *(const f32x4 *)(beta + q * 4);
    f32x4 sc, sh;
#pragma unroll
    for (int e = 0; e < 4; e++) { sc[e] = gm[e] * rstd; sh[e] = bt[e] - mean * sc[e]; }
    auto one = [&](int r, const f32x4 &v) {
        const int y = div_wp(r, magic), xx = r - y * wp;
        const bool in = y >= 1 && y < hp - 1 && xx >= 1 && xx < wp - 1;
        bf16x4 o;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            float t = v[e] * sc[e] + sh[e];
            if (swish) t = silu_f(t);
            o[e] = (bf16)(in ? t : 0.0f);
        }
        *(bf16x4 *)(out + (size_t)r * C + q * 4) = o;
        if (raw) {
            bf16x4 rw;
#pragma unroll
            for (int e = 0; e < 4; e++) rw[e] = (bf16)v[e];
            *(bf16x4 *)(raw + (size_t)r * C + q * 4) = rw;
        }
    };
    const T *src = x + q * 4;
    int r = row_begin + r0;
    for (; r + 3 * rpi < row_end; r += 4 * rpi) {
        f32x4 v[4];
#pragma unroll
        for (int k = 0; k < 4; k++) v[k] = load_quad(src + (size_t)(r + k * rpi) * C);
#pragma unroll
        for (int k = 0; k < 4; k++) one(r + k * rpi, v[k]);
    }
    for (; r < row_end; r += rpi) one(r, load_quad(src + (size_t)r * C));
}

/* gn_stats_kernel and gn_apply_kernel in one launch, for images whose convolutions leave few partial rows: a workgroup owns 64 channels of
 * `span` positions and sums those channels' partial rows itself, with its first positions already requested. What bounds the small images'
 * norms is the launches, not the bytes. Back to back, one launch against two, us: 16 x 16 x 512 (11 rows of sums) 3.3 / 5.4, 32 x 32 x 512 (37) 3.7 / 5.6,
 * 64 x 64 x 512 (137) 6.0 / 6.9, 84 x 84 x 512 (72) 6.9 / 7.7, 128 x 128 x 512 (128) 12.7 / 13.0. Every workgroup reads the rows anew: with 232
 * to 256 of them it is no gain (8.2 / 8.1, 9.0 / 8.5), with 512 a loss (18 / 13). */
#define GN_FUSED_ROWS 160
template <typename T>
__global__ __launch_bounds__(256) void gn_fused_kernel(bf16 *__restrict__ out, bf16 *__restrict__ raw, const T *__restrict__ x, const float *__restrict__ conv,
                                                       int prows, double count, float eps, const float *__restrict__ gamma, const float *__restrict__ beta,
                                                       int rows, int C, int hp, int wp, unsigned long long magic, int swish, int span) {
    __shared__ double part[16][16][2];
    __shared__ float norm[16][2];
    const int q = threadIdx.x & 15, r0 = threadIdx.x >> 4, quads = C >> 2, qpg = quads >> 5; /* quads of a group: 1, 2 or 4 */
    const int quad = blockIdx.y * 16 + q;
    const int row_begin = blockIdx.x * span, row_end = min(rows, row_begin + span);
    const T *src = x + quad * 4;
    f32x4 v[4];
    const auto request = [&](int r) {
#pragma unroll
        for (int k = 0; k < 4; k++) v[k] = load_quad(src + (size_t)min(r + 16 * k, row_end - 1) * C);
    };
    request(row_begin + r0);
    const f32x4 gm = *(const f32x4 *)(gamma + quad * 4), bt = *(const f32x4 *)(beta + quad * 4);
    double a = 0.0, b = 0.0;
#pragma unroll 8
    for (int r = r0; r < prows; r += 16) {
        const f32x2 t = *(const f32x2 *)(conv + ((size_t)r * quads + quad) * 2);
        a += (double)t[0];
        b += (double)t[1];
    }
    part[r0][q][0] = a;
    part[r0][q][1] = b;
    __syncthreads();
    if (threadIdx.x < 64) { /* four lanes a quad, then the quads of a group */
        const int p = threadIdx.x & 15, k = threadIdx.x >> 4;
        a = (part[k][p][0] + part[k + 4][p][0]) + (part[k + 8][p][0] + part[k + 12][p][0]);
        b = (part[k][p][1] + part[k + 4][p][1]) + (part[k + 8][p][1] + part[k + 12][p][1]);
        a += __shfl_xor(a, 16); b += __shfl_xor(b, 16);
        a += __shfl_xor(a, 32); b += __shfl_xor(b, 32);
        for (int o = 1; o < qpg; o <<= 1) { a += __shfl_xor(a, o); b += __shfl_xor(b, o); }
        const double mean = a / count;
        double var = b / count - mean * mean;
        if (var < 0.0) var = 0.0;
        if (k == 0) {
            norm[p][0] = (float)mean;
            norm[p][1] = (float)(1.0 / sqrt(var + (double)eps));
        }
    }
    __syncthreads();
    const float mean = norm[q][0], rstd = norm[q][1];
    f32x4 sc, sh;
#pragma unroll
    for (int e = 0; e < 4; e++) { sc[e] = gm[e] * rstd; sh[e] = bt[e] - mean * sc[e]; }
    for (int r = row_begin + r0; r < row_end; r += 64) {
        f32x4 w[4];
#pragma unroll
        for (int k = 0; k < 4; k++) w[k] = v[k];
        if (r + 64 < row_end) request(r + 64);
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int rk = r + 16 * k;
            if (rk >= row_end) break;
            const int y = div_wp(rk, magic), xx = rk - y * wp;
            const bool in = y >= 1 && y < hp - 1 && xx >= 1 && xx < wp - 1;
            bf16x4 o, rw;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                float t = w[k][e] * sc[e] + sh[e];
                if (swish) t = silu_f(t);
                o[e] = (bf16)(in ? t : 0.0f);
                rw[e] = (bf16)w[k][e];
            }
            *(bf16x4 *)(out + (size_t)rk * C + quad * 4) = o;
            if (raw) *(bf16x4 *)(raw + (size_t)rk * C + quad * 4) = rw;
        }
    }
}

/* The first norm of a residual block that changes the channel count, and its 1x1 shortcut, from one read of x: out bf16 = swish(norm(x)) as in
 * gn_apply_kernel, y fp32 [rows][cout] = bias + bf16(x) W^T, zeros on the border. What bounds it is HBM; as two kernels with the bf16 copy of x between
 * them, that copy was written and read once more. A workgroup takes P positions, whose bf16 values stay in LDS (64 KB at most, two workgroups to a
 * unit), a wave 16 output channels at a time; 16-byte chunk c of position p lies at c ^ p mod 16, so that a fragment's 16
 * rows fall on different banks. Two launches against this one, us: 1024 x 1024 x 256 -> 128 654, 410 (2.15 GB, 5.2 TB/s), 512 x 512 x 512 -> 256 335, 289 (its
 * weights are as many bytes out of the L2s as x is), 360 x 648 x 128 -> 256 123, 87, 180 x 324 x 256 -> 512 75, 50. With four waves of 32
 * channels 481 and 334. */
template <int CIN, int P>
__global__ __launch_bounds__(512, 4) void gn_skip_kernel(bf16 *__restrict__ out, float *__restrict__ y, const float *__restrict__ x, const float *__restrict__ stats,
                                                         const float *__restrict__ gamma, const float *__restrict__ beta, const bf16 *__restrict__ w,
                                                         const float *__restrict__ bias, int rows, int cout, int hp, int wp, unsigned long long magic) {
    constexpr int QUADS = CIN / 4, RPI = 512 / QUADS, KS = CIN / 32, PB = P / 16, U = 8;
    __shared__ __attribute__((aligned(16))) char raw[P * CIN * 2];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l15 = lane & 15, lq = lane >> 4;
    const int q = tid % QUADS, r0 = tid / QUADS, base = blockIdx.x * P;
    const auto inside = [&](int r) {
        const int py = div_wp(r, magic), px = r - py * wp;
        return py >= 1 && py < hp - 1 && px >= 1 && px < wp - 1;
    };
    bf16x8 fw[KS];
    const auto weights = [&](int n) {
#pragma unroll
        for (int k = 0; k < KS; k++) fw[k] = *(const bf16x8 *)(w + (size_t)(n + l15) * CIN + k * 32 + lq * 8);
    };
    {
        const int g = (q * 4) / (CIN >> 5);
        const float mean = stats[g * 2], rstd = stats[g * 2 + 1];
        const f32x4 gm = *(const f32x4 *)(gamma + q * 4), bt = *(const f32x4 *)(beta + q * 4);
        f32x4 sc, sh;
#pragma unroll
        for (int e = 0; e < 4; e++) { sc[e] = gm[e] * rstd; sh[e] = bt[e] - mean * sc[e]; }
        f32x4 v[U];
#pragma unroll 1
        for (int i = 0; i < P; i += U * RPI) {
#pragma unroll
            for (int u = 0; u < U; u++) v[u] = *(const f32x4 *)(x + (size_t)min(base + i + u * RPI + r0, rows - 1) * CIN + q * 4);
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int p = i + u * RPI + r0, r = base + p;
                const bool in = inside(r);
                bf16x4 o, rw;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    o[e] = (bf16)(in ? silu_f(v[u][e] * sc[e] + sh[e]) : 0.0f);
                    rw[e] = (bf16)v[u][e];
                }
                if (r < rows) *(bf16x4 *)(out + (size_t)r * CIN + q * 4) = o;
                *(bf16x4 *)(raw + p * (CIN * 2) + (((q >> 1) ^ (p & 15)) << 4) + (q & 1) * 8) = rw;
            }
        }
    }
    weights(wave * 16);
    __syncthreads();
#pragma unroll 1
    for (int n = wave * 16; n < cout; n += 128) {
        if (n >= 128) weights(n);
        const f32x4 bv = *(const f32x4 *)(bias + n + 4 * lq);
#pragma unroll 2
        for (int pb = 0; pb < PB; pb++) {
            f32x4 a = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int k = 0; k < KS; k++)
                a = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[k], *(const bf16x8 *)(raw + (16 * pb + l15) * (CIN * 2) + (((4 * k + lq) ^ l15) << 4)), a, 0, 0, 0);
            const int r = base + 16 * pb + l15;
            const bool in = inside(r);
            f32x4 v;
#pragma unroll
            for (int e = 0; e < 4; e++) v[e] = in ? a[e] + bv[e] : 0.0f;
            if (r < rows) *(f32x4 *)(y + (size_t)r * cout + n + 4 * lq) = v;
        }
    }
}

/* nearest-neighbour 2x upsample (flux_upsample_nearest, flux_kernels.c:1017-1036): fp32 or bf16
 * [hp*wp, C] -> bf16 [(2H+2)*(2W+2), C] with a fresh zero border. One thread per bordered source position and V
 * channels, which go to the source's up to four places: interior (y, x) to rows 2y-1, 2y and columns 2x-1, 2x of the bordered output,
 * and the border positions, as zeros, to what of that lies inside: its border. Each value is read once (a thread per
 * output read every one four times: 512 x 512 x 256 from fp32 took 234 us). */
template <typename T, int V>
__global__ __launch_bounds__(256) void vae_upsample_kernel(bf16 *__restrict__ out, const T *__restrict__ x, int hp, int wp, int C) {
    typedef __attribute__((ext_vector_type(V))) __bf16 ov;
    const int groups = C / V, hp2 = 2 * hp - 2, wp2 = 2 * wp - 2;
    const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (size_t)hp * wp * groups) return;
    const int p = (int)(idx / groups), q = (int)(idx - (size_t)p * groups);
    const int y = p / wp, xx = p - y * wp;
    ov o;
#pragma unroll
    for (int e = 0; e < V; e++) o[e] = (bf16)0.0f;
    if (interior(p, hp, wp)) {
#pragma unroll
        for (int k = 0; k < V; k += 4) {
            const f32x4 v = load_quad(x + (size_t)p * C + q * V + k);
#pragma unroll
            for (int e = 0; e < 4; e++) o[k + e] = (bf16)v[e];
        }
    }
#pragma unroll
    for (int dy = -1; dy <= 0; dy++)
#pragma unroll
        for (int dx = -1; dx <= 0; dx++) {
            const int oy = 2 * y + dy, ox = 2 * xx + dx;
            if (oy >= 0 && oy < hp2 && ox >= 0 && ox < wp2) *(ov *)(out + ((size_t)oy * wp2 + ox) * C + q * V) = o;
        }
}

/* ---- encoder side (flux_vae_encode, flux_vae.c:320-443) ---- */

/* image [3, H, W] fp32 -> the 3x3 neighbourhood of every position as one row of 64 bf16:
 * element (ky*3 + kx)*3 + c = img[c, y-1+ky, x-1+kx] (zero outside the image), elements 27..63
 * zero. The first convolution (3 -> 128 channels, flux_vae.c:336-338) is then a GEMM with K = 64
 * over these rows. 32 positions per workgroup of 256 threads. */
__global__ __launch_bounds__(256) void vae_image_in_kernel(bf16 *__restrict__ out, const float *__restrict__ img, int H, int W) {
    const int wp = W + 2, rows = (H + 2) * wp;
    const int p = blockIdx.x * 32 + (threadIdx.x >> 3), k0 = (threadIdx.x & 7) * 8; /* eight elements (16 bytes) per thread */
    if (p >= rows) return;
    const int py = p / wp, px = p - py * wp;
    bf16x8 o;
#pragma unroll
    for (int e = 0; e < 8; e++) {
        const int k = k0 + e;
        float v = 0.0f;
        if (k < 27) {
            const int tap = k / 3, c = k - tap * 3, ky = tap / 3, kx = tap - ky * 3;
            const int y = py - 2 + ky, x = px - 2 + kx; /* image coordinates: bordered position minus 1, tap offset minus 1 */
            if (y >= 0 && y < H && x >= 0 && x < W) v = img[((size_t)c * H + y) * W + x];
        }
        o[e] = (bf16)v;
    }
    *(bf16x8 *)(out + (size_t)p * 64 + k0) = o;
}

/* The downsampling step (flux_vae.c:363-377: one row of zeros below and one column on the right,
 * then a 3x3 convolution with stride 2): fp32 [hp*wp, C] -> bf16 [hp2*wp2, 9*C] over the bordered
 * half-size grid, row (y', x') holding in[2(y'-1)+ky, 2(x'-1)+kx] for the nine taps, in the K order
 * of flux_hip_conv's weights ([C/64 chunks][9 taps][64 channels]), so that the convolution is a
 * plain GEMM with K = 9*C over these rows. The input's own zero border
 * supplies the padding: the furthest row read is its bottom border. Border rows of the output
 * are zero. One thread per (position, tap, 4 channels). */
__global__ __launch_bounds__(256) void vae_downsample_gather_kernel(bf16 *__restrict__ out, const float *__restrict__ x, int hp, int wp, int C) {
    const int quads = C >> 2;
    const int H2 = (hp - 2) >> 1, W2 = (wp - 2) >> 1, hp2 = H2 + 2, wp2 = W2 + 2;
    const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (size_t)hp2 * wp2 * 9 * quads) return;
    const int q = (int)(idx % quads);
    const size_t pt = idx / quads;
    const int tap = (int)(pt % 9), p = (int)(pt / 9);
    const int y = p / wp2, xx = p - y * wp2;
    bf16x4 o = {(bf16)0.0f, (bf16)0.0f, (bf16)0.0f, (bf16)0.0f};
    if (y >= 1 && y <= H2 && xx >= 1 && xx <= W2) {
        const int ky = tap / 3, kx = tap - ky * 3;
        const int sy = 2 * (y - 1) + ky + 1, sx = 2 * (xx - 1) + kx + 1; /* bordered input coordinates, at most hp-1 / wp-1 */
        const f32x4 v = *(const f32x4 *)(x + ((size_t)sy * wp + sx) * C + q * 4);
#pragma unroll
        for (int e = 0; e < 4; e++) o[e] = (bf16)v[e];
    }
    const int c = q * 4;
    *(bf16x4 *)(out + (size_t)p * 9 * C + ((c >> 6) * 9 + tap) * 64 + (c & 63)) = o;
}

/* Output of the quant convolution, fp32 [(2h+2)*(2w+2), ldx] (channels 0..31 = the posterior's
 * mean, flux_vae.c:411-424) -> 2x2 patchify to 128 channels (flux_kernels.c:1038-1065) ->
 * (v - running_mean) / sqrt(running_var + eps) (flux_kernels.c:555-575) -> latent [128, h, w]. */
__global__ __launch_bounds__(256) void vae_latent_out_kernel(float *__restrict__ latent, const float *__restrict__ x, int ldx,
                                                             const float *__restrict__ bn_mean, const float *__restrict__ bn_var, int h, int w,
                                                             float eps) {
    const int idx = blockIdx.x * 256 + threadIdx.x;
    if (idx >= 128 * h * w) return;
    const int lc = idx / (h * w), r = idx - lc * (h * w), ph = r / w, pw = r - ph * w;
    const int c = lc >> 2, pi = (lc >> 1) & 1, pj = lc & 1, wp = 2 * w + 2;
    const float v = x[((size_t)(2 * ph + pi + 1) * wp + (2 * pw + pj + 1)) * ldx + c];
    latent[idx] = (v - bn_mean[lc]) / sqrtf(bn_var[lc] + eps);
}

/* ---- attention over all positions with one head (attnblock_forward, flux_vae.c:223-313).
 * Scores are materialised, as in the reference: S = q k^T (GEMM), P = softmax(S * scale + bias)
 * (below), O = P v (GEMM against v^T). Queries and keys are the image's interior positions, packed; keys are padded up to a
 * multiple of 256, and key_bias is 0 for real ones and -inf for the padding columns. ---- */
__global__ __launch_bounds__(256) void vae_key_bias_kernel(float *__restrict__ bias, int n, int keys) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    bias[i] = i < keys ? 0.0f : -INFINITY;
}

__global__ __launch_bounds__(256) void vae_softmax_kernel(bf16 *__restrict__ P, const float *__restrict__ S, const float *__restrict__ key_bias,
                                                          int ld, float scale) {
    __shared__ float red[4];
    const float *s = S + (size_t)blockIdx.x * ld;
    bf16 *p = P + (size_t)blockIdx.x * ld;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    float mx = -INFINITY;
    for (int i = threadIdx.x * 4; i < ld; i += 1024) {
        const f32x4 v = *(const f32x4 *)(s + i), kb = *(const f32x4 *)(key_bias + i);
#pragma unroll
        for (int e = 0; e < 4; e++) mx = fmaxf(mx, v[e] * scale + kb[e]);
    }
    for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
    if (lane == 0) red[wave] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    __syncthreads();
    float sum = 0.0f;
    for (int i = threadIdx.x * 4; i < ld; i += 1024) {
        const f32x4 v = *(const f32x4 *)(s + i), kb = *(const f32x4 *)(key_bias + i);
#pragma unroll
        for (int e = 0; e < 4; e++) sum += __expf(v[e] * scale + kb[e] - mx);
    }
    for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
    if (lane == 0) red[wave] = sum;
    __syncthreads();
    const float inv = 1.0f / (red[0] + red[1] + red[2] + red[3]);
    for (int i = threadIdx.x * 4; i < ld; i += 1024) {
        const f32x4 v = *(const f32x4 *)(s + i), kb = *(const f32x4 *)(key_bias + i);
        bf16x4 o;
#pragma unroll
        for (int e = 0; e < 4; e++) o[e] = (bf16)(__expf(v[e] * scale + kb[e] - mx) * inv);
        *(bf16x4 *)(p + i) = o;
    }
}

/* The same for rows of up to 1024 * SOFTMAX_REG_V4 * 4 columns (1024x1024 images have 16384), with
 * the row held in registers between the three steps: S is read once. */
#define SOFTMAX_REG_V4 20
__global__ __launch_bounds__(256) void vae_softmax_reg_kernel(bf16 *__restrict__ P, const float *__restrict__ S, const float *__restrict__ key_bias,
                                                              int ld, float scale) {
    __shared__ float red[4];
    const float *s = S + (size_t)blockIdx.x * ld;
    bf16 *p = P + (size_t)blockIdx.x * ld;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    f32x4 v[SOFTMAX_REG_V4];
    float mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < SOFTMAX_REG_V4; i++) {
        const int c = (i * 256 + threadIdx.x) * 4;
        if (c < ld) {
            const f32x4 t = *(const f32x4 *)(s + c), kb = *(const f32x4 *)(key_bias + c);
#pragma unroll
            for (int e = 0; e < 4; e++) { v[i][e] = t[e] * scale + kb[e]; mx = fmaxf(mx, v[i][e]); }
        }
    }
    for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
    if (lane == 0) red[wave] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    __syncthreads();
    float sum = 0.0f;
#pragma unroll
    for (int i = 0; i < SOFTMAX_REG_V4; i++)
        if ((i * 256 + threadIdx.x) * 4 < ld) {
#pragma unroll
            for (int e = 0; e < 4; e++) { v[i][e] = __expf(v[i][e] - mx); sum += v[i][e]; }
        }
    for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
    if (lane == 0) red[wave] = sum;
    __syncthreads();
    const float inv = 1.0f / (red[0] + red[1] + red[2] + red[3]);
#pragma unroll
    for (int i = 0; i < SOFTMAX_REG_V4; i++) {
        const int c = (i * 256 + threadIdx.x) * 4;
        if (c < ld) {
            bf16x4 o;
#pragma unroll
            for (int e = 0; e < 4; e++) o[e] = (bf16)(v[i][e] * inv);
            *(bf16x4 *)(p + c) = o;
        }
    }
}

/* ---- the same attention for many positions, without the scores: P leaves the first product as 2^(scale score - reference)
 * (flux_hip_linear_exp), the second product is divided by the row sums. A softmax does not care about its reference as long as
 * nothing overflows: here it is the row's largest score over 256 keys spread over the image (2 to 3 % of the first product's work). A row
 * with a score more than 2^100 above that - its sums show it - is computed once more by a kernel of its own. In a decode
 * of 1024 x 1024 (16384 positions): 394 us of scores + 347 of softmax + 222 of P v with the scores in memory; now 18 + 295 + 244, of which
 * the exponentials, which nothing overlaps, are about 80. (In chunks whose P the memory-side cache would hold it is no faster.) ---- */
#define ATT_C 512          /* channels of the one head */
#define ATT_SAMPLE 256     /* keys that give the reference */
#define ATT_SUM_MAX 0x1p100f

/* ref[row] = scale * the largest of the row's ATT_SAMPLE scores; one wave per row */
__global__ __launch_bounds__(256) void vae_attention_ref_kernel(float *__restrict__ ref, const float *__restrict__ s, int n, float scale) {
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (row >= n) return;
    const f32x4 v = *(const f32x4 *)(s + (size_t)row * ATT_SAMPLE + lane * 4);
    float m = fmaxf(fmaxf(v[0], v[1]), fmaxf(v[2], v[3]));
    for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
    if (lane == 0) ref[row] = m * scale;
}

__device__ __forceinline__ float wave_sum(float v) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
}

/* out[row] = (sum of the slices) / (sum of the row's sums), one wave per row, eight channels per lane; missed[row] = 1 where a sum says that
 * the reference was too low, else 0 */
__global__ __launch_bounds__(256) void vae_attention_out_kernel(bf16 *__restrict__ out, float *__restrict__ missed, const float *__restrict__ o, int slices,
                                                                const float *__restrict__ sums, int pieces, int n) {
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63, c = lane * 8;
    if (row >= n) return;
    const size_t slice = (size_t)n * ATT_C;
    float acc[8];
#pragma unroll
    for (int e = 0; e < 8; e++) acc[e] = 0.0f;
    for (int k = 0; k < slices; k++) {
        const f32x4 *p = (const f32x4 *)(o + k * slice + (size_t)row * ATT_C + c);
        const f32x4 a = p[0], b = p[1];
#pragma unroll
        for (int e = 0; e < 4; e++) { acc[e] += a[e]; acc[4 + e] += b[e]; }
    }
    float sum = 0.0f;
    bool beyond = false;
    for (int i = lane; i < pieces; i += 64) {
        const float v = sums[(size_t)row * pieces + i];
        sum += v;
        beyond = beyond || v > ATT_SUM_MAX;
    }
    sum = wave_sum(sum);
    beyond = __any(beyond);
    if (lane == 0) missed[row] = beyond ? 1.0f : 0.0f;
    const float inv = 1.0f / sum;
    bf16x8 r;
#pragma unroll
    for (int e = 0; e < 8; e++) r[e] = (bf16)(acc[e] * inv);
    *(bf16x8 *)(out + (size_t)row * ATT_C + c) = r;
}

/* The rows that missed, anew. A workgroup looks at 16 rows at a time (usually none of them missed), each of its waves takes every fourth run of 32
 * keys with a running maximum, and the four results are joined. S^T = K Q^T leaves a lane four scores of one row and block; the second block's keys lie
 * between the first one's, so that the lane's eight are those it holds of the second product's operand. Probabilities stay fp32 as far as
 * two bf16 operands carry them (2^-17). What bounds it is how long the loads of a run take: one wave per SIMD, whose 32 of K and then of V are requested
 * together. Attention over 16384 positions, us: 590 with no row missed, 1740 with one, 4250 with all (4096: 64, 311, 304); key by key in one wave, with a
 * reduction for each score, one row took 19900 (3790). The launch itself is 2 us. */
#define REDO_ROWS 16
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void vae_attention_redo_kernel(
    bf16 *__restrict__ out, const float *__restrict__ missed, const bf16 *__restrict__ q, const bf16 *__restrict__ qkv, const bf16 *__restrict__ vt, int n, int keys,
    int ld, float scale) {
    __shared__ __attribute__((aligned(16))) float so[REDO_ROWS][ATT_C + 4];
    __shared__ float sm[4][REDO_ROWS], sl[4][REDO_ROWS];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l15 = lane & 15, lq = lane >> 4;
    constexpr int KS = ATT_C / 32, CB = ATT_C / 16;
    constexpr float LOW = -3.402823466e38f; /* finite: no difference of two of them is NaN */
    const __amdgpu_buffer_rsrc_t kbuf = __builtin_amdgcn_make_buffer_rsrc((void *)qkv, 0, (int)((unsigned)ld * 3 * ATT_C * 2), 0x00020000);
    const __amdgpu_buffer_rsrc_t vbuf = __builtin_amdgcn_make_buffer_rsrc((void *)vt, 0, (int)((unsigned)ld * ATT_C * 2), 0x00020000);
    const auto load = [](__amdgpu_buffer_rsrc_t b, unsigned off, int soff) { return __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(b, off, soff, 0)); };
    for (int r0 = blockIdx.x * REDO_ROWS; r0 < n; r0 += gridDim.x * REDO_ROWS) {
        if (!__any(r0 + l15 < n && missed[min(r0 + l15, n - 1)] != 0.0f)) continue; /* the same in all four waves */
        bf16x8 fq[KS], f[KS];
#pragma unroll
        for (int k = 0; k < KS; k++) fq[k] = *(const bf16x8 *)(q + (size_t)min(r0 + l15, n - 1) * 3 * ATT_C + 32 * k + 8 * lq);
        f32x4 o[CB];
#pragma unroll
        for (int i = 0; i < CB; i++) o[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        float m = LOW, l = 0.0f;
        for (int k0 = 32 * wave; k0 < ld; k0 += 128) { /* ld is a multiple of 256, and every wave's first run has keys */
            float p[8], mx = m;
#pragma unroll
            for (int b = 0; b < 2; b++) {
                const unsigned at = (unsigned)((k0 + 8 * (l15 >> 2) + 4 * b + (l15 & 3)) * 3 * ATT_C + ATT_C + 8 * lq) * 2u;
                f32x4 s = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int k = 0; k < KS; k++) f[k] = load(kbuf, at + 64 * k, 0);
#pragma unroll
                for (int k = 0; k < KS; k++) s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f[k], fq[k], s, 0, 0, 0);
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    p[4 * b + e] = k0 + 8 * lq + 4 * b + e < keys ? s[e] * scale : LOW;
                    mx = fmaxf(mx, p[4 * b + e]);
                }
            }
            mx = fmaxf(mx, __shfl_xor(mx, 16));
            mx = fmaxf(mx, __shfl_xor(mx, 32));
            if (__any(mx > m)) {
                const float a = fast_exp2(m - mx);
                l *= a;
#pragma unroll
                for (int i = 0; i < CB; i++)
#pragma unroll
                    for (int e = 0; e < 4; e++) o[i][e] *= a;
                m = mx;
            }
            bf16x8 hi, lo;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float v = k0 + 8 * lq + e < keys ? fast_exp2(p[e] - m) : 0.0f;
                l += v;
                hi[e] = (bf16)v;
                lo[e] = (bf16)(v - (float)hi[e]);
            }
#pragma unroll
            for (int h = 0; h < CB; h += KS) {
#pragma unroll
                for (int i = 0; i < KS; i++) f[i] = load(vbuf, (unsigned)(l15 * ld + k0 + 8 * lq) * 2u, 32 * (h + i) * ld);
#pragma unroll
                for (int i = 0; i < KS; i++) {
                    o[h + i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f[i], hi, o[h + i], 0, 0, 0);
                    o[h + i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f[i], lo, o[h + i], 0, 0, 0);
                }
            }
        }
        l += __shfl_xor(l, 16);
        l += __shfl_xor(l, 32);
        if (lq == 0) {
            sm[wave][l15] = m;
            sl[wave][l15] = l;
        }
        __syncthreads();
        const float share = fast_exp2(m - fmaxf(fmaxf(sm[0][l15], sm[1][l15]), fmaxf(sm[2][l15], sm[3][l15])));
        for (int w = 0; w < 4; w++) {
            if (wave == w)
#pragma unroll
                for (int i = 0; i < CB; i++) {
                    f32x4 *d = (f32x4 *)&so[l15][16 * i + 4 * lq];
                    f32x4 v = w ? *d : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                    for (int e = 0; e < 4; e++) v[e] += o[i][e] * share;
                    *d = v;
                }
            __syncthreads();
        }
        const int r = threadIdx.x >> 4, c0 = (threadIdx.x & 15) * 8, row = r0 + r;
        if (row < n && missed[row] != 0.0f) {
            const float top = fmaxf(fmaxf(sm[0][r], sm[1][r]), fmaxf(sm[2][r], sm[3][r]));
            float sum = 0.0f;
#pragma unroll
            for (int w = 0; w < 4; w++) sum += sl[w][r] * fast_exp2(sm[w][r] - top);
            const float inv = 1.0f / sum;
#pragma unroll
            for (int k = 0; k < 4; k++) {
                bf16x8 v;
#pragma unroll
                for (int e = 0; e < 8; e++) v[e] = (bf16)(so[r][c0 + 128 * k + e] * inv);
                *(bf16x8 *)(out + (size_t)row * ATT_C + c0 + 128 * k) = v;
            }
        }
        __syncthreads(); /* the next 16 rows write the same LDS */
    }
}

/* vt[c][j] = v[j][c] for j < rows, 0 for rows <= j < ld: the value matrix as the "weight" operand
 * of the second attention GEMM. 64 x 64 tiles through LDS. */
__global__ __launch_bounds__(256) void vae_transpose_kernel(bf16 *__restrict__ vt, int ld, const bf16 *__restrict__ v, int ldv, int rows) {
    __shared__ bf16 tile[64][66];
    const int j0 = blockIdx.x * 64, c0 = blockIdx.y * 64;
    for (int i = threadIdx.x; i < 64 * 64; i += 256) {
        const int jj = i >> 6, cc = i & 63;
        tile[jj][cc] = (j0 + jj < rows) ? v[(size_t)(j0 + jj) * ldv + c0 + cc] : (bf16)0.0f;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < 64 * 64; i += 256) {
        const int cc = i >> 6, jj = i & 63;
        if (j0 + jj < ld) vt[(size_t)(c0 + cc) * ld + j0 + jj] = tile[jj][cc];
    }
}

/* ------------------------------------------------------------------ host entry points */

extern "C" int flux_hip_vae_latent_in(void *out_bf16, const float *latent, const float *bn_mean, const float *bn_var,
                                      const float *pq_w, const float *pq_b, int h, int w, float eps) {
    if (h <= 0 || w <= 0) return flux_hip_fail("flux_hip_vae_latent_in: bad size %d x %d", h, w);
    const int positions = (2 * h + 2) * (2 * w + 2);
    hipLaunchKernelGGL(vae_latent_kernel, dim3((positions + 8 * LATENT_TRIPS - 1) / (8 * LATENT_TRIPS)), dim3(256), 0, flux_hip_stream_handle(), (bf16 *)out_bf16, latent, bn_mean, bn_var,
                       pq_w, pq_b, h, w, eps);
    LAUNCH_OK("vae_latent_kernel");
    return 1;
}

/* mean and 1/sqrt(var + eps) of the 32 groups, at the head of the scratch */
template <typename T>
static int group_norm_statistics(const T *x, float *scratch, int hp, int wp, int C, float eps, const float *conv_stats, int conv_stats_rows) {
    const int rows = hp * wp, nblocks = (rows + GN_ROWS - 1) / GN_ROWS;
    float *partial = scratch + 64, *stats = scratch;
    hipStream_t st = flux_hip_stream_handle();
    const double count = (double)(hp - 2) * (wp - 2) * (C / 32);
    if (conv_stats && conv_stats_rows <= GN_ONE_PASS_ROWS) {
        hipLaunchKernelGGL(gn_stats_kernel, dim3(32), dim3(256), 0, st, stats, conv_stats, conv_stats_rows, C, count, eps);
        LAUNCH_OK("gn_stats_kernel");
    } else if (conv_stats) {
        const int rpi = 256 / (C / 4);
        int nb = (conv_stats_rows + 8 * rpi - 1) / (8 * rpi); /* about eight trips per thread, at most as many workgroups as the scratch has rows */
        nb = nb < 1 ? 1 : nb > nblocks ? nblocks : nb > 256 ? 256 : nb;
        hipLaunchKernelGGL(gn_fold_quads_kernel, dim3(nb), dim3(256), 0, st, partial, conv_stats, conv_stats_rows, C);
        LAUNCH_OK("gn_fold_quads_kernel");
        hipLaunchKernelGGL(gn_finalize_kernel, dim3(32), dim3(256), 0, st, stats, partial, nb, count, eps);
        LAUNCH_OK("gn_finalize_kernel");
    } else {
        hipLaunchKernelGGL(gn_partial_kernel<T>, dim3(nblocks), dim3(256), 0, st, partial, x, rows, C);
        LAUNCH_OK("gn_partial_kernel");
        hipLaunchKernelGGL(gn_finalize_kernel, dim3(32), dim3(256), 0, st, stats, partial, nblocks, count, eps);
        LAUNCH_OK("gn_finalize_kernel");
    }
    return 1;
}

template <typename T>
static int group_norm_run(void *out_bf16, void *raw_bf16, const T *x, const float *gamma, const float *beta, float *scratch, int hp, int wp,
                          int C, float eps, int swish, const float *conv_stats, int conv_stats_rows) {
    const int rows = hp * wp;
    hipStream_t st = flux_hip_stream_handle();
    const double count = (double)(hp - 2) * (wp - 2) * (C / 32);
    const unsigned long long magic = ((1ull << 40) + (unsigned)wp - 1) / (unsigned)wp;
    if (conv_stats && conv_stats_rows <= GN_FUSED_ROWS) {
        const int span = (rows + 63) / 64 * (C / 64) > 1024 ? 128 : 64;
        hipLaunchKernelGGL(gn_fused_kernel<T>, dim3((rows + span - 1) / span, C / 64), dim3(256), 0, st, (bf16 *)out_bf16, (bf16 *)raw_bf16, x, conv_stats,
                           conv_stats_rows, count, eps, gamma, beta, rows, C, hp, wp, magic, swish, span);
        LAUNCH_OK("gn_fused_kernel");
        return 1;
    }
    if (!group_norm_statistics(x, scratch, hp, wp, C, eps, conv_stats, conv_stats_rows)) return 0;
    const float *stats = scratch;
    /* as many positions per workgroup as leave 2048 workgroups, at least four per thread */
    int span = GN_ROWS;
    while (span > 4 * (256 / (C / 4)) && (rows + span - 1) / span < 2048) span >>= 1;
    hipLaunchKernelGGL(gn_apply_kernel<T>, dim3((rows + span - 1) / span), dim3(256), 0, st, (bf16 *)out_bf16, (bf16 *)raw_bf16, x, stats, gamma, beta, rows, C, hp,
                       wp, magic, swish, span);
    LAUNCH_OK("gn_apply_kernel");
    return 1;
}

extern "C" int flux_hip_group_norm_stats(void *out_bf16, void *raw_bf16, const void *x, int x_is_bf16, const float *gamma, const float *beta,
                                         float *scratch, int hp, int wp, int C, float eps, int swish, const float *conv_stats,
                                         int conv_stats_rows) {
    if (C != 128 && C != 256 && C != 512) return flux_hip_fail("flux_hip_group_norm: C=%d (128, 256 or 512)", C);
    if (hp < 3 || wp < 3 || wp >= 4096 || (long long)hp * wp >= (1 << 22)) return flux_hip_fail("flux_hip_group_norm: bad image %d x %d", hp, wp);
    if (conv_stats && conv_stats_rows <= 0) return flux_hip_fail("flux_hip_group_norm_stats: conv_stats_rows=%d", conv_stats_rows);
    return x_is_bf16 ? group_norm_run(out_bf16, raw_bf16, (const bf16 *)x, gamma, beta, scratch, hp, wp, C, eps, swish, conv_stats, conv_stats_rows)
                     : group_norm_run(out_bf16, raw_bf16, (const float *)x, gamma, beta, scratch, hp, wp, C, eps, swish, conv_stats, conv_stats_rows);
}

/* The first norm (with swish) of a residual block whose channel counts differ, and its 1x1 shortcut: y = conv(bf16(x)) as flux_hip_conv's fp32 epilogue
 * writes it. w: [cout][cin]; raw: room for a bf16 copy of x, which only the two launches of small images use. */
extern "C" int flux_hip_vae_group_norm_skip(void *out_bf16, void *raw_bf16, float *y, const float *x, const float *gamma, const float *beta, float *scratch, int hp,
                                            int wp, int cin, float eps, const float *conv_stats, int conv_stats_rows, const void *w, const float *bias, int cout) {
    if (cin != 128 && cin != 256 && cin != 512) return flux_hip_fail("flux_hip_vae_group_norm_skip: %d channels (128, 256 or 512)", cin);
    if (hp < 3 || wp < 3 || (long long)hp * wp >= 1 << 22 || wp >= 1 << 12 || cout <= 0 || cout % 128)
        return flux_hip_fail("flux_hip_vae_group_norm_skip: bad shape (hp=%d wp=%d cout=%d)", hp, wp, cout);
    if (!out_bf16 || !raw_bf16 || !y || !x || !gamma || !beta || !scratch || !w || !bias) return flux_hip_fail("flux_hip_vae_group_norm_skip: NULL argument");
    if (conv_stats && conv_stats_rows <= 0) return flux_hip_fail("flux_hip_vae_group_norm_skip: conv_stats_rows=%d", conv_stats_rows);
    if (((uintptr_t)out_bf16 | (uintptr_t)raw_bf16 | (uintptr_t)y | (uintptr_t)x | (uintptr_t)gamma | (uintptr_t)beta | (uintptr_t)w | (uintptr_t)bias) & 15)
        return flux_hip_fail("flux_hip_vae_group_norm_skip: operands must be 16-byte aligned");
    const int rows = hp * wp, P = cin == 512 ? 64 : 128;
    /* Two launches of more workgroups win where this one leaves most units with none or one: decoder, 128 x 128 x 512 -> 256 (265 workgroups) 31 + 5 us for the
     * sums against 30, 128 x 128 x 256 -> 128 (133) no difference; encoder 128 x 128 x 128 -> 256 (133) 10 us longer together with 64 x 64 x 256 -> 512,
     * 160 x 160 (206) 8 us shorter. */
    if ((rows + P - 1) / P < (cin == 512 ? 300 : 150))
        return flux_hip_group_norm_stats(out_bf16, raw_bf16, x, 0, gamma, beta, scratch, hp, wp, cin, eps, 1, conv_stats, conv_stats_rows) &&
               flux_hip_conv_stats(FLUX_HIP_EPI_CONV_F32, raw_bf16, w, bias, nullptr, y, rows, wp, cin, cout, 1, nullptr, nullptr);
    if (!group_norm_statistics(x, scratch, hp, wp, cin, eps, conv_stats, conv_stats_rows)) return 0;
    const unsigned long long magic = ((1ull << 40) + (unsigned)wp - 1) / (unsigned)wp;
    auto kern = cin == 128 ? gn_skip_kernel<128, 128> : cin == 256 ? gn_skip_kernel<256, 128> : gn_skip_kernel<512, 64>;
    const int slot = conv_probe_begin(FLUX_HIP_EPI_CONV_F32, 19);
    hipLaunchKernelGGL(kern, dim3((rows + P - 1) / P), dim3(512), 0, flux_hip_stream_handle(), (bf16 *)out_bf16, y, x, scratch, gamma, beta, (const bf16 *)w, bias, rows,
                       cout, hp, wp, magic);
    conv_probe_end(slot);
    LAUNCH_OK("gn_skip_kernel");
    return 1;
}

extern "C" int flux_hip_group_norm(void *out_bf16, void *raw_bf16, const void *x, int x_is_bf16, const float *gamma, const float *beta,
                                   float *scratch, int hp, int wp, int C, float eps, int swish) {
    return flux_hip_group_norm_stats(out_bf16, raw_bf16, x, x_is_bf16, gamma, beta, scratch, hp, wp, C, eps, swish, nullptr, 0);
}

extern "C" size_t flux_hip_group_norm_scratch_floats(int hp, int wp) {
    return 64 + (size_t)((hp * wp + GN_ROWS - 1) / GN_ROWS) * 64;
}

extern "C" int flux_hip_upsample2x(void *out_bf16, const float *x, int hp, int wp, int C) {
    if (C <= 0 || (C & 3) || hp < 3 || wp < 3) return flux_hip_fail("flux_hip_upsample2x: bad shape");
    const size_t total = (size_t)hp * wp * (C / 4);
    hipLaunchKernelGGL((vae_upsample_kernel<float, 4>), dim3((unsigned)((total + 255) / 256)), dim3(256), 0, flux_hip_stream_handle(), (bf16 *)out_bf16,
                       x, hp, wp, C);
    LAUNCH_OK("vae_upsample_kernel");
    return 1;
}

/* the same from a bf16 image, C a multiple of 8 */
extern "C" int flux_hip_vae_upsample2x_bf16(void *out_bf16, const void *x_bf16, int hp, int wp, int C) {
    if (C <= 0 || (C & 7) || hp < 3 || wp < 3) return flux_hip_fail("flux_hip_vae_upsample2x_bf16: bad shape");
    const size_t total = (size_t)hp * wp * (C / 8);
    hipLaunchKernelGGL((vae_upsample_kernel<bf16, 8>), dim3((unsigned)((total + 255) / 256)), dim3(256), 0, flux_hip_stream_handle(), (bf16 *)out_bf16,
                       (const bf16 *)x_bf16, hp, wp, C);
    LAUNCH_OK("vae_upsample_kernel");
    return 1;
}

extern "C" int flux_hip_vae_image_in(void *out_bf16, const float *img, int H, int W) {
    if (H <= 0 || W <= 0) return flux_hip_fail("flux_hip_vae_image_in: bad shape");
    const int rows = (H + 2) * (W + 2);
    hipLaunchKernelGGL(vae_image_in_kernel, dim3((rows + 31) / 32), dim3(256), 0, flux_hip_stream_handle(), (bf16 *)out_bf16, img, H, W);
    LAUNCH_OK("vae_image_in_kernel");
    return 1;
}

extern "C" int flux_hip_downsample_gather(void *out_bf16, const float *x, int hp, int wp, int C) {
    if (C <= 0 || (C & 3) || hp < 4 || wp < 4 || ((hp | wp) & 1)) return flux_hip_fail("flux_hip_downsample_gather: bad shape (the image must have even sides)");
    const size_t total = (size_t)((hp - 2) / 2 + 2) * ((wp - 2) / 2 + 2) * 9 * (C / 4);
    hipLaunchKernelGGL(vae_downsample_gather_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, flux_hip_stream_handle(), (bf16 *)out_bf16,
                       x, hp, wp, C);
    LAUNCH_OK("vae_downsample_gather_kernel");
    return 1;
}

extern "C" int flux_hip_vae_latent_out(float *latent, const float *x, int ldx, const float *bn_mean, const float *bn_var, int h, int w, float eps) {
    if (h <= 0 || w <= 0 || ldx < 32) return flux_hip_fail("flux_hip_vae_latent_out: bad shape");
    hipLaunchKernelGGL(vae_latent_out_kernel, dim3((128 * h * w + 255) / 256), dim3(256), 0, flux_hip_stream_handle(), latent, x, ldx, bn_mean,
                       bn_var, h, w, eps);
    LAUNCH_OK("vae_latent_out_kernel");
    return 1;
}

extern "C" int flux_hip_vae_key_bias(float *bias, int n, int keys) {
    hipLaunchKernelGGL(vae_key_bias_kernel, dim3((n + 255) / 256), dim3(256), 0, flux_hip_stream_handle(), bias, n, keys);
    LAUNCH_OK("vae_key_bias_kernel");
    return 1;
}

extern "C" int flux_hip_softmax_rows(void *p_bf16, const float *s, const float *key_bias, int rows, int ld, float scale) {
    if (rows <= 0 || ld <= 0 || (ld & 3)) return flux_hip_fail("flux_hip_softmax_rows: bad shape %d x %d", rows, ld);
    if (ld <= 1024 * SOFTMAX_REG_V4)
        hipLaunchKernelGGL(vae_softmax_reg_kernel, dim3(rows), dim3(256), 0, flux_hip_stream_handle(), (bf16 *)p_bf16, s, key_bias, ld, scale);
    else
        hipLaunchKernelGGL(vae_softmax_kernel, dim3(rows), dim3(256), 0, flux_hip_stream_handle(), (bf16 *)p_bf16, s, key_bias, ld, scale);
    LAUNCH_OK("vae_softmax_kernel");
    return 1;
}

extern "C" int flux_hip_linear_exp_available(void);
extern "C" int flux_hip_linear_exp(const void *A, const void *W, void *P, int M, int N, int K, int lda, int ldw, const float *ref, float scale, int keys,
                                   float *sums, int *pieces);
extern "C" int flux_hip_linear_f32_slices(const void *A, const void *W, float *C, int M, int N, int K, const float **ws, int *slices);

extern "C" size_t flux_hip_vae_attention_work_floats(int n, int ld) { return (size_t)n * (ATT_SAMPLE + 1 + ld / 64) + 4; }

/* The reference's keys are 0, step, 2 step, ...: the largest step that stays within the image and has no factor in common with
 * its positions, hence none with its width. Multiples of it then fall on as many columns as there are samples (every 64th of 128 x 128
 * positions are two columns, one of them at the border). From 2560 positions on that is at most 13 below the largest that stays within, and the
 * samples span 46 % of the image at least. */
extern "C" int flux_hip_vae_attention_sample_step(int keys) {
    const auto common = [](int a, int b) {
        while (b) { const int r = a % b; a = b; b = r; }
        return a;
    };
    int step = keys / ATT_SAMPLE;
    while (step > 1 && common(keys, step) != 1) step--;
    return step;
}

/* Attention of n queries (rows of qkv from q on, 3 * 512 wide) over `keys` positions: out [n][512]. qkv: every position's [q | k | v], ld rows of
 * them (zeros beyond keys); vt: v transposed, [512][ld]; P: n x ld bf16; o32: n x 512; work: flux_hip_vae_attention_work_floats. At least
 * 256 keys, ld a multiple of 256. *done = 0 where the scores' kernel is switched off: nothing is launched. */
extern "C" int flux_hip_vae_attention(void *out, const void *q, const void *qkv, const void *vt, void *P, float *o32, float *work, int n, int keys, int ld,
                                      float scale, int *done) {
    *done = 0;
    if (n <= 0 || keys < ATT_SAMPLE || ld < keys || (ld & 255)) return flux_hip_fail("flux_hip_vae_attention: bad shape (%d queries, %d keys, %d columns)", n, keys, ld);
    if (!flux_hip_linear_exp_available()) return 1;
    const float scale2 = scale * 1.44269504088896341f;
    float *sample = work, *ref = work + (size_t)n * ATT_SAMPLE, *sums = ref + ((n + 3) & ~3);
    hipStream_t st = flux_hip_stream_handle();
    const bf16 *k = (const bf16 *)qkv + ATT_C;
    flux_hip_linear_part sp = {q, k, sample, nullptr, n};
    if (!flux_hip_linear(FLUX_HIP_EPI_F32, 1, &sp, ATT_SAMPLE, ATT_C, 3 * ATT_C, flux_hip_vae_attention_sample_step(keys) * 3 * ATT_C, ATT_SAMPLE, 0, 0)) return 0;
    hipLaunchKernelGGL(vae_attention_ref_kernel, dim3((n + 3) / 4), dim3(256), 0, st, ref, sample, n, scale2);
    LAUNCH_OK("vae_attention_ref_kernel");
    int pieces = 0, slices = 0;
    if (!flux_hip_linear_exp(q, k, P, n, ld, ATT_C, 3 * ATT_C, 3 * ATT_C, ref, scale2, keys, sums, &pieces)) return 0;
    const float *ws = nullptr;
    if (!flux_hip_linear_f32_slices(P, vt, o32, n, ATT_C, ld, &ws, &slices)) return 0;
    hipLaunchKernelGGL(vae_attention_out_kernel, dim3((n + 3) / 4), dim3(256), 0, st, (bf16 *)out, ref, slices ? ws : o32, slices ? slices : 1, sums, pieces, n);
    LAUNCH_OK("vae_attention_out_kernel");
    hipLaunchKernelGGL(vae_attention_redo_kernel, dim3(min((n + REDO_ROWS - 1) / REDO_ROWS, 256)), dim3(256), 0, st, (bf16 *)out, ref, (const bf16 *)q, (const bf16 *)qkv,
                       (const bf16 *)vt, n, keys, ld, scale2);
    LAUNCH_OK("vae_attention_redo_kernel");
    *done = 1;
    return 1;
}

extern "C" int flux_hip_transpose_bf16(void *vt, int ld, const void *v, int ldv, int rows, int cols) {
    if (cols <= 0 || (cols & 63) || ld < rows) return flux_hip_fail("flux_hip_transpose_bf16: bad shape");
    hipLaunchKernelGGL(vae_transpose_kernel, dim3((ld + 63) / 64, cols / 64), dim3(256), 0, flux_hip_stream_handle(), (bf16 *)vt, ld, (const bf16 *)v,
                       ldv, rows);
    LAUNCH_OK("vae_transpose_kernel");
    return 1;
}
