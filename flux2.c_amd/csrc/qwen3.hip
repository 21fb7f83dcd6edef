/*
 * qwen3.hip - the kernels of the Qwen3 text encoder that are not GEMMs (reference: CPU arms of
 * flux_qwen3.c): embedding lookup, RMS norm, per-head RMS norm + rotate-half RoPE, causal
 * grouped-query attention with a padding mask, and the copy that collects three layers' hidden
 * states side by side. The projections and the MLP run through flux_hip_linear (gemm.hip).
 */
#include "common.h"
#include "../../include/flux_hip.h"
#include <math.h>

#define LAUNCH_OK(what)                                                                         \
    do {                                                                                        \
        hipError_t e_ = hipGetLastError();                                                      \
        if (e_ != hipSuccess) return flux_hip_fail("%s launch failed: %s", what, hipGetErrorString(e_)); \
    } while (0)

/* x[s] = embed[ids[s]], or zeros for an id outside the vocabulary (qwen3_forward,
 * flux_qwen3.c:1046-1056). One workgroup per token. */
__global__ __launch_bounds__(256) void qwen3_embed_kernel(float *__restrict__ x, const bf16 *__restrict__ embed, const int *__restrict__ ids,
                                                          int hidden, int vocab) {
    const int s = blockIdx.x, id = ids[s];
    const bool ok = id >= 0 && id < vocab;
    for (int i = threadIdx.x; i < hidden; i += 256) x[(size_t)s * hidden + i] = ok ? (float)embed[(size_t)id * hidden + i] : 0.0f;
}

/* out bf16 = x / sqrt(mean(x^2) + eps) * w per row (qwen3_rms_norm, flux_qwen3.c:177-197) */
__global__ __launch_bounds__(256) void qwen3_rms_norm_kernel(bf16 *__restrict__ out, const float *__restrict__ x, const float *__restrict__ w,
                                                             int hidden, float eps) {
    __shared__ float red[4];
    const float *xr = x + (size_t)blockIdx.x * hidden;
    float ss = 0.0f;
    for (int i = threadIdx.x * 4; i < hidden; i += 1024) {
        const f32x4 v = *(const f32x4 *)(xr + i);
        ss += v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + v[3] * v[3];
    }
    for (int o = 32; o > 0; o >>= 1) ss += __shfl_xor(ss, o);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
    __syncthreads();
    const float inv = 1.0f / sqrtf((red[0] + red[1] + red[2] + red[3]) / hidden + eps);
    for (int i = threadIdx.x * 4; i < hidden; i += 1024) {
        const f32x4 v = *(const f32x4 *)(xr + i), g = *(const f32x4 *)(w + i);
        bf16x4 o;
#pragma unroll
        for (int e = 0; e < 4; e++) o[e] = (bf16)(v[e] * inv * g[e]);
        *(bf16x4 *)(out + (size_t)blockIdx.x * hidden + i) = o;
    }
}

/* In place on the fused projection output qkv bf16 [seq, (heads + 2 kv_heads) * 128]: every q and k
 * head gets RMS norm * weight over its 128 values (qwen3_head_rms_norm, flux_qwen3.c:199-220)
 * and rotate-half RoPE, pairs (i, i + 64) with the table's angle for (position, i)
 * (apply_rope, flux_qwen3.c:264-307). The v heads are written transposed to vt [kv_heads * 128, ldv] (keys contiguous), the
 * layout the attention kernel's second product reads.
 * 16 lanes share a head's row, four pairs each (8-byte accesses), 16 rows per workgroup; the v heads go through LDS in blocks of
 * 64 tokens, so that a dim's tokens leave as 16-byte stores. With one wave per row and a 2-byte store per lane and token
 * for V the launch took 10.8 us at 512 tokens x 48 heads. VEC = false: pointers or ldv that do not allow the wide accesses.
 * SLICES: the projection ran as K slices and its partial sums are read here, summed in slice order and rounded to bf16 as its second
 * pass would (which at 67 tokens was a launch of 4.8 us); the v columns of qkv are then not written. A thread's columns are requested
 * together, of several slices at a time: value by value, eight and two sums one after the other, 67 tokens took 5.9 us for 4.9. */
template <bool VEC, typename V4, typename T>
__device__ __forceinline__ V4 qw_load4(const T *p) {
    if (VEC) return *(const V4 *)p;
    V4 v;
#pragma unroll
    for (int e = 0; e < 4; e++) v[e] = p[e];
    return v;
}
template <bool VEC>
__device__ __forceinline__ void qw_store4(bf16 *p, bf16x4 v) {
    if (VEC) {
        *(bf16x4 *)p = v;
    } else {
#pragma unroll
        for (int e = 0; e < 4; e++) p[e] = v[e];
    }
}
template <bool VEC, bool SLICES>
__global__ __launch_bounds__(256) void qwen3_qk_rope_kernel(bf16 *__restrict__ qkv, bf16 *__restrict__ vt, int ldv, const float *__restrict__ q_w,
                                                            const float *__restrict__ k_w, const float *__restrict__ rope_cos,
                                                            const float *__restrict__ rope_sin, int seq, int heads, int kv_heads, float eps,
                                                            const float *__restrict__ ws, int slices) {
    __shared__ bf16 tile[64][130]; /* (rows of 65 words: a column's reads fall on different banks) */
    const int width = (heads + 2 * kv_heads) * 128, nqk = heads + kv_heads, rows = seq * nqk, qk_blocks = (rows + 15) / 16;
    /* n times four columns of the projection, at elements at[0 .. n): all of a slice's on their way together, and several slices' */
    const auto load = [&](auto &o, const size_t *at) {
        constexpr int n = sizeof(o) / sizeof(o[0]);
        if (!SLICES) {
#pragma unroll
            for (int i = 0; i < n; i++) o[i] = qw_load4<VEC, bf16x4>(qkv + at[i]);
            return;
        }
        f32x4 sum[n];
#pragma unroll
        for (int i = 0; i < n; i++) sum[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        constexpr int U = n > 2 ? 2 : 4;
        const size_t slice = (size_t)seq * width;
        for (int k = 0; k < slices; k += U) {
            f32x4 v[U][n];
#pragma unroll
            for (int u = 0; u < U; u++)
#pragma unroll
                for (int i = 0; i < n; i++)
                    if (k + u < slices) v[u][i] = *(const f32x4 *)(ws + (k + u) * slice + at[i]);
#pragma unroll
            for (int u = 0; u < U; u++)
                if (k + u < slices) {
#pragma unroll
                    for (int i = 0; i < n; i++)
#pragma unroll
                        for (int e = 0; e < 4; e++) sum[i][e] += v[u][i][e];
                }
        }
#pragma unroll
        for (int i = 0; i < n; i++)
#pragma unroll
            for (int e = 0; e < 4; e++) o[i][e] = (bf16)sum[i][e];
    };
    if ((int)blockIdx.x >= qk_blocks) { /* 64 tokens of a v head: transpose */
        const int vb = blockIdx.x - qk_blocks, vh = vb % kv_heads, s0 = vb / kv_heads * 64;
        size_t at[8];
        bf16x4 v[8];
#pragma unroll
        for (int i = 0; i < 8; i++) at[i] = (size_t)min(s0 + i * 8 + (int)(threadIdx.x >> 5), seq - 1) * width + (nqk + vh) * 128 + (threadIdx.x & 31) * 4;
        load(v, at);
#pragma unroll
        for (int i = 0; i < 8; i++)
#pragma unroll
            for (int e = 0; e < 4; e++) tile[i * 8 + (threadIdx.x >> 5)][(threadIdx.x & 31) * 4 + e] = v[i][e];
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int idx = i * 256 + threadIdx.x, d = idx >> 3, c = (idx & 7) * 8;
            bf16 *o = vt + (size_t)(vh * 128 + d) * ldv + s0 + c;
            bf16x8 v;
#pragma unroll
            for (int e = 0; e < 8; e++) v[e] = tile[c + e][d];
            if (VEC && s0 + c + 8 <= seq) {
                *(bf16x8 *)o = v;
            } else {
#pragma unroll
                for (int e = 0; e < 8; e++)
                    if (s0 + c + e < seq) o[e] = v[e];
            }
        }
        return;
    }
    const int row = min((int)blockIdx.x * 16 + (int)(threadIdx.x >> 4), rows - 1), i0 = (threadIdx.x & 15) * 4;
    const bool mine = (int)blockIdx.x * 16 + (int)(threadIdx.x >> 4) < rows;
    const int s = row / nqk, h = row - s * nqk;
    bf16 *p = qkv + (size_t)s * width + h * 128 + i0;
    const float *w = (h < heads ? q_w : k_w) + i0;
    const size_t at[2] = {(size_t)s * width + h * 128 + i0, (size_t)s * width + h * 128 + i0 + 64};
    const f32x4 w0 = qw_load4<VEC, f32x4>(w), w1 = qw_load4<VEC, f32x4>(w + 64);
    const f32x4 cs = qw_load4<VEC, f32x4>(rope_cos + s * 64 + i0), sn = qw_load4<VEC, f32x4>(rope_sin + s * 64 + i0);
    bf16x4 half[2];
    load(half, at);
    const bf16x4 lo = half[0], hi = half[1];
    float ss = 0.0f;
#pragma unroll
    for (int e = 0; e < 4; e++) ss += (float)lo[e] * (float)lo[e] + (float)hi[e] * (float)hi[e];
#pragma unroll
    for (int o = 8; o > 0; o >>= 1) ss += __shfl_xor(ss, o);
    const float inv = 1.0f / sqrtf(ss / 128.0f + eps);
    bf16x4 olo, ohi;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const float a = (float)lo[e] * inv * w0[e], b = (float)hi[e] * inv * w1[e];
        olo[e] = (bf16)(a * cs[e] - b * sn[e]);
        ohi[e] = (bf16)(a * sn[e] + b * cs[e]);
    }
    if (mine) {
        qw_store4<VEC>(p, olo);
        qw_store4<VEC>(p + 64, ohi);
    }
}

/*
 * Causal grouped-query attention, head_dim 128, up to 512 keys (qwen3_attention_forward,
 * flux_qwen3.c:352-437): scores = q.k / sqrt(128); a key after the query, or one whose mask entry
 * is 0, gets the score -1e9 (not -inf: a row with no admissible key then comes out uniform over all
 * seq columns, exactly as in the reference); softmax over all seq columns; out = P v.
 *
 * One workgroup per (16 queries, kv head): its waves are the query heads that share that kv head,
 * so each 32-key tile of K and of V^T is fetched once and shared through LDS (two slots; tiles travel global -> registers, D
 * of them on their way, then registers -> LDS, one barrier per tile). A tile is 16 MFMAs per wave, far less than the time
 * its load takes: with one tile on its way every step waited for memory, 22 us at 512 tokens x 32 heads. The V^T tiles continue
 * the K tiles' sequence, so the first ones arrive during the softmax. A wave keeps all scores of its 16 queries against all keys in registers
 * (S^T = K Q^T as 16 x 16 blocks, keys x queries: 32 blocks of 4 registers), so the softmax is
 * the plain three-step one. Inside each group of 32 keys the K rows are assigned to MFMA rows so
 * that a lane ends up with 8 consecutive keys of one query: that is the B-operand layout of the
 * second product O^T = V^T P^T. LDS rows are chunk-swizzled so that the 16 rows a fragment read
 * touches fall into different banks.
 */
#define QW_MAXT 16 /* 32-key steps: 512 keys */
__device__ __forceinline__ int qw_kswz(int j) { return (j & 15) ^ ((j >> 4) << 2); } /* K tile: 32 rows of 16 chunks */
__device__ __forceinline__ int qw_vswz(int d) { return (d >> 2) & 3; }               /* V^T tile: 128 rows of 4 chunks */

/* The body for NT 32-key steps, NT a compile-time constant (straight-line code). Steps beyond the
 * sequence read clamped rows and are masked like the padding of the last step. */
template <int NT, int G>
__device__ __forceinline__ void qwen3_attend(bf16 *__restrict__ out, const bf16 *__restrict__ qkv, const bf16 *__restrict__ vt, int ldv,
                                             const unsigned long long (&keep)[QW_MAXT / 2], int seq, int heads, int kv_heads, char *smem) {
    const int tid = threadIdx.x, lane = tid & 63, l15 = lane & 15, lq = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    constexpr int nthreads = 64 * G;
    const int q0 = blockIdx.x * 16, kh = blockIdx.y, h = kh * (heads / kv_heads) + wave;
    const int width = (heads + 2 * kv_heads) * 128;
    const float scale = 0.08838834764831845f; /* 1 / sqrt(128) */
    constexpr int per_lane = 512 / nthreads;  /* 16-byte chunks of a tile per lane: 8, 4, 2 or 1 */

    /* Q^T fragments (MFMA B operand): lane (query l15, lq) holds dims [32 ks + 8 lq, +8) */
    const int qrow = min(q0 + l15, seq - 1);
    bf16x8 qf[4];
#pragma unroll
    for (int ks = 0; ks < 4; ks++) qf[ks] = *(const bf16x8 *)(qkv + (size_t)qrow * width + h * 128 + ks * 32 + lq * 8);

    constexpr int D = NT < 8 / per_lane || per_lane > 8 ? NT : 8 / per_lane; /* tiles on their way: 32 registers */
    bf16x8 stage[D][per_lane];
    /* K tile t: LDS row j = key 32 t + j, 16 chunks of 8 dims, chunk c stored at c ^ kswz(j) */
    auto fetch_k = [&](int t) { /* into stage[t % D] */
#pragma unroll
        for (int u = 0; u < per_lane; u++)
            {
                const int idx = tid + u * nthreads, j = idx >> 4, c = idx & 15;
                stage[t % D][u] = *(const bf16x8 *)(qkv + (size_t)min(32 * t + j, seq - 1) * width + (heads + kh) * 128 + c * 8);
            }
    };
    auto put_k = [&](int t) {
#pragma unroll
        for (int u = 0; u < per_lane; u++)
            {
                const int idx = tid + u * nthreads, j = idx >> 4, c = idx & 15;
                *(bf16x8 *)(smem + (t & 1) * 8192 + j * 256 + ((c ^ qw_kswz(j)) << 4)) = stage[t % D][u];
            }
    };
    /* V^T tile t: LDS row d = head dim, 4 chunks of 8 keys, chunk c stored at c ^ vswz(d) */
    auto fetch_v = [&](int t) { /* into stage[(NT + t) % D] */
#pragma unroll
        for (int u = 0; u < per_lane; u++)
            {
                const int idx = tid + u * nthreads, d = idx >> 2, c = idx & 3;
                stage[(NT + t) % D][u] = *(const bf16x8 *)(vt + (size_t)(kh * 128 + d) * ldv + min(32 * t, ldv - 32) + c * 8);
            }
    };
    auto put_v = [&](int t) {
#pragma unroll
        for (int u = 0; u < per_lane; u++)
            {
                const int idx = tid + u * nthreads, d = idx >> 2, c = idx & 3;
                *(bf16x8 *)(smem + 16384 + (t & 1) * 8192 + d * 64 + ((c ^ qw_vswz(d)) << 4)) = stage[(NT + t) % D][u];
            }
    };

    f32x4 sc[2 * NT];
#pragma unroll
    for (int t = 0; t < D; t++) fetch_k(t);
    put_k(0);
    __syncthreads();
#pragma unroll
    for (int t = 0; t < NT; t++) {
        if (t + D < NT) fetch_k(t + D);
        else fetch_v(t + D - NT);
        const char *kt = smem + (t & 1) * 8192;
#pragma unroll
        for (int half = 0; half < 2; half++) {
            /* MFMA row m = l15 of this block is key 32 t + j with j = 8 (m / 4) + 4 half + (m % 4) */
            const int j = 8 * (l15 >> 2) + 4 * half + (l15 & 3);
            f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int ks = 0; ks < 4; ks++) {
                const bf16x8 kf = *(const bf16x8 *)(kt + j * 256 + (((ks * 4 + lq) ^ qw_kswz(j)) << 4));
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[ks], acc, 0, 0, 0);
            }
            sc[2 * t + half] = acc;
        }
        if (t + 1 < NT) {
            put_k(t + 1);
            __syncthreads();
        }
    }

    /* accumulator element e of block (t, half): query l15, key 32 t + 8 lq + 4 half + e */
    const int qi = q0 + l15;
    float mx = -3.0e38f;
#pragma unroll
    for (int t = 0; t < NT; t++) {
        const unsigned bits = (unsigned)(keep[t >> 1] >> (32 * (t & 1))) >> (8 * lq); /* this lane's 8 keys of step t */
#pragma unroll
        for (int half = 0; half < 2; half++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int key = 32 * t + 8 * lq + 4 * half + e;
                float v = sc[2 * t + half][e] * scale;
                if (key > qi || !((bits >> (4 * half + e)) & 1)) v = -1e9f;
                if (key >= seq) v = -INFINITY; /* padding of the last 32-key step: no column of the reference's matrix */
                sc[2 * t + half][e] = v;
                mx = fmaxf(mx, v);
            }
    }
    mx = fmaxf(mx, __shfl_xor(mx, 16));
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    float sum = 0.0f;
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int half = 0; half < 2; half++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float p = __expf(sc[2 * t + half][e] - mx);
                sc[2 * t + half][e] = p;
                sum += p;
            }
    sum += __shfl_xor(sum, 16);
    sum += __shfl_xor(sum, 32);
    const float inv = 1.0f / sum;

    /* O^T[d][q] = sum_key V^T[d][key] P^T[key][q]: A operand = V^T rows (lane: dim l15, keys
     * [32 t + 8 lq, +8)), B operand = this lane's 8 probabilities of step t */
    f32x4 o[8];
#pragma unroll
    for (int d = 0; d < 8; d++) o[d] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
    put_v(0);
    __syncthreads();
#pragma unroll
    for (int t = 0; t < NT; t++) {
        if (t + D < NT) fetch_v(t + D);
        const char *vtile = smem + 16384 + (t & 1) * 8192;
        bf16x8 pf;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            pf[e] = (bf16)(sc[2 * t][e] * inv);
            pf[4 + e] = (bf16)(sc[2 * t + 1][e] * inv);
        }
#pragma unroll
        for (int d = 0; d < 8; d++) {
            const int row = d * 16 + l15;
            const bf16x8 vf = *(const bf16x8 *)(vtile + row * 64 + ((lq ^ qw_vswz(row)) << 4));
            o[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pf, o[d], 0, 0, 0);
        }
        if (t + 1 < NT) {
            put_v(t + 1);
            __syncthreads();
        }
    }
    /* accumulator element e of block d: query l15, dim 16 d + 4 lq + e */
    if (qi < seq) {
        bf16 *op = out + (size_t)qi * heads * 128 + h * 128 + 4 * lq;
#pragma unroll
        for (int d = 0; d < 8; d++) {
            bf16x4 ov;
#pragma unroll
            for (int e = 0; e < 4; e++) ov[e] = (bf16)o[d][e];
            *(bf16x4 *)(op + d * 16) = ov;
        }
    }
}

/* Steps whose 32 keys all lie after the block's last query, or after the last key that the mask admits, hold no
 * admissible key and are left out - unless the first key is masked: only then can a row have no admissible key at all, and such
 * a row is uniform over every column (see above), so every step is computed. Otherwise a left-out key's probability is
 * exp(-1e9 - maximum), which is 0, and the result is the same bit for bit. The step count is
 * rounded up to one of five compiled bodies. A prompt of 67 tokens padded to 512 with 32 heads: 18.9 us with the causal bound alone, 11.2 with
 * both (the longest blocks had 16 steps, now 4). Workgroup = heads / kv_heads waves. */
template <int G>
__global__ __launch_bounds__(64 * G) void qwen3_attention_kernel(bf16 *__restrict__ out, const bf16 *__restrict__ qkv, const bf16 *__restrict__ vt,
                                                              int ldv, const int *__restrict__ mask, int seq, int heads, int kv_heads) {
    __shared__ __attribute__((aligned(16))) char smem[32768]; /* K tiles: 2 x 8 KB, V^T tiles: 2 x 8 KB */
    const int lane = threadIdx.x & 63, all = (seq + 31) >> 5;
    /* padding mask, all of it at once (one round trip to memory), then as bits: word w covers keys [64 w, 64 w + 64), one ballot per word */
    int mv[QW_MAXT / 2];
#pragma unroll
    for (int w = 0; w < QW_MAXT / 2; w++) mv[w] = mask ? mask[min(64 * w + lane, seq - 1)] : 1;
    unsigned long long keep[QW_MAXT / 2];
    int last = 0; /* the last admissible key */
#pragma unroll
    for (int w = 0; w < QW_MAXT / 2; w++) {
        keep[w] = __ballot(64 * w + lane < seq && mv[w] != 0);
        if (keep[w]) last = 64 * w + 63 - __builtin_clzll(keep[w]);
    }
    const int need = keep[0] & 1 ? min(min(all, (last >> 5) + 1), ((blockIdx.x * 16 + 15) >> 5) + 1) : all;
    if (need <= 2) qwen3_attend<2, G>(out, qkv, vt, ldv, keep, seq, heads, kv_heads, smem);
    else if (need <= 4) qwen3_attend<4, G>(out, qkv, vt, ldv, keep, seq, heads, kv_heads, smem);
    else if (need <= 8) qwen3_attend<8, G>(out, qkv, vt, ldv, keep, seq, heads, kv_heads, smem);
    else if (need <= 12) qwen3_attend<12, G>(out, qkv, vt, ldv, keep, seq, heads, kv_heads, smem);
    else qwen3_attend<16, G>(out, qkv, vt, ldv, keep, seq, heads, kv_heads, smem);
}

/* dst[s, col0 + i] = src[s, i]: one layer's hidden state into its third of the output rows */
__global__ __launch_bounds__(256) void qwen3_collect_kernel(float *__restrict__ dst, int ldd, int col0, const float *__restrict__ src, int hidden) {
    for (int i = threadIdx.x; i < hidden; i += 256) dst[(size_t)blockIdx.x * ldd + col0 + i] = src[(size_t)blockIdx.x * hidden + i];
}

/* ------------------------------------------------------------------ host entry points */

extern "C" int flux_hip_qwen3_embed(float *x, const void *embed_bf16, const int *ids_dev, int seq, int hidden, int vocab) {
    if (seq <= 0 || hidden <= 0) return flux_hip_fail("flux_hip_qwen3_embed: bad shape");
    hipLaunchKernelGGL(qwen3_embed_kernel, dim3(seq), dim3(256), 0, flux_hip_stream_handle(), x, (const bf16 *)embed_bf16, ids_dev, hidden, vocab);
    LAUNCH_OK("qwen3_embed_kernel");
    return 1;
}

extern "C" int flux_hip_rms_norm(void *out_bf16, const float *x, const float *w, int rows, int hidden, float eps) {
    if (rows <= 0 || hidden <= 0 || (hidden & 3)) return flux_hip_fail("flux_hip_rms_norm: bad shape %d x %d", rows, hidden);
    hipLaunchKernelGGL(qwen3_rms_norm_kernel, dim3(rows), dim3(256), 0, flux_hip_stream_handle(), (bf16 *)out_bf16, x, w, hidden, eps);
    LAUNCH_OK("qwen3_rms_norm_kernel");
    return 1;
}

/* ws, slices: what flux_hip_linear_slices left; slices = 0: qkv holds the projection */
extern "C" int flux_hip_qwen3_qk_rope_slices(void *qkv_bf16, void *vt_bf16, int ldv, const float *q_w, const float *k_w, const float *rope_cos,
                                             const float *rope_sin, int seq, int heads, int kv_heads, float eps, const float *ws, int slices) {
    if (seq <= 0 || heads <= 0 || kv_heads <= 0 || ldv < seq) return flux_hip_fail("flux_hip_qwen3_qk_rope: bad shape");
    const bool vec = !((((uintptr_t)qkv_bf16 | (uintptr_t)vt_bf16 | (uintptr_t)q_w | (uintptr_t)k_w | (uintptr_t)rope_cos | (uintptr_t)rope_sin) & 15) | (ldv & 7));
    if (slices > 0 && (!vec || !ws || ((uintptr_t)ws & 15))) return flux_hip_fail("flux_hip_qwen3_qk_rope_slices: unaligned operand");
    const dim3 grid((seq * (heads + kv_heads) + 15) / 16 + (seq + 63) / 64 * kv_heads);
    auto kern = slices > 0 ? qwen3_qk_rope_kernel<true, true> : vec ? qwen3_qk_rope_kernel<true, false> : qwen3_qk_rope_kernel<false, false>;
    hipLaunchKernelGGL(kern, grid,
                       dim3(256), 0, flux_hip_stream_handle(), (bf16 *)qkv_bf16, (bf16 *)vt_bf16, ldv, q_w, k_w, rope_cos, rope_sin, seq, heads, kv_heads,
                       eps, ws, slices);
    LAUNCH_OK("qwen3_qk_rope_kernel");
    return 1;
}

extern "C" int flux_hip_qwen3_qk_rope(void *qkv_bf16, void *vt_bf16, int ldv, const float *q_w, const float *k_w, const float *rope_cos,
                                      const float *rope_sin, int seq, int heads, int kv_heads, float eps) {
    return flux_hip_qwen3_qk_rope_slices(qkv_bf16, vt_bf16, ldv, q_w, k_w, rope_cos, rope_sin, seq, heads, kv_heads, eps, NULL, 0);
}

extern "C" int flux_hip_causal_attention(void *out_bf16, const void *qkv_bf16, const void *vt_bf16, int ldv, const int *mask_dev, int seq,
                                         int heads, int kv_heads) {
    if (seq <= 0 || seq > 32 * QW_MAXT) return flux_hip_fail("flux_hip_causal_attention: seq=%d (1..%d)", seq, 32 * QW_MAXT);
    if (heads <= 0 || kv_heads <= 0 || heads % kv_heads) return flux_hip_fail("flux_hip_causal_attention: heads=%d kv_heads=%d", heads, kv_heads);
    const int group = heads / kv_heads; /* waves per workgroup */
    if (group != 1 && group != 2 && group != 4 && group != 8)
        return flux_hip_fail("flux_hip_causal_attention: %d query heads per kv head (1, 2, 4 or 8)", group);
    if (ldv < ((seq + 31) & ~31) || (ldv & 7)) return flux_hip_fail("flux_hip_causal_attention: ldv=%d too small or not a multiple of 8", ldv);
    const dim3 grid((seq + 15) / 16, kv_heads);
#define QW_LAUNCH(G)                                                                                                                   \
    hipLaunchKernelGGL(qwen3_attention_kernel<G>, grid, dim3(64 * G), 0, flux_hip_stream_handle(), (bf16 *)out_bf16, (const bf16 *)qkv_bf16, \
                       (const bf16 *)vt_bf16, ldv, mask_dev, seq, heads, kv_heads)
    if (group == 1) QW_LAUNCH(1);
    else if (group == 2) QW_LAUNCH(2);
    else if (group == 4) QW_LAUNCH(4);
    else QW_LAUNCH(8);
#undef QW_LAUNCH
    LAUNCH_OK("qwen3_attention_kernel");
    return 1;
}

extern "C" int flux_hip_qwen3_collect(float *dst, int ldd, int col0, const float *src, int seq, int hidden) {
    hipLaunchKernelGGL(qwen3_collect_kernel, dim3(seq), dim3(256), 0, flux_hip_stream_handle(), dst, ldd, col0, src, hidden);
    LAUNCH_OK("qwen3_collect_kernel");
    return 1;
}
