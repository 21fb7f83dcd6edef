/*
 * conv.hip - 3x3 convolutions of the VAE's large images, bf16 operands, for gfx950.
 *
 * The convolution is the GEMM of gemm.hip's convolution epilogues (rows = positions, K = [cin / 64 chunks][9 taps][64
 * channels], the same order of additions, hence the same bits as its ring tiles), with two things done otherwise because of
 * what bounds it there:
 *
 *   - There every K step fetches its 256 positions x 64 channels again, nine times what a chunk holds, and the path from the
 *     L2s into the LDS (58 bytes per cycle and compute unit) is busy three quarters of the time. Here a tile is 16 x 16
 *     positions, whose 18 x 18 neighbourhood of one 64-channel chunk lies in LDS while the nine taps go over it: 48 KB per
 *     nine steps instead of 288.
 *   - There the finished tile's epilogue - 128 KB of residual in and 128 KB out for fp32 - runs between two K loops with the
 *     matrix pipes idle. 256 x 128 accumulators are half of the AGPRs: here the other half holds the finished tile, which is
 *     stored unit by unit (one image row x 32 channels a wave) behind the MFMAs of the next tile's first two chunks.
 *
 * Measured in turn with the tile that gemm.hip chose before, us: 1024 x 1024 x 128 -> 128 to bf16 323 -> 231, with residual to fp32
 * 442 -> 336; 512 x 512 x 256 -> 256 229 -> 204 and 318 -> 253; 256 x 256 x 512 -> 512 209 -> 196 and 251 -> 225. What
 * bounds it now: with many channels the power limit (196 us are 1575 TFLOP/s; on operands of zeros the kernel reaches 1923),
 * with 128 channels HBM (to fp32 with residual 1.35 GB, 4.0 TB/s; without its stores the bf16 form takes 22 % less).
 *
 * LDS (160 KB): two patches of 384 rows x 128 bytes (18 rows of 20 positions, 18 of them used), the chunk at work and the next
 * one, and a ring of four 16 KB slots for the weights of one tap and chunk. Requests per K step and wave: four weight loads for
 * step + 3, in the first six steps of a chunk two patch loads for the next chunk, the residual of the unit after next. A
 * barrier per step waits with a count for the weights of the next step: vector memory operations of a wave complete in order, so
 * the count is the number of operations issued after those (Ops::pending). Operations that a wave may issue beyond that number
 * (the zero border) only make the wait stricter. None of those counted is skipped: stores and loads of positions outside the image go
 * to an offset beyond the buffer resource, where stores are dropped and loads give zero. (The same with 32-channel patches, which leave room
 * for weights twelve half-steps ahead and so for slower stores, was slower by 5 to 10 % where there is a residual: twice the
 * requests for the same lines.)
 *
 * Fragment addresses: patch row r = 20 (row) + column; a row's 16-byte chunks are swizzled by lds_swz(r mod 16) as in gemm.hip.
 * A step down by one image row moves r by 20, which changes the swizzle by 2 (r / 2 mod 8), two rows by 4, i.e. one XOR: twelve
 * addresses per lane (3 dx x row parity x half) and immediates cover all taps and rows.
 *
 * up = 1: the operand is the nearest-neighbour 2x enlargement of the image that is given. Bordered position (y, x) of the enlargement holds position
 * ((y + 1) / 2, (x + 1) / 2) of the bordered source, border included, and a tile starts at multiples of 16, so that only the patch's source
 * offsets differ.
 */
#include "common.h"
#include "../../include/flux_hip.h"

namespace {

struct Args {
    const bf16 *in, *w;
    const float *bias, *res;
    void *out;
    float *stats;
    int H, W, cin, cout;
    int tiles_x, ntiles, total, vgrid; /* total = tiles of positions x tiles of channels */
    int up; /* fp32 results without residual alone */
    unsigned magic_x, magic_n;         /* ceil(2^32 / tiles_x), ceil(2^32 / ntiles): exact for numbers below 2^16 */
};

constexpr int TM = 8, TN = 4, NM = TM * TN, NF = TM + TN, RD = 2; /* blocks of a wave, MFMAs and fragments of a half-step, MFMAs per fragment read */
constexpr int PITCH = 20, PATCH = 384 * 128, SLOT = 128 * 128, W0 = 2 * PATCH, LDS_BYTES = 2 * PATCH + 4 * SLOT;
/* Beyond every buffer: the host admits images of less than 3.7e9 bytes, and seven image rows of results of less than 2^28, so that a column
 * beyond the image stays there with a row's offset added (and 2 * OUTSIDE mod 2^32 = 3.76e9, a column and a row beyond it, as well). */
constexpr unsigned OUTSIDE = 0xF0000000u;
static_assert(LDS_BYTES <= 160 * 1024, "LDS");

#define LDS_PTR(p) ((__attribute__((address_space(3))) void *)(p))
#define LDS_FRAG(addr) (*(const __attribute__((address_space(3))) bf16x8 *)(uintptr_t)(addr))
/* All 256 accumulator registers are used by name, block n of the tile at work at a[4 n], of the finished one at a[128 + 4 n], and
 * the compiler uses none (the tests look at its output for that). Left to allocate both sets it moved whole sets at the joins of the
 * paths, 128 moves and some spills per chunk. */
#define BLOCK(n) "i"(4 * (n)), "i"(4 * (n) + 3)
#define MFMA(n, a, b) asm volatile("v_mfma_f32_16x16x32_bf16 a[%2:%3], %0, %1, a[%2:%3]" ::"v"(a), "v"(b), BLOCK(n))
#define MFMA_NEW(n, a, b) asm volatile("v_mfma_f32_16x16x32_bf16 a[%2:%3], %0, %1, 0" ::"v"(a), "v"(b), BLOCK(n))
/* the last half-step of a tile: the sums go to the finished tile's registers */
#define MFMA_LAST(n, a, b) asm volatile("v_mfma_f32_16x16x32_bf16 a[%4:%5], %0, %1, a[%2:%3]" ::"v"(a), "v"(b), BLOCK(n), BLOCK(32 + (n)))
__device__ __forceinline__ float finished(int n, int e) {
    float a;
    asm volatile("v_accvgpr_read_b32 %0, a[%1]" : "=v"(a) : "i"(128 + 4 * n + e));
    return a;
}

template <int V> struct IntC { static constexpr int value = V; };
template <bool V> struct BoolC { static constexpr bool value = V; };

__device__ __forceinline__ int lds_swz(int r) { return ((r >> 1) & 7) ^ ((r & 1) << 2); }
__device__ __forceinline__ int bf16_pair_feature(int blk, int r) { return 32 * (blk >> 1) + 8 * (r >> 2) + 4 * (blk & 1) + (r & 3); }

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer(const void *base, long long bytes) {
    return __builtin_amdgcn_make_buffer_rsrc((void *)base, 0, (int)(unsigned)bytes, 0x00020000);
}
__device__ __forceinline__ f32x4 load4(__amdgpu_buffer_rsrc_t r, unsigned off, int soff) {
    const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, off, soff, 0);
    return __builtin_bit_cast(f32x4, v);
}

/* v summed over the 16 lanes of equal lane / 16 */
__device__ __forceinline__ float row_sum(float v) {
    const auto ror = [](float x, auto n) { return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x120 + decltype(n)::value, 0xF, 0xF, true)); };
    v += ror(v, IntC<8>{});
    v += ror(v, IntC<4>{});
    v += ror(v, IntC<2>{});
    v += ror(v, IntC<1>{});
    return v;
}

struct Tile { int y0, x0, n0, tm; };

__device__ __forceinline__ bool decode(const Args &g, int vb, Tile &t) {
    const int i = (vb & 7) * (g.vgrid >> 3) + (vb >> 3); /* each XCD gets a contiguous run of tiles */
    if (i >= g.total) return false;
    t.tm = g.ntiles == 1 ? i : (int)__umulhi((unsigned)i, g.magic_n);
    const int ty = g.tiles_x == 1 ? t.tm : (int)__umulhi((unsigned)t.tm, g.magic_x);
    t.n0 = (i - t.tm * g.ntiles) * 128;
    t.y0 = ty * 16;
    t.x0 = (t.tm - ty * g.tiles_x) * 16;
    return true;
}

/* One tile's results: F32 or bf16, with a residual or without. A wave owns 8 image rows x 16 columns (wm) and 64 channels (wn);
 * unit u is image row u / 2 and 32 of the channels, two MFMA blocks. The two units that share 128-byte lines of bf16 follow each other: with
 * all rows of one half first, 1024 x 1024 x 128 wrote 377 MB for 275. */
template <bool F32, bool RES>
struct Epilogue {
    static constexpr int E = F32 ? 4 : 2; /* bytes per output element */
    __amdgpu_buffer_rsrc_t out, res, stats;
    unsigned vo, vr, vs; /* this lane's byte offsets: output, residual, statistics */
    int rows;            /* image rows of the wave's eight that exist */
    bool col_ok;
    unsigned pitch; /* elements per image row */
    f32x4 bias[2][2], x[3][2];
    float st[2][2][2]; /* of the wave's channels 32 p .. 32 p + 31 */

    __device__ __forceinline__ void begin(const Args &g, const Tile &t, bool any, int wm, int wn, int l15, int lq) {
        const long long wp = g.W + 2, origin = ((t.y0 + 8 * wm + 1) * wp + t.x0 + 1) * g.cout + t.n0 + wn * 64, all = (g.H + 2) * wp * g.cout;
        rows = __builtin_amdgcn_readfirstlane(any ? max(0, min(8, g.H - t.y0 - 8 * wm)) : 0);
        const long long left = rows > 0 ? all - origin : 0; /* a wave whose rows all lie below the image starts beyond its end */
        out = buffer((char *)g.out + origin * E, left * E);
        if (RES) res = buffer(g.res + origin, left * 4);
        const int quads = g.cout >> 2;
        stats = buffer(g.stats, g.stats && any ? ((long long)(2 * t.tm + wm) * quads + quads) * 8 : 0);
        col_ok = t.x0 + l15 < g.W;
        const unsigned lane = (unsigned)l15 * g.cout + (F32 ? 4 : 8) * lq;
        vo = col_ok ? lane * E : OUTSIDE;
        vr = col_ok ? lane * 4 : OUTSIDE;
        vs = l15 == 0 ? (unsigned)((2 * t.tm + wm) * quads + ((t.n0 + wn * 64) >> 2) + (F32 ? lq : 2 * lq)) * 8 : OUTSIDE;
        pitch = (unsigned)(wp * g.cout);
    }
    /* offset of the wave's image row j, formed where it is used (kept for all rows, loads and stores they are sixteen registers) */
    __device__ __forceinline__ unsigned at(unsigned lane_off, int j, int bytes) const {
        int n = rows;
        asm volatile("" : "+s"(n), "+v"(lane_off));
        return lane_off + (j < n ? j * pitch * bytes : OUTSIDE);
    }
    __device__ __forceinline__ void load_bias(const Args &g, int c) { /* c: the wave's first channel */
        const __amdgpu_buffer_rsrc_t b = buffer(g.bias, (long long)g.cout * 4);
#pragma unroll
        for (int p = 0; p < 2; p++)
#pragma unroll
            for (int k = 0; k < 2; k++) bias[p][k] = load4(b, (unsigned)(c + p * 32 + k * (F32 ? 16 : 4)) * 4, 0);
    }
    __device__ __forceinline__ void fetch(int u) { /* two loads */
        const unsigned o = at(vr, u >> 1, 4);
#pragma unroll
        for (int k = 0; k < 2; k++) x[u % 3][k] = load4(res, o + (u & 1) * 128 + k * (F32 ? 64 : 16), 0);
    }
    /* A unit's eight values per lane, in pieces of one or two instructions that hide behind an MFMA: out of the accumulators, the
     * value, its share of the sums, and per block the sums of the rows that exist */
    f32x4 v[2];
    float s, q;
    __device__ __forceinline__ void take(int u, int n) { v[n >> 2][n & 3] = finished((2 * (u & 1) + (n >> 2)) * TM + (u >> 1), n & 3); }
    __device__ __forceinline__ void value(int u, int n) {
        const int k = n >> 2, e = n & 3;
        float a = v[k][e];
        a = RES ? x[u % 3][k][e] + a + bias[u & 1][k][e] : a + bias[u & 1][k][e];
        asm volatile("" : "+v"(a));
        v[k][e] = a;
    }
    __device__ __forceinline__ void add(int n) {
        const int k = n >> 2, e = n & 3;
        s = e ? s + v[k][e] : v[k][e];
        q = e ? q + v[k][e] * v[k][e] : v[k][e] * v[k][e];
        asm volatile("" : "+v"(s), "+v"(q));
    }
    /* block k of unit u behind MFMA b of a half-step */
    __device__ __forceinline__ void piece(int u, int k, int b) {
        if (b % 6 == 1 && b < 24) take(u, 4 * k + b / 6);
        if (b % 6 == 3 && b < 24) value(u, 4 * k + b / 6);
        if (b % 6 == 5 && b < 24) add(4 * k + b / 6);
        if (b == 25) keep(u, k);
        if (k == 1 && b == 27) store(u);
        if (k == 1 && u >= 14 && b == 29) sums(u & 1);
    }
    __device__ __forceinline__ void keep(int u, int k) {
        const bool ok = col_ok && (u >> 1) < rows;
        float(&t)[2] = st[u & 1][k];
        t[0] = (u > 1 ? t[0] : 0.0f) + (ok ? s : 0.0f);
        t[1] = (u > 1 ? t[1] : 0.0f) + (ok ? q : 0.0f);
        asm volatile("" : "+v"(t[0]), "+v"(t[1]));
    }
    __device__ __forceinline__ void store(int u) { /* two stores of fp32, one of bf16 */
        const unsigned o = at(vo, u >> 1, E) + (u & 1) * 32 * E;
        if (F32) {
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v[0]), out, o, 0, 0);
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v[1]), out, o + 64, 0, 0);
        } else {
            bf16x8 b;
#pragma unroll
            for (int e = 0; e < 4; e++) { b[e] = (bf16)v[0][e]; b[4 + e] = (bf16)v[1][e]; }
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, b), out, o, 0, 0);
        }
    }
    __device__ __forceinline__ void sums(int p) { /* behind the last row: two stores of fp32's sums, one of bf16's, whose two blocks' are neighbours (the
                                                   * compiler made one of two there, and Ops counted two) */
        const f32x4 t = {row_sum(st[p][0][0]), row_sum(st[p][0][1]), row_sum(st[p][1][0]), row_sum(st[p][1][1])};
        if (F32) {
            typedef __attribute__((ext_vector_type(2))) unsigned u32x2;
            __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, f32x2{t[0], t[1]}), stats, vs + p * 64, 0, 0);
            __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, f32x2{t[2], t[3]}), stats, vs + p * 64 + 32, 0, 0);
        } else {
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, t), stats, vs + p * 64, 0, 0);
        }
    }
};

/* the zeros around the image that touch this tile: its 18 x 18 neighbourhood's rim, as far as that is border */
template <bool F32>
__device__ __forceinline__ void zero_border(const Args &g, const Tile &t, int tid) {
    if (t.y0 > 0 && t.x0 > 0 && t.y0 + 16 < g.H && t.x0 + 16 < g.W) return;
    constexpr int E = F32 ? 4 : 2, LANES = 8 * E, PER = 256 / LANES; /* 16 bytes per lane, positions per pass */
    for (int k = tid / LANES; k < 68; k += PER) {
        const int py = k < 18 ? 0 : k < 36 ? 17 : k < 52 ? k - 35 : k - 51, px = k < 18 ? k : k < 36 ? k - 18 : k < 52 ? 0 : 17;
        const int y = min(t.y0 + py, g.H + 1), x = min(t.x0 + px, g.W + 1);
        if (y == 0 || y == g.H + 1 || x == 0 || x == g.W + 1)
            *(u32x4 *)((char *)g.out + (((long long)y * (g.W + 2) + x) * g.cout + t.n0) * E + tid % LANES * 16) = u32x4{0, 0, 0, 0};
    }
}

/* Steps of a tile: 0 .. 17 are its first two chunks, with the finished tile's epilogue behind their MFMAs (unit u: its first block in the
 * second half of step u + 1, its second one and the stores in the first half of step u + 2); 18 + tap is any later chunk. Vector memory
 * operations of a step (as they are in the compiled code, which the tests count: a number that is too large lets a barrier through while
 * weights are on their way), in this order: 4 weight loads and epilogue() in the first half, patch() in the second. */
template <bool F32, bool RES>
struct Ops {
    static constexpr int patch(int s) { return s % 9 < 6 ? 2 : 0; }
    static constexpr int epilogue(int s) {
        if (s >= 18) return 0;
        const int loads = s == 0 ? 4 + (RES ? 4 : 0) : RES && s <= 14 ? 2 : 0;                       /* bias, residual */
        const int stores = s < 2 ? 0 : (F32 ? 2 : 1) * (s >= 16 ? 2 : 1);                            /* results, sums */
        return loads + stores;
    }
    /* issued after the weights that the barrier of step s waits for, which were requested at the head of step s - 2. Of the
     * steps in front of step 0 or 18 the epilogue's operations, which may be there or not, are not counted */
    static constexpr int pending(int s) {
        const int first = s < 18 ? 0 : 18;
        int n = 4 + 4 + epilogue(s);
        for (int k = 1; k <= 2; k++) n += s - k >= first ? patch(s - k) + epilogue(s - k) : 0; /* (taps 7 and 8 request no patch) */
        return n;
    }
};

template <bool F32, bool RES>
__global__ __launch_bounds__(256) void conv3_kernel(Args g) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    using O = Ops<F32, RES>;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6) & 3, wm = wave >> 1, wn = wave & 1;
    const int l15 = lane & 15, lq = lane >> 4;
    const int up = F32 && !RES ? g.up : 0, wp = (g.W >> up) + 2, nch = g.cin >> 6, ldw = 9 * g.cin; /* wp: the source's */

    Tile t, nx;
    int vb = blockIdx.x;
    if (!decode(g, vb, t)) return;

    /* patch loads: LDS row r = 8 (4 q + wave) + lane / 8 holds position (r / 20, r % 20) of the neighbourhood (the two columns and the
     * rows beyond it repeat others) */
    unsigned prel[12], wrel[4];
#pragma unroll
    for (int q = 0; q < 12; q++) {
        const int r = 8 * (4 * q + wave) + (lane >> 3), py = min(r / PITCH, 17), px = min(r % PITCH, 17);
        prel[q] = (unsigned)((((py + up) >> up) * wp + ((px + up) >> up)) * g.cin + (((lane & 7) ^ lds_swz(r)) << 3)) * 2u;
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int v = 32 * i + 8 * wave + (lane >> 3), n = F32 ? v : (v & 64) + bf16_pair_feature((v & 63) >> 4, v & 15);
        wrel[i] = (unsigned)(n * ldw + (((lane & 7) ^ lds_swz(v)) << 3)) * 2u;
    }
    const long long in_elems = (long long)((g.H >> up) + 2) * wp * g.cin;
    const __amdgpu_buffer_rsrc_t wbuf = buffer(g.w, (long long)g.cout * ldw * 2);
    auto patch_buffer = [&](const Tile &tt, int chunk) {
        const long long o = ((long long)(tt.y0 >> up) * wp + (tt.x0 >> up)) * g.cin + chunk * 64;
        return buffer(g.in + o, (in_elems - o) * 2);
    };
    auto load_patch = [&](__amdgpu_buffer_rsrc_t b, int to, int q) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(b, LDS_PTR(smem + to + (4 * q + wave) * 1024), 16, prel[q], 0, 0, 0);
    };
    auto load_w = [&](int woff, int slot, int i) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(wbuf, LDS_PTR(smem + W0 + slot * SLOT + (4 * i + wave) * 1024), 16, wrel[i], woff, 0, 0);
    };

    /* this lane's fragment addresses in the patch at work, see the file comment, and in a weight slot */
    const unsigned lds0 = (unsigned)(uintptr_t)LDS_PTR(smem);
    unsigned pa[3][2][2], wa[2];
#pragma unroll
    for (int dx = 0; dx < 3; dx++)
#pragma unroll
        for (int mp = 0; mp < 2; mp++) {
            const int c = l15 + dx, sw = ((2 * mp + (c >> 1)) & 7) ^ ((c & 1) << 2);
#pragma unroll
            for (int h = 0; h < 2; h++) pa[dx][mp][h] = lds0 + (unsigned)((8 * wm * PITCH + c) * 128 + (((lq ^ sw) ^ (4 * h)) << 4));
        }
#pragma unroll
    for (int h = 0; h < 2; h++) wa[h] = lds0 + (unsigned)(W0 + (wn * 64 + l15) * 128 + (((lq + 4 * h) ^ lds_swz(l15)) << 4));
    /* fragment q of half kk of a tap: weights first, then the wave's eight image rows */
    auto frag = [&](int tap, int kk, unsigned wslot, int q) -> bf16x8 {
        const int dy = tap / 3, dx = tap % 3, m = q - TN + dy;
        return q < TN ? LDS_FRAG(wa[kk] + wslot + q * 2048) : LDS_FRAG(pa[dx][m & 1][(kk ^ (m >> 1)) & 1] + m * PITCH * 128);
    };

    asm volatile("" ::: "a255"); /* all AGPRs belong to the kernel */
    bf16x8 f0[NF], f1[NF];
    Epilogue<F32, RES> ep;
    bool any = false; /* there is a finished tile */
    Tile done = t;

    /* the first tile's first patch and weights */
    int slot = 0, to = PATCH;
    {
        const __amdgpu_buffer_rsrc_t b = patch_buffer(t, 0);
#pragma unroll
        for (int q = 0; q < 12; q++) load_patch(b, 0, q);
#pragma unroll
        for (int k = 0; k < 3; k++)
#pragma unroll
            for (int i = 0; i < 4; i++) load_w(t.n0 * ldw * 2 + k * 128, k, i);
    }
    int woff = t.n0 * ldw * 2 + 3 * 128; /* the weights of the step three ahead */
    asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)\n\ts_barrier" ::: "memory"); /* the patch and the first tap's weights have landed */
#pragma unroll
    for (int q = 0; q < NF; q++) f0[q] = frag(0, 0, 0, q);

    auto serp = [](int b) { return ((b / TN) & 1) ? TN - 1 - b % TN : b % TN; };

    for (;;) {
        vb += gridDim.x;
        const bool again = vb < g.vgrid && decode(g, vb, nx);
        if (!again) nx = t; /* requested once more, into LDS that nobody reads again */
        ep.begin(g, done, any, wm, wn, l15, lq);
        if (any) zero_border<F32>(g, done, tid);
        __amdgpu_buffer_rsrc_t pb;
        bool last = false;

        auto first_half = [&](auto step_c) {
            constexpr int S = decltype(step_c)::value, TAP = S % 9;
            constexpr bool EPI = S < 18;
            const int free_slot = (slot + 3) & 3;
            const unsigned ws = slot * SLOT;
#pragma unroll
            for (int b = 0; b < NM; b++) {
                if (S == 0) MFMA_NEW(serp(b) * TM + b / TN, f0[serp(b)], f0[TN + b / TN]);
                else MFMA(serp(b) * TM + b / TN, f0[serp(b)], f0[TN + b / TN]);
                if (b % RD == 0 && b / RD < NF) f1[b / RD] = frag(TAP, 1, ws, b / RD);
                if (b % 4 == 1 && b / 4 < 4) load_w(woff, free_slot, b / 4);
                if (EPI && S == 0 && b == 17) ep.load_bias(g, done.n0 + wn * 64 + (F32 ? 4 : 8) * lq);
                if (EPI && RES && S == 0 && b == 21) ep.fetch(0);
                if (EPI && RES && S <= 14 && b == 30) ep.fetch(S + 1);
                if (EPI && S >= 2) ep.piece(S - 2, 1, b);
            }
            woff += 128;
            if (TAP == 5 && last) woff = nx.n0 * ldw * 2; /* from the next step on: the next tile's */
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(O::pending(S)) : "memory");
            if (TAP == 8) { /* the next step reads the other patch */
                const unsigned d = to - (PATCH - to);
#pragma unroll
                for (int k = 0; k < 12; k++) pa[k / 4][k / 2 % 2][k % 2] += d;
            }
        };
        auto second_half = [&](auto step_c, auto last_c) {
            constexpr int S = decltype(step_c)::value, TAP = S % 9, NEXT = (TAP + 1) % 9;
            const unsigned ws = ((slot + 1) & 3) * SLOT;
#pragma unroll
            for (int b = 0; b < NM; b++) {
                if (decltype(last_c)::value) MFMA_LAST(serp(b) * TM + b / TN, f1[serp(b)], f1[TN + b / TN]);
                else MFMA(serp(b) * TM + b / TN, f1[serp(b)], f1[TN + b / TN]);
                if (b % RD == 0 && b / RD < NF) f0[b / RD] = frag(NEXT, 0, ws, b / RD);
                if (O::patch(S) && (b == 5 || b == 19)) load_patch(pb, to, 2 * TAP + (b == 19));
                if (S >= 1 && S <= 16) ep.piece(S - 1, 0, b);
            }
            if (TAP == 8) to = PATCH - to;
            slot = (slot + 1) & 3;
        };
        auto step = [&](auto step_c) {
            first_half(step_c);
            second_half(step_c, BoolC<false>{});
        };
        auto chunk_of = [&](int c) {
            last = c == nch - 1;
            pb = last ? patch_buffer(nx, 0) : patch_buffer(t, c + 1);
        };
#define STEPS8(s0) step(IntC<s0>{}); step(IntC<s0 + 1>{}); step(IntC<s0 + 2>{}); step(IntC<s0 + 3>{}); step(IntC<s0 + 4>{}); \
                   step(IntC<s0 + 5>{}); step(IntC<s0 + 6>{}); step(IntC<s0 + 7>{}); first_half(IntC<s0 + 8>{})
        chunk_of(0);
        STEPS8(0);
        second_half(IntC<8>{}, BoolC<false>{});
        chunk_of(1);
        STEPS8(9);
        if (last) {
            second_half(IntC<17>{}, BoolC<true>{});
        } else {
            second_half(IntC<17>{}, BoolC<false>{});
            for (int c = 2;; c++) {
                chunk_of(c);
                STEPS8(18);
                if (last) break;
                second_half(IntC<26>{}, BoolC<false>{});
            }
            second_half(IntC<26>{}, BoolC<true>{});
        }
        done = t;
        any = true;
        if (!again) break;
        t = nx;
    }
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory"); /* the last results retire before they are read */
    ep.begin(g, done, true, wm, wn, l15, lq);
    zero_border<F32>(g, done, tid);
    ep.load_bias(g, done.n0 + wn * 64 + (F32 ? 4 : 8) * lq);
    if (RES) { ep.fetch(0); ep.fetch(1); }
#pragma unroll
    for (int u = 0; u < 16; u++) {
        if (RES && u + 2 < 16) ep.fetch(u + 2);
#pragma unroll
        for (int b = 0; b < 64; b++) ep.piece(u, b >> 5, b & 31);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); /* the requests in place of a next tile's land in this workgroup's LDS */
}

template <bool F32, bool RES>
int launch(const Args &g, int grid) {
    static bool attr_done = false;
    auto kern = conv3_kernel<F32, RES>;
    if (!attr_done) {
        HIP_OK(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, LDS_BYTES));
        attr_done = true;
    }
    hipLaunchKernelGGL(kern, dim3(grid), dim3(256), LDS_BYTES, flux_hip_stream_handle(), g);
    HIP_OK(hipGetLastError());
    return 1;
}

/* ---- the first and the last convolution, which have three channels on one side ---- */

/* 128 -> 3 channels and the picture itself. As a GEMM with its outputs padded to 64 columns and fp32 rows for a second kernel to read this was
 * 288 + 56 us at 1024 x 1024, and is 75; HBM: 268 MB in. A workgroup makes 16 x 32 pixels: every position of
 * their 18 x 34 neighbourhood is read once and multiplied with the weights of all nine taps, 27 outputs (two MFMA blocks, K = 128), which go
 * to LDS; a pixel is the sum of nine of its neighbours' numbers. */
#define OUT_PH 16
#define OUT_PW 32
#define OUT_LD 28 /* floats per position: 9 taps x 3 channels, and one to keep 16-byte alignment */
__global__ __launch_bounds__(256) void conv_out_kernel(uint8_t *__restrict__ rgb, float *__restrict__ rgb_f32, const bf16 *__restrict__ in, const bf16 *__restrict__ w,
                                                       const float *__restrict__ bias, int H, int W) {
    __shared__ __attribute__((aligned(16))) float part[(OUT_PH + 2) * (OUT_PW + 2) * OUT_LD];
    constexpr int POS = (OUT_PH + 2) * (OUT_PW + 2), BLOCKS = (POS + 15) / 16, PER = (BLOCKS + 3) / 4;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l15 = lane & 15, lq = lane >> 4;
    const int x0 = blockIdx.x * OUT_PW, y0 = blockIdx.y * OUT_PH, wp = W + 2;
    bf16x8 fw[2][4]; /* row r = 3 tap + output channel */
#pragma unroll
    for (int b = 0; b < 2; b++) {
        const int r = min(16 * b + l15, 26), tap = r / 3, o = r - 3 * tap;
#pragma unroll
        for (int k = 0; k < 4; k++) fw[b][k] = *(const bf16x8 *)(w + (size_t)o * 9 * 128 + (k >> 1) * 9 * 64 + tap * 64 + (k & 1) * 32 + lq * 8);
    }
    const auto row = [&](int blk) { /* this lane's position of a block; those beyond the image repeat its last row and column */
        const int p = min(blk * 16 + l15, POS - 1), py = p / (OUT_PW + 2), px = p - py * (OUT_PW + 2);
        return in + ((size_t)min(y0 + py, H + 1) * wp + min(x0 + px, W + 1)) * 128 + lq * 8;
    };
#pragma unroll
    for (int i = 0; i < PER; i += 2) { /* two blocks' loads on their way together */
        bf16x8 f[2][4];
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const bf16 *src = row(min((i + u) * 4 + wave, BLOCKS - 1));
#pragma unroll
            for (int k = 0; k < 4; k++) f[u][k] = *(const bf16x8 *)(src + k * 32);
        }
#pragma unroll
        for (int u = 0; u < 2; u++) {
            f32x4 a[2] = {{0.0f, 0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f, 0.0f}};
#pragma unroll
            for (int k = 0; k < 4; k++)
#pragma unroll
                for (int b = 0; b < 2; b++) a[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[b][k], f[u][k], a[b], 0, 0, 0);
            const int p = ((i + u) * 4 + wave) * 16 + l15;
            if (p < POS) {
                *(f32x4 *)(part + p * OUT_LD + 4 * lq) = a[0];
                if (lq < 3) *(f32x4 *)(part + p * OUT_LD + 16 + 4 * lq) = a[1];
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < OUT_PH * OUT_PW / 256; i++) {
        const int n = i * 256 + threadIdx.x, py = n / OUT_PW, px = n % OUT_PW, y = y0 + py, x = x0 + px;
        if (y >= H || x >= W) continue;
#pragma unroll
        for (int c = 0; c < 3; c++) {
            float v = 0.0f;
#pragma unroll
            for (int tap = 0; tap < 9; tap++) v += part[((py + tap / 3) * (OUT_PW + 2) + px + tap % 3) * OUT_LD + 3 * tap + c];
            v += bias[c];
            float val = (v + 1.0f) * 0.5f * 255.0f; /* flux_vae.c:820-833 */
            val = val < 0.0f ? 0.0f : val > 255.0f ? 255.0f : val;
            if (rgb) rgb[((size_t)y * W + x) * 3 + c] = (uint8_t)val;
            if (rgb_f32) rgb_f32[((size_t)c * H + y) * W + x] = v;
        }
    }
}

/* 3 -> 128 channels (flux_vae.c:336-338): the 27 values under a position's window are one MFMA's K, gathered from the fp32 picture
 * as the operand. As rows of 64 bf16 written by one kernel and multiplied by the next it was 69 + 146 us at 720 x 1296, and is 129; HBM: 478 MB out. A wave
 * makes IN_BLOCKS blocks of 16 bordered positions (zeros on the border) and leaves one row of sums for the group norm (none if all its
 * positions lie behind the last one). */
#define IN_BLOCKS 8
__global__ __launch_bounds__(256) void conv_in_kernel(float *__restrict__ out, const float *__restrict__ img, const bf16 *__restrict__ w, const float *__restrict__ bias,
                                                      float *__restrict__ stats, int H, int W) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l15 = lane & 15, lq = lane >> 4;
    const int wp = W + 2, rows = (H + 2) * wp, first = (blockIdx.x * 4 + wave) * IN_BLOCKS * 16;
    bf16x8 fw[8]; /* w: [128][64], element 3 tap + channel, zeros from 27 on */
    f32x4 bv[8];
#pragma unroll
    for (int i = 0; i < 8; i++) {
        fw[i] = *(const bf16x8 *)(w + (16 * i + l15) * 64 + lq * 8);
        bv[i] = *(const f32x4 *)(bias + 16 * i + 4 * lq);
    }
    float s[8], q[8];
#pragma unroll
    for (int i = 0; i < 8; i++) s[i] = q[i] = 0.0f;
    float g[8]; /* a block's values, requested one block ahead */
    bool inside_next;
    const auto gather = [&](int blk) {
        const int p = first + blk * 16 + l15, py = p / wp, px = p - py * wp;
        inside_next = p < rows && py >= 1 && py <= H && px >= 1 && px <= W;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const int k = lq * 8 + e, tap = k / 3, c = k - 3 * tap, y = py - 2 + tap / 3, x = px - 2 + tap % 3;
            g[e] = inside_next && k < 27 && y >= 0 && y < H && x >= 0 && x < W ? img[((size_t)c * H + y) * W + x] : 0.0f;
        }
    };
    gather(0);
    for (int blk = 0; blk < IN_BLOCKS; blk++) {
        const int p = first + blk * 16 + l15;
        const bool inside = inside_next;
        bf16x8 f;
#pragma unroll
        for (int e = 0; e < 8; e++) f[e] = (bf16)g[e];
        gather(blk + 1);
#pragma unroll
        for (int i = 0; i < 8; i++) {
            f32x4 v = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[i], f, f32x4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
#pragma unroll
            for (int e = 0; e < 4; e++) {
                v[e] = inside ? v[e] + bv[i][e] : 0.0f;
                s[i] += v[e];
                q[i] += v[e] * v[e];
            }
            if (p < rows) *(f32x4 *)(out + (size_t)p * 128 + 16 * i + 4 * lq) = v;
        }
    }
    if (first >= rows) return; /* a wave behind the last position has no sums */
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const f32x2 t = {row_sum(s[i]), row_sum(q[i])};
        if (l15 == 0) *(f32x2 *)(stats + ((size_t)(blockIdx.x * 4 + wave) * 32 + 4 * i + lq) * 2) = t;
    }
}

} // namespace

/* in: bf16 [(H + 2) * (W + 2)][128]; w: the first three rows of flux_hip_conv's weights; rgb 8-bit [H][W][3] and/or rgb_f32 [3][H][W] */
extern "C" int flux_hip_vae_conv_out(uint8_t *rgb, float *rgb_f32, const void *in, const void *w, const float *bias, int H, int W) {
    if (H <= 0 || W <= 0 || !in || !w || !bias) return flux_hip_fail("flux_hip_vae_conv_out: bad argument");
    const int slot = conv_probe_begin(FLUX_HIP_EPI_CONV_F32, 17);
    hipLaunchKernelGGL(conv_out_kernel, dim3((W + OUT_PW - 1) / OUT_PW, (H + OUT_PH - 1) / OUT_PH), dim3(256), 0, flux_hip_stream_handle(), rgb, rgb_f32, (const bf16 *)in,
                       (const bf16 *)w, bias, H, W);
    conv_probe_end(slot);
    HIP_OK(hipGetLastError());
    return 1;
}

/* img: fp32 [3][H][W]; w: bf16 [128][64]; out: fp32 [(H + 2) * (W + 2)][128], its border zeros; stats: as flux_hip_conv_stats */
extern "C" int flux_hip_vae_conv_in(float *out, const float *img, const void *w, const float *bias, int H, int W, float *stats, int *stats_rows) {
    if (H <= 0 || W <= 0 || !out || !img || !w || !bias || !stats || !stats_rows) return flux_hip_fail("flux_hip_vae_conv_in: bad argument");
    const int rows = (H + 2) * (W + 2), wg = (rows + 64 * IN_BLOCKS - 1) / (64 * IN_BLOCKS);
    const int slot = conv_probe_begin(FLUX_HIP_EPI_CONV_F32, 18);
    hipLaunchKernelGGL(conv_in_kernel, dim3(wg), dim3(256), 0, flux_hip_stream_handle(), out, img, (const bf16 *)w, bias, stats, H, W);
    conv_probe_end(slot);
    HIP_OK(hipGetLastError());
    *stats_rows = (rows + 16 * IN_BLOCKS - 1) / (16 * IN_BLOCKS); /* one per wave that has positions, within the rows / 32 + 2 that a caller provides */
    return 1;
}

/* Whether the kernel takes this convolution: two chunks of input channels at least, the image in 32-bit byte offsets below OUTSIDE, tile
 * numbers below 2^16, no more rows of statistics than one per 32 positions of the bordered image + 2, and rows short enough for OUTSIDE
 * (16 x 20001 positions x 512 channels came round to the start of the image). */
bool conv3_takes(int H, int W, int cin, int cout) {
    const long long pos = (long long)(H + 2) * (W + 2), tiles = (long long)((H + 15) / 16) * ((W + 15) / 16);
    return H > 0 && W > 0 && cin >= 128 && cin % 64 == 0 && cout % 128 == 0 && pos * max(cin * 2, cout * 4) < 3700000000LL &&
           (long long)cout * cin * 18 < 2000000000LL && tiles * (cout / 128) < 65536 && 2 * tiles <= pos / 32 + 2 &&
           7LL * (W + 2) * cout * 4 + 65536 <= 1LL << 28;
}
long conv3_tiles(int H, int W, int cout) { return (long)((H + 15) / 16) * ((W + 15) / 16) * (cout / 128); }

/* up: H x W is the 2x enlargement of the image at `in`; fp32 without residual alone */
int conv3_launch(bool f32, bool up, const void *in, const void *w, const float *bias, const float *res, void *out, int H, int W, int cin, int cout, float *stats,
                 int *stats_rows, int units) {
    Args g = {};
    g.in = (const bf16 *)in; g.w = (const bf16 *)w; g.bias = bias; g.res = res; g.out = out; g.stats = stats;
    g.H = H; g.W = W; g.cin = cin; g.cout = cout; g.up = up;
    g.tiles_x = (W + 15) / 16;
    g.ntiles = cout / 128;
    g.total = (int)conv3_tiles(H, W, cout);
    g.vgrid = (g.total + 7) & ~7;
    g.magic_x = (unsigned)(((1ull << 32) + g.tiles_x - 1) / g.tiles_x);
    g.magic_n = (unsigned)(((1ull << 32) + g.ntiles - 1) / g.ntiles);
    if (stats_rows) *stats_rows = 2 * (g.total / g.ntiles);
    const int grid = min(g.vgrid, units);
    if (up && (!f32 || res || ((H | W) & 1))) return flux_hip_fail("conv3_launch: an enlargement has even sides, fp32 results and no residual");
    if (f32) return res ? launch<true, true>(g, grid) : launch<true, false>(g, grid);
    return res ? launch<false, true>(g, grid) : launch<false, false>(g, grid);
}
