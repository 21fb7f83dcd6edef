/*
 * gemm.hip - bf16 MFMA GEMM  C[M,N] = A[M,K] * W[N,K]^T  with fused epilogues, for gfx950.
 *
 * This is the linear layer of the denoising transformer (reference: flux_linear,
 * flux_kernels.c:210-282, cblas_sgemm NoTrans x Trans). Both operands have K contiguous, so
 * an MFMA operand fragment (8 consecutive bf16 of one row) is one 16-byte LDS read.
 *
 * Tiling: a workgroup owns a BM x BN tile; K is walked in steps of 64 through two LDS stages.
 * Tiles go from global memory straight into LDS (global_load_lds_dwordx4, no register
 * staging, no ds_write): the next stage is in flight while the current one is multiplied, with
 * one barrier per step. Each 64-lane wave owns a WM x WN sub-tile made of 16x16 blocks of
 * v_mfma_f32_16x16x32_bf16. On this part the matrix pipes are power limited with real data;
 * the 16x16x32 form sustains about 15 % more than 32x32x16 at the same tile, and skipping the
 * register/ds_write hop saves both time and energy (measured: 800 -> 1000 TFLOP/s on the
 * 4608 x 18432 x 3072 projection).
 *
 * The weight fragment is the MFMA "A" operand and the activation fragment the "B" operand,
 * so that in the accumulator a lane holds one token (m) and four consecutive output features
 * (n): epilogues use 8/16-byte accesses and pair gate/up columns inside a lane.
 *
 * Two kernels share the tile decode and the epilogues. gemm_kernel<BM,BN,WGM,WGN> (8 or 4
 * waves, two waves per SIMD) serves the small tiles. gemm4w_kernel<TM,TN> is for the
 * large projections, as a 256 x 256 or a 288 x 192 tile (the second divides 4608-token problems
 * into a whole number of rounds over 256 CUs): 4 waves, one per SIMD, each owning 128 x 128
 * (144 x 96) of the tile with its 256 (216) accumulator registers pinned to AGPRs. A 128 x 128 wave tile needs 16 fragment reads per 64
 * MFMAs instead of 12 per 32, i.e. a third less LDS traffic per FLOP, which under the power
 * limit is what buys throughput (1020 -> 1145 TFLOP/s sustained back to back on the
 * 4608 x 18432 x 3072 projection). With a single wave per SIMD nothing hides latency for free,
 * so the loop is software-pipelined by hand: fragments are double-buffered in registers, every
 * third or fourth MFMA is followed by one LDS read for the next half-step and (in the second half) one
 * global->LDS load for the stage after next, and there is one barrier per 64-wide K step. The
 * reads come after their MFMA, not before it, so that the half-step opens with an MFMA whose
 * operands arrived long ago: the compiler puts an lgkmcnt(0) wait in front of the first MFMA after
 * the loop's back edge, and with a read issued just before it that wait exposed a full LDS latency
 * per K step. Global sources are a scalar base plus a 32-bit offset per lane, so stepping along K
 * is scalar work. Blocks are walked in serpentine order (one MFMA operand changes at a time).
 * A workgroup goes on to further tiles (one workgroup per compute unit is launched) and requests the
 * next tile's first stage before it stores the finished one.
 * One wave per SIMD does keep the matrix pipe full when its MFMAs are written by hand: a register-
 * resident loop of independent v_mfma_f32_16x16x32_bf16 reaches 2.4 PFLOP/s on zero operands and
 * 1.86 on random bits with 256 threads per compute unit, accumulators in VGPRs or AGPRs alike (the
 * same loop left to the compiler's builtin gets 1.46: it shuffles accumulators between the two
 * register files). Cycle stamps in this kernel on zero operands (4608 x 18432 x 3072, clocks near
 * their maximum) put 91 % of a wave's life in the K loop, 7 % in the epilogue and next-tile
 * set-up, 4 % in the mid-step wait and barrier; the K loop ran at 75 % of the MFMA issue rate
 * before the reads moved behind their MFMAs. On real operands the chip is at its power limit, in a
 * denoising step as well as back to back: removing those stalls made the kernel 5 % faster back to
 * back and the step 1 % faster.
 * The same loop also exists over a WGM x WGN grid of waves; with 8 waves (2 x 4, 128 x 64 each, two
 * per SIMD) on the 256 x 256 tile it runs at the speed of the 4-wave form and is kept for comparison
 * runs (tile id 4).
 *
 * Four kernels, then: gemm_kernel (small tiles), gemm_few_kernel (row ranges of at most 128 rows, where a
 * launch only streams weights), gemm4w_kernel (large tiles, two LDS stages; the
 * comparison form of the next one) and gemm4d_kernel (large tiles with an LDS ring per operand, the form the
 * transformer's projections and the VAE's convolutions run). What separates the last two is the barrier: __syncthreads() carries a fence
 * that waits for every global->LDS load in flight, so a two-stage loop can never have more than the next stage
 * on its way, requested one to two half-steps earlier; operands that come from HBM arrive later than that now and
 * then, and a wave that waits holds its three neighbours up at the barrier (measured: the same launch takes
 * 232-241 us when its operands are reused from the memory-side cache and 272-277 us when they rotate through
 * six buffer sets; a copy without the barrier does not care). gemm4d_kernel waits with a count instead
 * (s_waitcnt vmcnt(n) + s_barrier in one asm statement): everything but the last n loads, which belong to the
 * operand whose ring has a third slot and are needed a whole K step later.
 *
 * LDS rows are 128 bytes (64 bf16); the 16-byte chunk index is XOR-swizzled with a function of
 * the row so that the 16 rows a fragment read touches spread over all banks. A direct-to-LDS
 * load writes lane i's 16 bytes at (wave base + 16 i), so the swizzle is applied on the global
 * side: each lane fetches the chunk that belongs at its LDS position.
 */
#include "common.h"
#include <type_traits>
#include "../../include/flux_hip.h"
#include "../../include/flux_hip_debug.h"

#define GEMM_MAX_PARTS 4
struct GemmArgs {
    const bf16 *A[GEMM_MAX_PARTS];
    const bf16 *W[GEMM_MAX_PARTS];
    void *C[GEMM_MAX_PARTS];
    const float *gate[GEMM_MAX_PARTS];
    int M[GEMM_MAX_PARTS];
    int mt_end[GEMM_MAX_PARTS]; /* row tiles of parts 0..i together; unused parts repeat the total */
    int mtiles, ntiles, total_tiles;
    int vgrid; /* workgroups' worth of tiles (a multiple of 8); a launch with fewer workgroups walks them in strides of its size */
    int N, K, lda, ldw, ldc, w_row0, w_row1;
    /* fused [Q | K | V | gate | up] projection (EPI_QKV_SWIGLU): the first nq_cols columns (weight rows from w_row0)
     * are stored as bf16 to C, the other N - nq_cols are gate / up pairs (gate rows from w_row1, up rows from
     * w_row2) whose silu(gate) * up goes to C2; nq_tiles = nq_cols / tile width */
    int w_row2, nq_cols, nq_tiles, ldc2;
    void *C2;
    /* split-K: workgroup (tile, s) multiplies K-steps [s*kt_per, (s+1)*kt_per) and stores its
     * fp32 partial tile into ws[s][moff[part] + m][n]; a second kernel sums the slices */
    int ksplit, kt_per;
    float *ws;
    int moff[GEMM_MAX_PARTS], ws_rows;
    /* convolution epilogues (see flux_hip_conv): the operand's rows are the conv_rows positions of a zero-bordered
     * image conv_wp wide, channels contiguous; the GEMM's rows are its interior positions alone (conv_row), so that an
     * image of 2^n positions is a whole number of tiles (with the border rows computed and thrown away, 256 x 256 positions
     * x 512 channels were 522 tiles of 256 x 256, three rounds of 256 compute units instead of two). conv_wp = 0:
     * every row is computed. With 9 taps K runs over
     * [cin / 64 channel chunks][9 taps][64 channels]: K step kt = 9 * chunk + tap reads the
     * activation rows shifted by its tap's (dy, dx). The nine taps of a chunk follow each other so
     * that what one tap fetched is still in L2 when the next asks for the neighbouring rows
     * (tap-major order re-fetched wide images 3 to 10 times from HBM). */
    int conv_taps, conv_wp, conv_rows;
    int conv_stride, conv_in_wp; /* the operand's image: the same one, or for the downsampling steps one twice as large; stride 0: packed rows */
    int conv_packed_out;         /* the output holds the interior positions only, row m = GEMM row m */
    unsigned conv_magic; /* (2^32 - 1) / (conv_wp - 2) */
    const float *bias, *res;
    /* optional: per (row-tile half, 4-channel group) sums and sums of squares of what a convolution
     * epilogue writes, [prow][N/4][2], for the group norm that follows */
    float *stats;
    /* exponentials of attention scores (EPI_EXP): 2^(exp_scale * score - bias[row]) for columns below exp_keys, 0 beyond; the sums over each
     * wave's columns go to stats [row][2 * column tile + wave] */
    float exp_scale;
    int exp_keys;
};

/* internal epilogue: fp32 partial sums of one K slice of a convolution, rows = interior positions */
#define EPI_CONV_PARTIAL 9
template <int EPI> struct IsConv { static constexpr bool value = EPI == FLUX_HIP_EPI_CONV_BF16 || EPI == FLUX_HIP_EPI_CONV_F32 || EPI == EPI_CONV_PARTIAL; };

/* m / (conv_wp - 2): the product with the truncated reciprocal is the quotient or one less for every 32-bit m */
__device__ __forceinline__ int conv_div(const GemmArgs &g, int m) {
    const unsigned w = g.conv_wp - 2, q = __umulhi((unsigned)m, g.conv_magic);
    return (int)(q + ((unsigned)m - q * w >= w));
}
/* row of GEMM row m in the output: the m-th interior position of the bordered image */
template <int EPI>
__device__ __forceinline__ int conv_row(const GemmArgs &g, int m) {
    if (!IsConv<EPI>::value || g.conv_wp == 0 || g.conv_packed_out) return m;
    return m + 2 * conv_div(g, m) + g.conv_wp + 1;
}

/* ... and in the operand, where the 3x3 window is centred. With stride 2 (flux_vae.c:363-377: a row of zeros below and a column on
 * the right, no padding above and left) the window of output (y, x) starts at input (2 y, 2 x), so its centre is
 * (2 y + 2, 2 x + 2) of the bordered input; with stride 1 it is (y + 1, x + 1). */
template <int EPI>
__device__ __forceinline__ int conv_in_row(const GemmArgs &g, int m) {
    if (!IsConv<EPI>::value || g.conv_wp == 0 || g.conv_stride == 0) return m;
    const int y = conv_div(g, m), x = m - y * (g.conv_wp - 2);
    return g.conv_stride * ((y + 1) * g.conv_in_wp + x + 1);
}

/* Element offset of K step kt within an activation row. Plain GEMM: kt * 64. 3x3 convolution:
 * kt = 9 * chunk + tap; the tap selects a neighbour dy*Wp + dx rows away (uniform for the whole
 * launch, because border positions are rows of the operand too), the chunk a 64-channel slice. */
template <int EPI>
__device__ __forceinline__ int a_step_offset(const GemmArgs &g, int kt) {
    if (IsConv<EPI>::value) {
        /* kt / 9, kt % 9 for kt < 2048; a 1x1 convolution's step is a chunk at the middle tap. No branch: this stands in the K loops */
        const int nine = -(int)(g.conv_taps == 9), q = (kt * 7282) >> 16, chunk = kt + (nine & (q - kt)), tap = 4 + (nine & (kt - 9 * q - 4));
        const int dy = (tap * 11) >> 5, dx = tap - dy * 3;         /* tap / 3, tap % 3 for tap < 9 */
        return ((dy - 1) * g.conv_in_wp + (dx - 1)) * g.lda + chunk * 64;
    }
    return kt * 64;
}

/* internal epilogue: fp32 partial sums of one K slice (see split-K above) */
#define EPI_PARTIAL 5
/* internal epilogue of flux_hip_linear_qkv_swiglu: bf16 store for the leading column tiles, SiLU(gate) * up beyond */
#define EPI_QKV_SWIGLU 8
/* internal epilogue of flux_hip_linear_exp, see GemmArgs */
#define EPI_EXP 10

__device__ __forceinline__ int lds_swz(int r) { return ((r >> 1) & 7) ^ ((r & 1) << 2); }

#define GROUP_M 4
#define GLOBAL_PTR(p) ((const __attribute__((address_space(1))) void *)(p))
#define LDS_PTR(p) ((__attribute__((address_space(3))) void *)(p))
/* s_waitcnt vmcnt(0) only (expcnt and lgkmcnt fields left at their maxima) */
#define WAIT_VMCNT0() __builtin_amdgcn_s_waitcnt(0x0F70)

/* A convolution kernel's arguments, read anew: what only the epilogue and the step to the next tile need (and what the compiler
 * derives from it for their divisions) is more than the scalar registers hold across the K loops. */
__device__ __forceinline__ GemmArgs conv_args_again() {
    auto *ka = (const __attribute__((address_space(4))) GemmArgs *)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(ka));
    GemmArgs a = {};
    a.M[0] = ka->M[0]; a.C[0] = ka->C[0]; a.bias = ka->bias; a.res = ka->res; a.stats = ka->stats;
    a.N = ka->N; a.ldc = ka->ldc; a.mtiles = ka->mtiles; a.ntiles = ka->ntiles; a.total_tiles = ka->total_tiles; a.vgrid = ka->vgrid;
    a.ksplit = ka->ksplit;
    a.conv_wp = ka->conv_wp; a.conv_rows = ka->conv_rows; a.conv_magic = ka->conv_magic; a.conv_packed_out = ka->conv_packed_out;
    return a;
}

/* Which tile (and K slice) a workgroup owns. Workgroups are dealt round-robin to the 8 XCDs;
 * each XCD gets a contiguous run of tiles so that its L2 sees the reuse, and tiles are walked in
 * groups of GROUP_M rows. */
struct TileId {
    int ks, tm, tn, prob, tml;
};
template <bool ONE> /* one matrix, not parts */
__device__ __forceinline__ bool decode_tile(const GemmArgs &g, int vb, TileId &t) {
    int per_xcd = g.vgrid >> 3;
    int logical = (vb & 7) * per_xcd + (vb >> 3);
    if (logical >= g.total_tiles * g.ksplit) return false;
    t.ks = logical / g.total_tiles;
    logical -= t.ks * g.total_tiles;
    int per_group = GROUP_M * g.ntiles;
    int grp = logical / per_group;
    int first_m = grp * GROUP_M;
    int gsz = min(g.mtiles - first_m, GROUP_M);
    int in_grp = logical - grp * per_group;
    t.tm = first_m + in_grp % gsz;
    t.tn = in_grp / gsz;
    if (ONE) {
        t.prob = 0;
        t.tml = t.tm;
        return true;
    }
    t.prob = (t.tm >= g.mt_end[0]) + (t.tm >= g.mt_end[1]) + (t.tm >= g.mt_end[2]);
    t.tml = t.prob ? t.tm - g.mt_end[t.prob - 1] : t.tm;
    return true;
}

/* Which feature of its wave's slice of the output row r of MFMA block blk computes, for the two epilogues that
 * store bf16. In the accumulator a lane holds four consecutive MFMA rows of a block (rows 4 (lane / 16) .. + 3): with
 * rows numbered plainly that is four consecutive features, an 8-byte store, and a wave's store instruction writes
 * 32 bytes to each of 16 output rows. Here two neighbouring blocks interleave instead: block 2p takes features
 * 32 p + 8 q + 0 .. 3 on its rows 4 q .. 4 q + 3 and block 2p + 1 features 32 p + 8 q + 4 .. 7, so that a lane's
 * results of the two blocks are eight consecutive features: one 16-byte store, 64 bytes per output row and
 * instruction, half as many store instructions and write requests. Only the weight rows a block reads change. */
__device__ __forceinline__ int bf16_pair_feature(int blk, int r) { return 32 * (blk >> 1) + 8 * (r >> 2) + 4 * (blk & 1) + (r & 3); }
/* the same for a wave that owns TN blocks: with TN odd the last block has no neighbour and keeps the plain numbering */
template <int TN>
__device__ __forceinline__ int bf16_feature(int blk, int r) { return blk < (TN & ~1) ? bf16_pair_feature(blk, r) : 16 * blk + r; }
/* Tile widths that do not divide all of the models' matrix widths (224: 3072 = 13 x 224 + 160, 9216 = 41 x 224 + 32; 96: 19456 = 202 x 96 + 64): the
 * last column tile is cut off. Its missing weight rows are read from the matrix's last row and its missing columns are
 * not stored (whole 16-column blocks for fp32 outputs, whole pairs of blocks for bf16: N is a multiple of 32). */
template <int BN> struct CutTile { static constexpr bool value = BN % 64 != 0; };
/* the tiles of gemm4x_kernel */
template <int BN, int WM> struct IsWide { static constexpr bool value = 2 * WM * BN > 256 * 256; };
/* tiles whose last column tile is cut at any multiple of eight columns, lane by lane: those, 256 x 160 and gemm_few_kernel's */
template <int BN, int WM> struct LaneCut { static constexpr bool value = CutTile<BN>::value && (IsWide<BN, WM>::value || BN == 160 || WM == 16); };
/* SiLU(gate) * up: blocks alternate gate, up, so that a lane holds matching pairs; the (gate, up) pairs interleave
 * two by two in the same way, and a last odd pair keeps the plain numbering (features 16 k + r). With an odd number of
 * blocks the last one holds gate rows and up rows, two and two: a lane's four results are gate, gate, up, up of two features. */
template <int TN>
__device__ __forceinline__ int swiglu_feature(int blk, int r) {
    const int k = blk >> 1;
    if (TN % 2 && blk == TN - 1) return 16 * k + 2 * (r >> 2) + (r & 1);
    return k < 2 * (TN / 4) ? bf16_pair_feature(k, r) : 16 * k + r;
}
template <int TN>
__device__ __forceinline__ bool swiglu_up(int blk, int r) { return TN % 2 && blk == TN - 1 ? r & 2 : blk & 1; }

/* Weight row that feeds column v of the tile. */
template <int BN, int WN, int EPI>
__device__ __forceinline__ int weight_row(const GemmArgs &g, int tn, int v) {
    constexpr int TN = WN / 16;
    const int wv = v / WN, blk = (v % WN) >> 4, r = v & 15;
    if (EPI == FLUX_HIP_EPI_SWIGLU || (EPI == EPI_QKV_SWIGLU && tn >= g.nq_tiles)) {
        int idx = wv * (WN / 2) + swiglu_feature<TN>(blk, r);
        if (CutTile<BN>::value && EPI == FLUX_HIP_EPI_SWIGLU) idx = min(idx, g.N / 2 - 1 - tn * (BN / 2));
        if (CutTile<BN>::value && EPI == EPI_QKV_SWIGLU) idx = min(idx, g.w_row2 - g.w_row1 - 1 - (tn - g.nq_tiles) * (BN / 2));
        if (EPI == EPI_QKV_SWIGLU) return (swiglu_up<TN>(blk, r) ? g.w_row2 : g.w_row1) + (tn - g.nq_tiles) * (BN / 2) + idx;
        return (swiglu_up<TN>(blk, r) ? g.w_row1 : g.w_row0) + tn * (BN / 2) + idx;
    }
    int col;
    if (EPI == FLUX_HIP_EPI_BF16 || EPI == EPI_QKV_SWIGLU || EPI == FLUX_HIP_EPI_CONV_BF16 || EPI == EPI_EXP) col = tn * BN + wv * WN + bf16_feature<TN>(blk, r);
    else col = tn * BN + v;
    if (CutTile<BN>::value) col = min(col, (EPI == EPI_QKV_SWIGLU ? g.nq_cols : g.N) - 1);
    return g.w_row0 + col;
}

/* eight bf16 to consecutive addresses: one 16-byte store where the address allows it, else two of 8 bytes */
__device__ __forceinline__ void store_bf16x8(bf16 *p, bf16x4 lo, bf16x4 hi, bool aligned16) {
    if (aligned16) {
        bf16x8 o;
#pragma unroll
        for (int e = 0; e < 4; e++) { o[e] = lo[e]; o[4 + e] = hi[e]; }
        *(bf16x8 *)p = o;
    } else {
        *(bf16x4 *)p = lo;
        *(bf16x4 *)(p + 4) = hi;
    }
}

template <bool V> struct BoolC { static constexpr bool value = V; };
template <int V> struct IntC { static constexpr int value = V; };

/* Accumulator element e of block (i, j): feature n = 4*(lane/16) + e of the 16-column block,
 * token m = lane%16 of the 16-row block. */
template <int BN, int WM, int WN, int EPI, bool HERE = false>
__device__ __forceinline__ void store_tile_to(const GemmArgs &g, const TileId &t, f32x4 (&acc_in)[WN / 16][WM / 16], int m0, int M,
                                              int wm, int wn, int l15, int lq, int prow, void *Cp, const int ldc, const int tn, const int cols) {
    constexpr int TM = WM / 16, TN = WN / 16;
    const int prob = t.prob, n0 = tn * BN, ks = t.ks;
    constexpr bool LANE_CUT = LaneCut<BN, WM>::value;
    const bool aligned16 = (((uintptr_t)Cp | ((uintptr_t)ldc << 1)) & 15) == 0; /* every 8-feature group of the output starts on 16 bytes */
    f32x4 acc_here[HERE ? TN : 1][HERE ? TM : 1];
    auto &acc = [&]() -> auto & { if constexpr (HERE) return acc_here; else return acc_in; }();
    if constexpr (EPI == FLUX_HIP_EPI_RESID && HERE) {
        /* x += gate * acc on the fp32 residual: a read, and a write that depends on it. Row block by row block in
         * program order that is a chain of round trips to memory (request a row's values, wait, store; the wait
         * counter also holds the stores of the row before, so every wait is for those as well): nine such chains made
         * up most of the 57 us that this epilogue cost a 288 x 192 x 12288 tile's launch of 261 us. Here the values of
         * row block j + 1 are requested before row block j is touched: the wait for block j's values leaves the block
         * before's stores and the next block's loads in flight. Rows beyond M read the last row (no branch around the
         * loads) and store nothing; a wave whose rows are all valid runs a copy without that test, i.e. without
         * branches (behind a skipped store the compiler must assume that the loads in front of it are still under
         * way, and it waits for them before it reuses their registers: one row block in flight instead of two). */
        const auto cut = [&](int i) { return CutTile<BN>::value && n0 + wn * WN + i * 16 >= g.N; }; /* the same for the whole wave */
        /* the unit that is requested ahead: a row block's TN column blocks, or half of them with eight (256 x 256, 192 x 256), where
         * two whole ones, the gate and the next tile's fragments are more than the VGPRs hold (192 x 256 parked seven in AGPRs) */
        constexpr int UN = TN > 6 && TN % 2 == 0 ? TN / 2 : TN, UPR = TN / UN, NU = TM * UPR;
        constexpr int NB = 2; /* units in flight, the one being stored included (a third one measured no different: what is left is the burst itself) */
        f32x4 gt[TN], xb[NB][UN];
#pragma unroll
        for (int i = 0; i < TN; i++)
            if (!cut(i)) gt[i] = *(const f32x4 *)(g.gate[prob] + n0 + wn * WN + i * 16 + lq * 4);
        const auto fetch = [&](int u) {
            const int j = u / UPR, i0 = u % UPR * UN;
            const float *p = (const float *)Cp + (size_t)min(m0 + wm * WM + j * 16 + l15, M - 1) * ldc + n0 + wn * WN + lq * 4;
#pragma unroll
            for (int i = 0; i < UN; i++)
                if (!cut(i0 + i)) xb[u % NB][i] = *(const f32x4 *)(p + (i0 + i) * 16);
        };
        const auto rows = [&](auto full_c) {
#pragma unroll
            for (int u = 0; u < NB - 1 && u < NU; u++) fetch(u);
#pragma unroll
            for (int u = 0; u < NU; u++) {
                const int j = u / UPR, i0 = u % UPR * UN;
                if (u + NB - 1 < NU) fetch(u + NB - 1);
                const int m = m0 + wm * WM + j * 16 + l15;
                float *p = (float *)Cp + (size_t)m * ldc + n0 + wn * WN + lq * 4;
#pragma unroll
                for (int i = 0; i < UN; i++) {
                    if (cut(i0 + i)) continue;
                    f32x4 a = acc_in[i0 + i][j]; /* out of its AGPRs here, one block at a time */
                    asm volatile("" : "+v"(a));
                    f32x4 x = xb[u % NB][i];
#pragma unroll
                    for (int e = 0; e < 4; e++) x[e] += gt[i0 + i][e] * a[e];
                    if (decltype(full_c)::value || m < M) *(f32x4 *)(p + (i0 + i) * 16) = x;
                }
            }
        };
        if (m0 + wm * WM + WM <= M) rows(BoolC<true>{});
        else rows(BoolC<false>{});
        return;
    }
#pragma unroll
    for (int j = 0; j < TM; j++) {
        const int m = m0 + wm * WM + j * 16 + l15;
        if (m >= M) continue;
        if constexpr (HERE) {
#pragma unroll
            for (int i = 0; i < TN; i++) {
                acc[i][j] = acc_in[i][j];
                asm volatile("" : "+v"(acc[i][j]));
            }
        }
        if (EPI == FLUX_HIP_EPI_SWIGLU) {
            if (CutTile<BN>::value && tn * BN + wn * WN >= cols) continue; /* the same for the whole wave (gate and up columns count) */
            /* see swiglu_feature: two (gate, up) pairs give eight consecutive features, a last odd pair four, a last odd block two */
            const int left = LANE_CUT ? cols / 2 - tn * (BN / 2) - wn * (WN / 2) : 0; /* features of the wave's that exist */
            bf16 *C = (bf16 *)Cp + (size_t)m * ldc + tn * (BN / 2) + wn * (WN / 2);
            bf16x4 o[TN / 2];
#pragma unroll
            for (int k = 0; k < TN / 2; k++)
#pragma unroll
                for (int e = 0; e < 4; e++) o[k][e] = (bf16)(silu_f(acc[2 * k][j][e]) * acc[2 * k + 1][j][e]);
#pragma unroll
            for (int p = 0; p < TN / 4; p++)
                if (!LANE_CUT || 32 * p + 8 * lq < left) store_bf16x8(C + 32 * p + 8 * lq, o[2 * p], o[2 * p + 1], aligned16);
            if (TN / 2 % 2 && (!LANE_CUT || 16 * (TN / 2 - 1) + 4 * lq < left)) *(bf16x4 *)(C + 16 * (TN / 2 - 1) + 4 * lq) = o[TN / 2 - 1];
            if (TN % 2 && (!LANE_CUT || 16 * (TN / 2) + 2 * lq < left)) {
                const f32x4 a = acc[TN - 1][j];
                *(bf16x2 *)(C + 16 * (TN / 2) + 2 * lq) = bf16x2{(bf16)(silu_f(a[0]) * a[2]), (bf16)(silu_f(a[1]) * a[3])};
            }
        } else if (EPI == FLUX_HIP_EPI_BF16) {
            /* see bf16_pair_feature: blocks 2p and 2p + 1 give eight consecutive features */
            bf16 *C = (bf16 *)Cp + (size_t)m * ldc + n0 + wn * WN + 8 * lq;
#pragma unroll
            for (int p = 0; p < TN / 2; p++) {
                if (CutTile<BN>::value && n0 + wn * WN + 32 * p + (LANE_CUT ? 8 * lq : 0) >= cols) continue; /* (without LANE_CUT the same for the whole wave) */
                bf16x4 lo, hi;
#pragma unroll
                for (int e = 0; e < 4; e++) { lo[e] = (bf16)acc[2 * p][j][e]; hi[e] = (bf16)acc[2 * p + 1][j][e]; }
                store_bf16x8(C + 32 * p, lo, hi, aligned16);
            }
            if (TN % 2 && !(CutTile<BN>::value && n0 + wn * WN + 16 * (TN - 1) + (LANE_CUT ? 4 * lq : 0) >= cols)) { /* a last block without a neighbour */
                bf16x4 o;
#pragma unroll
                for (int e = 0; e < 4; e++) o[e] = (bf16)acc[TN - 1][j][e];
                *(bf16x4 *)((bf16 *)Cp + (size_t)m * ldc + n0 + wn * WN + 16 * (TN - 1) + 4 * lq) = o;
            }
        } else {
#pragma unroll
            for (int i = 0; i < TN; i++) {
                if (CutTile<BN>::value && n0 + wn * WN + i * 16 >= g.N) continue; /* the same for the whole wave */
                const int n = n0 + wn * WN + i * 16 + lq * 4;
                if (EPI == EPI_PARTIAL || EPI == EPI_CONV_PARTIAL) {
                    *(f32x4 *)(g.ws + ((size_t)ks * g.ws_rows + g.moff[prob] + m) * g.N + n) = acc[i][j];
                } else if (EPI == FLUX_HIP_EPI_F32) {
                    *(f32x4 *)((float *)Cp + (size_t)m * ldc + n) = acc[i][j];
                } else if (EPI == FLUX_HIP_EPI_F32_T) {
#pragma unroll
                    for (int e = 0; e < 4; e++) ((float *)Cp)[(size_t)(n + e) * ldc + m] = acc[i][j][e];
                } else if (EPI == FLUX_HIP_EPI_RESID) {
                    float *p = (float *)Cp + (size_t)m * ldc + n;
                    f32x4 x = *(f32x4 *)p;
                    f32x4 gt = *(const f32x4 *)(g.gate[prob] + n);
#pragma unroll
                    for (int e = 0; e < 4; e++) x[e] += gt[e] * acc[i][j][e];
                    *(f32x4 *)p = x;
                }
            }
        }
    }
}

/* What a convolution's tile stores: acc + bias [+ residual] at the interior positions, zeros at the border, and (g.stats) the
 * sums for the group norm that follows. Two column blocks at a time over all row blocks, so that bias and sums of the
 * whole tile never sit in registers beside the accumulators and the next tile's fragments; as in the residual epilogue above,
 * the residual of the next row blocks is requested before the present ones are touched. bf16 outputs leave as 16-byte
 * stores (bf16_pair_feature). The border is not computed: the positions behind the last pixel of an image row go with the
 * tile that holds that pixel, the rows above and below the image are shared out over all row tiles. */
template <int BN, int WM, int WN, int EPI, int WGM, bool HERE>
__device__ __forceinline__ void store_conv_tile(const GemmArgs &g, const TileId &t, f32x4 (&acc_in)[WN / 16][WM / 16], int m0, int M,
                                                int wm, int wn, int l15, int lq, int prow) {
    constexpr int TM = WM / 16, TN = WN / 16, BM = WM * WGM;
    constexpr bool F32 = EPI == FLUX_HIP_EPI_CONV_F32;
    static_assert(TN % 2 == 0, "bf16 outputs pair 16-column blocks");
    const int nw = t.tn * BN + wn * WN, ldc = g.ldc;
    constexpr int RB = TM * TN * 4 > 224 ? 1 : 2, UPP = (TM + RB - 1) / RB, NU = TN / 2 * UPP; /* a unit: RB row blocks of one pair of column blocks */
    using Off = std::conditional_t<HERE, unsigned, size_t>; /* (conv_launch sends outputs beyond 2^32 elements to the small tiles) */
    Off off[TM]; /* first element of the wave's columns in each of this lane's rows; rows beyond M repeat the last one */
#pragma unroll
    for (int j = 0; j < TM; j++) off[j] = (Off)conv_row<EPI>(g, min(m0 + wm * WM + j * 16 + l15, M - 1)) * (Off)ldc + nw;
    const auto rows = [&](auto res_c) {
        constexpr bool RES = decltype(res_c)::value;
        f32x4 xb[2][RB][2];
        const auto fetch = [&](int u) {
            const int i0 = u / UPP * 2, j0 = u % UPP * RB;
#pragma unroll
            for (int r = 0; r < RB; r++)
#pragma unroll
                for (int k = 0; k < 2; k++)
                    if (j0 + r < TM) xb[u & 1][r][k] = *(const f32x4 *)(g.res + (size_t)off[j0 + r] + i0 * 16 + (F32 ? k * 16 + lq * 4 : lq * 8 + k * 4));
        };
        if (RES) fetch(0);
#pragma unroll
        for (int ip = 0; ip < TN / 2; ip++) {
            const int c0 = F32 ? ip * 32 + lq * 4 : ip * 32 + lq * 8, cs = F32 ? 16 : 4; /* columns of block 2 ip, and block 2 ip + 1 behind it */
            const f32x4 bv[2] = {*(const f32x4 *)(g.bias + nw + c0), *(const f32x4 *)(g.bias + nw + c0 + cs)};
            float st[2][2] = {{0.0f, 0.0f}, {0.0f, 0.0f}};
            int left = M - (m0 + wm * WM + l15); /* rows of this lane's column of row blocks below M, compared anew per pair: TM kept lane masks are spilled */
            asm volatile("" : "+v"(left));
#pragma unroll
            for (int ju = 0; ju < UPP; ju++) {
                const int u = ip * UPP + ju;
                if (RES && u + 1 < NU) fetch(u + 1);
#pragma unroll
                for (int r = 0; r < RB; r++) {
                    const int j = ju * RB + r;
                    if (j >= TM) continue;
                    const bool ok = j * 16 < left;
                    f32x4 v[2];
#pragma unroll
                    for (int k = 0; k < 2; k++) {
                        f32x4 a = acc_in[2 * ip + k][j];
                        if (HERE) asm volatile("" : "+v"(a)); /* out of its AGPRs here, one block at a time */
                        float s = 0.0f, q = 0.0f;
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            v[k][e] = RES ? xb[u & 1][r][k][e] + a[e] + bv[k][e] : a[e] + bv[k][e];
                            s += v[k][e];
                            q += v[k][e] * v[k][e];
                        }
                        st[k][0] += ok ? s : 0.0f;
                        st[k][1] += ok ? q : 0.0f;
                    }
                    if (F32) {
                        float *p = (float *)g.C[0] + (size_t)off[j] + c0;
                        if (ok) {
                            *(f32x4 *)p = v[0];
                            *(f32x4 *)(p + 16) = v[1];
                        }
                    } else {
                        bf16x4 o[2];
#pragma unroll
                        for (int e = 0; e < 4; e++) { o[0][e] = (bf16)v[0][e]; o[1][e] = (bf16)v[1][e]; }
                        if (ok) store_bf16x8((bf16 *)g.C[0] + (size_t)off[j] + c0, o[0], o[1], true);
                    }
                }
            }
            if (g.stats) {
                /* sum over the 16 rows held by lanes of equal lane/16, then one lane per column quad stores */
#pragma unroll
                for (int k = 0; k < 2; k++) {
#pragma unroll
                    for (int o = 1; o < 16; o <<= 1) {
                        st[k][0] += __shfl_xor(st[k][0], o);
                        st[k][1] += __shfl_xor(st[k][1], o);
                    }
                    const f32x2 v = {st[k][0], st[k][1]};
                    if (l15 == 0) *(f32x2 *)(g.stats + ((size_t)prow * (g.N >> 2) + ((nw + c0 + k * cs) >> 2)) * 2) = v;
                }
            }
        }
    };
    if (g.res) rows(BoolC<true>{});
    else rows(BoolC<false>{});
    const int lane = lq * 16 + l15;
    if (g.conv_wp > 0 && !g.conv_packed_out) {
        constexpr int QPW = WN / 4, PPI = 64 / QPW; /* lanes per position, positions per instruction */
        const int wp = g.conv_wp, y0 = conv_div(g, m0), y1 = conv_div(g, min(m0 + BM, M));
        const int nside = 2 * (y1 - y0), nedge = 2 * wp + 1, per = (nedge + g.mtiles - 1) / g.mtiles;
        const int e0 = min(nedge, t.tm * per), total = nside + min(nedge - e0, per);
        for (int k = wm * PPI + lane / QPW; k < total; k += WGM * PPI) {
            const int e = e0 + k - nside;
            const int p = k < nside ? (y0 + (k >> 1) + 2) * wp - 1 + (k & 1) : e <= wp ? e : g.conv_rows - wp + (e - wp - 1);
            const size_t at = (size_t)p * ldc + nw + (lane % QPW) * 4;
            if (F32) *(f32x4 *)((float *)g.C[0] + at) = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            else *(bf16x4 *)((bf16 *)g.C[0] + at) = bf16x4{(bf16)0.0f, (bf16)0.0f, (bf16)0.0f, (bf16)0.0f};
        }
    }
}

/* Attention scores as unnormalised probabilities, see GemmArgs. The rows' references are requested together in front of everything, so that
 * no row block waits for the stores of the one before; only the last column tile has columns to clear. Stores as for bf16 above. */
template <int BN, int WM, int WN>
__device__ __forceinline__ void store_exp_tile(const GemmArgs &g, const TileId &t, f32x4 (&acc)[WN / 16][WM / 16], int m0, int M, int wm, int wn, int l15, int lq) {
    constexpr int TM = WM / 16, TN = WN / 16;
    const int n = t.tn * BN + wn * WN + 8 * lq, first = m0 + wm * WM + l15;
    float r[TM];
#pragma unroll
    for (int j = 0; j < TM; j++) r[j] = g.bias[min(first + 16 * j, M - 1)];
    const auto rows = [&](auto cut_c) {
#pragma unroll
        for (int j = 0; j < TM; j++) {
            const int m = min(first + 16 * j, M - 1); /* rows beyond the last one are copies of it, operand and reference: they store the same */
            bf16 *C = (bf16 *)g.C[0] + (size_t)m * g.ldc + n;
            float sum = 0.0f;
            int keys = g.exp_keys - n;
            asm volatile("" : "+v"(keys)); /* compared anew for each row: 32 kept lane masks are spilled */
#pragma unroll
            for (int p = 0; p < TN / 2; p++) {
                float v[8];
#pragma unroll
                for (int k = 0; k < 2; k++) {
                    f32x4 a = acc[2 * p + k][j];
                    asm volatile("" : "+v"(a)); /* out of its AGPRs here, one block at a time */
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        v[4 * k + e] = fast_exp2(fmaf(a[e], g.exp_scale, -r[j]));
                        if (decltype(cut_c)::value && 32 * p + 4 * k + e >= keys) v[4 * k + e] = 0.0f;
                    }
                }
                bf16x4 lo, hi;
#pragma unroll
                for (int e = 0; e < 4; e++) { lo[e] = (bf16)v[e]; hi[e] = (bf16)v[4 + e]; }
                store_bf16x8(C + 32 * p, lo, hi, true);
                /* of what is stored: a row's largest probability then carries no rounding of its own into the quotient */
#pragma unroll
                for (int e = 0; e < 4; e++) sum += (float)lo[e] + (float)hi[e];
            }
            sum += __shfl_xor(sum, 16);
            sum += __shfl_xor(sum, 32);
            if (lq == 0) g.stats[(size_t)m * (2 * g.ntiles) + 2 * t.tn + wn] = sum;
        }
    };
    if (t.tn * BN + BN > g.exp_keys) rows(BoolC<true>{});
    else rows(BoolC<false>{});
}

/* Cp, ldc, tn: where the tile goes - the part's output, or for the fused [Q|K|V|gate|up] projection the output of the
 * side of the boundary the tile lies on (the tile width divides nq_cols, so a tile is wholly on one side) */
template <int BN, int WM, int WN, int EPI, int WGM, bool PINNED = false>
__device__ __forceinline__ void store_tile(const GemmArgs &g, const TileId &t, f32x4 (&acc)[WN / 16][WM / 16], int m0, int M,
                                           int wm, int wn, int l15, int lq, int prow) {
    if constexpr (EPI == FLUX_HIP_EPI_CONV_BF16 || EPI == FLUX_HIP_EPI_CONV_F32) {
        store_conv_tile<BN, WM, WN, EPI, WGM, PINNED>(g, t, acc, m0, M, wm, wn, l15, lq, prow);
    } else if constexpr (EPI == EPI_EXP) {
        store_exp_tile<BN, WM, WN>(g, t, acc, m0, M, wm, wn, l15, lq);
    } else if constexpr (EPI == EPI_QKV_SWIGLU) {
        /* HERE = true: each side reads the accumulators through an empty asm statement, row by row. The conversions
         * are then work of that side; left to itself the compiler converted the whole tile to bf16 in front of the
         * branch, for both sides, and kept the hundred results in registers next to the other side's work, past
         * what the register file holds beside the fragments. */
        if (t.tn < g.nq_tiles) store_tile_to<BN, WM, WN, FLUX_HIP_EPI_BF16, true>(g, t, acc, m0, M, wm, wn, l15, lq, prow, g.C[0], g.ldc, t.tn, g.nq_cols);
        else store_tile_to<BN, WM, WN, FLUX_HIP_EPI_SWIGLU, true>(g, t, acc, m0, M, wm, wn, l15, lq, prow, g.C2, g.ldc2, t.tn - g.nq_tiles, g.N - g.nq_cols);
    } else {
        /* PINNED: the kernels whose accumulators live in AGPRs take them out row by row as well (the 16-byte / 8-byte
         * choice of the bf16 stores is a branch with the same conversions on both sides) */
        store_tile_to<BN, WM, WN, EPI, PINNED>(g, t, acc, m0, M, wm, wn, l15, lq, prow, g.C[t.prob], g.ldc, t.tn, g.N);
    }
}

template <int BM, int BN, int WGM, int WGN, int EPI>
__global__ __launch_bounds__(WGM *WGN * 64) void gemm_kernel(GemmArgs g) {
    constexpr int T = WGM * WGN * 64;
    constexpr int WM = BM / WGM, WN = BN / WGN, TM = WM / 16, TN = WN / 16;
    constexpr int RPP = T / 8; /* tile rows fetched per pass: one wave instruction covers 8 rows */
    constexpr int PA = BM / RPP, PB = BN / RPP;
    constexpr int STAGE = (BM + BN) * 128;
    static_assert(BM % RPP == 0 && BN % RPP == 0, "tile rows must divide evenly over threads");
    static_assert((EPI != FLUX_HIP_EPI_SWIGLU && EPI != EPI_QKV_SWIGLU) || (TN % 2 == 0), "swiglu pairs 16-column blocks");
    extern __shared__ __attribute__((aligned(16))) char smem[];

    TileId t;
    if (!decode_tile<IsConv<EPI>::value>(g, blockIdx.x, t)) return;
    const int ks = t.ks, tn = t.tn, prob = t.prob;
    const bf16 *__restrict__ A = g.A[prob];
    const bf16 *__restrict__ W = g.W[prob];
    const int M = g.M[prob];
    const int m0 = t.tml * BM;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WGN, wn = wave % WGN;
    const int lrow = tid >> 3, lchunk = tid & 7;

    /* Per-lane global sources (already un-swizzled) and per-wave LDS destinations. */
    const bf16 *a_ptr[PA];
    const bf16 *b_ptr[PB];
    int a_lds[PA], b_lds[PB];
#pragma unroll
    for (int i = 0; i < PA; i++) {
        int r = lrow + i * RPP;
        int gm = conv_in_row<EPI>(g, min(m0 + r, M - 1));
        a_ptr[i] = A + (size_t)gm * g.lda + ((lchunk ^ lds_swz(r)) << 3);
        a_lds[i] = (wave * 8 + i * RPP) * 128;
    }
#pragma unroll
    for (int i = 0; i < PB; i++) {
        int v = lrow + i * RPP; /* column of the tile */
        int wrow = weight_row<BN, WN, EPI>(g, tn, v);
        b_ptr[i] = W + (size_t)wrow * g.ldw + ((lchunk ^ lds_swz(v)) << 3);
        b_lds[i] = BM * 128 + (wave * 8 + i * RPP) * 128;
    }
    auto issue = [&](int kt, int stage) {
        char *base = smem + stage * STAGE;
        const int aoff = a_step_offset<EPI>(g, kt);
#pragma unroll
        for (int i = 0; i < PA; i++)
            __builtin_amdgcn_global_load_lds(GLOBAL_PTR(a_ptr[i] + aoff), LDS_PTR(base + a_lds[i]), 16, 0, 0);
#pragma unroll
        for (int i = 0; i < PB; i++)
            __builtin_amdgcn_global_load_lds(GLOBAL_PTR(b_ptr[i] + kt * 64), LDS_PTR(base + b_lds[i]), 16, 0, 0);
    };
    const int kt_begin = ks * g.kt_per;
    const int KT = min(g.K >> 6, kt_begin + g.kt_per) - kt_begin;
    if (KT > 0) issue(kt_begin, 0);

    f32x4 acc[TN][TM];
#pragma unroll
    for (int i = 0; i < TN; i++)
#pragma unroll
        for (int j = 0; j < TM; j++)
#pragma unroll
            for (int e = 0; e < 4; e++) acc[i][j][e] = 0.0f;

    const int l15 = lane & 15, lq = lane >> 4;
    const int swzl = lds_swz(l15);
    const int a_frag = (wm * WM + l15) * 128;
    const int b_frag = BM * 128 + (wn * WN + l15) * 128;

    for (int kt = 0; kt < KT; kt++) {
        /* the stage has landed for this wave; after the barrier it has for all, and everyone is done reading the other one, which is refilled */
        WAIT_VMCNT0();
        __syncthreads();
        const int cur = kt & 1;
        if (kt + 1 < KT) issue(kt_begin + kt + 1, cur ^ 1);
        const char *st = smem + cur * STAGE;
#pragma unroll
        for (int kk = 0; kk < 2; kk++) {
            const int coff = ((kk * 4 + lq) ^ swzl) << 4;
            bf16x8 fa[TM], fb[TN];
#pragma unroll
            for (int t = 0; t < TM; t++) fa[t] = *(const bf16x8 *)(st + a_frag + t * 16 * 128 + coff);
#pragma unroll
            for (int t = 0; t < TN; t++) fb[t] = *(const bf16x8 *)(st + b_frag + t * 16 * 128 + coff);
#pragma unroll
            for (int i = 0; i < TN; i++)
#pragma unroll
                for (int j = 0; j < TM; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[i], fa[j], acc[i][j], 0, 0, 0);
        }
    }

    store_tile<BN, WM, WN, EPI, WGM>(g, t, acc, m0, M, wm, wn, l15, lq, t.tm * WGM + wm);
}

/* Projections of few rows (at most 128 per part): weights streamed once, hardly any arithmetic. What bounds them is how fast a compute unit takes in
 * cold lines, 50 to 55 KB a microsecond however many it has requested beyond 32 KB (loads return in order, so activations from the L2 wait
 * behind weights from HBM), and then HBM itself. Hence: as many columns per workgroup as leave every unit one tile (BN = 80 to 144 in steps
 * of 16, the last column tile cut off), and no loads for rows that do not exist: the loads of a K step, eight rows each, are dealt out to
 * the eight waves, those of ceil(M / 8) activation groups and BN / 8 weight groups. A wave owns 16 rows and all columns; waves beyond the last row only
 * load. One ring of 4 to 6 stages fills the LDS. The order of additions is that of the other tiles.
 * Against a ring of 96 x 96 and 128 x 96 tiles in which every wave loaded its share of all 96 or 128 rows, weights from HBM: 80 rows (64 + 16)
 * of the fused 27648 x 3072 37.7 -> 35.8 us, 9216 x 3072 with two weight matrices 29.6 -> 25.4, their SwiGLU 18432 49.5 -> 44.5, 3072 x 9216 34.6 ->
 * 29.8, 3072 x 3072 18.1 -> 16.6; 19456 x 2560 at 16 rows 24.8 -> 21.4 (4.7 TB/s), at 128 rows 34.4 -> 30.2. */
template <int BN, int EPI>
__global__ __launch_bounds__(512) void gemm_few_kernel(GemmArgs g) {
    constexpr int BM = 128, TN = BN / 16, STAGE = (BM + BN) * 128, NS = 160 * 1024 / STAGE < 6 ? 160 * 1024 / STAGE : 6;
    constexpr int CM = (BM / 8 + BN / 8 + 7) / 8; /* a wave's loads per K step, at most */
    extern __shared__ __attribute__((aligned(16))) char smem[];
    TileId t;
    if (!decode_tile<false>(g, blockIdx.x, t)) return;
    const int M = g.M[t.prob], lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int na = (M + 7) >> 3, own = (na + BN / 8 - wave + 7) >> 3; /* this wave's loads */
    const bf16 *src[CM];
    int dst[CM];
#pragma unroll
    for (int k = 0; k < CM; k++) {
        const int i = wave + 8 * k;
        const bool act = i < na;
        const int r = 8 * (act ? i : min(i - na, BN / 8 - 1)) + (lane >> 3), chunk = ((lane & 7) ^ lds_swz(r)) << 3;
        src[k] = act ? g.A[t.prob] + (size_t)min(r, M - 1) * g.lda + chunk : g.W[t.prob] + (size_t)weight_row<BN, BN, EPI>(g, t.tn, r) * g.ldw + chunk;
        dst[k] = act ? i * 1024 : BM * 128 + (i - na) * 1024;
    }
    const int kt_begin = t.ks * g.kt_per, KT = min(g.K >> 6, kt_begin + g.kt_per) - kt_begin;
    auto issue = [&](int kt, int stage) {
#pragma unroll
        for (int k = 0; k < CM; k++)
            if (k < own) __builtin_amdgcn_global_load_lds(GLOBAL_PTR(src[k] + (kt_begin + kt) * 64), LDS_PTR(smem + stage * STAGE + dst[k]), 16, 0, 0);
    };
#pragma unroll
    for (int s = 0; s < NS - 1; s++)
        if (s < KT) issue(s, s);
    f32x4 acc[TN][1];
#pragma unroll
    for (int i = 0; i < TN; i++)
#pragma unroll
        for (int e = 0; e < 4; e++) acc[i][0][e] = 0.0f;
    const int l15 = lane & 15, lq = lane >> 4, swzl = lds_swz(l15);
    const bool works = wave * 16 < M;
    int cur = 0;
    for (int kt = 0; kt < KT; kt++) {
        /* stage `cur` has landed for this wave (the NS - 2 stages requested after it may still be on their way); after the barrier it has for all, and
         * everyone is done reading the stage before it, which is refilled */
        if (kt + NS - 2 < KT) {
            if (own == 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NS - 2) : "memory");
            else if (own == 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * (NS - 2)) : "memory");
            else if (own == 3) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(3 * (NS - 2)) : "memory");
            else if (own == 4) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(4 * (NS - 2)) : "memory");
            else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(5 * (NS - 2)) : "memory");
        } else {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        }
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        const int refill = cur == 0 ? NS - 1 : cur - 1;
        if (kt + NS - 1 < KT) issue(kt + NS - 1, refill);
        if (works) {
            const char *st = smem + cur * STAGE;
#pragma unroll
            for (int kk = 0; kk < 2; kk++) {
                const int coff = ((kk * 4 + lq) ^ swzl) << 4;
                const bf16x8 fa = *(const bf16x8 *)(st + (wave * 16 + l15) * 128 + coff);
                bf16x8 fb[TN];
#pragma unroll
                for (int i = 0; i < TN; i++) fb[i] = *(const bf16x8 *)(st + (BM + i * 16 + l15) * 128 + coff);
#pragma unroll
                for (int i = 0; i < TN; i++) acc[i][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[i], fa, acc[i][0], 0, 0, 0);
            }
        }
        cur = cur == NS - 1 ? 0 : cur + 1;
    }
    static_assert(CM <= 5 && NS >= 4, "a case for every count");
    if (works) store_tile<BN, 16, BN, EPI, 8>(g, t, acc, 0, M, wave, 0, l15, lq, t.tm * 8 + wave);
}

/* The large tiles: 4 waves (2 x 2), one per SIMD, each owning a (16 TM) x (16 TN) part of a
 * (32 TM) x (32 TN) tile, see the file comment. The MFMA is issued through inline asm so that the
 * accumulator stays in one AGPR quad for the whole loop (left to the register allocator,
 * accumulators migrate between VGPRs and AGPRs with hundreds of copies per K step). Statements with
 * side effects keep their program order, which is what places the LDS reads and global->LDS
 * loads between the MFMAs. */
#define MFMA_AGPR(acc, a, b) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b))
/* the first MFMA of an accumulator block: adds to zero instead of to the register's old contents */
#define MFMA_AGPR_NEW(acc, a, b) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=a"(acc) : "v"(a), "v"(b))

/* accumulators in VGPRs (gemm4x_kernel) */
#define MFMA_VGPR(acc, a, b) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(acc) : "v"(a), "v"(b))
#define MFMA_VGPR_NEW(acc, a, b) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=&v"(acc) : "v"(a), "v"(b))

/* The compiler neither sees those MFMAs' register hazards nor keeps plain register moves in order
 * around them. acc_fence passes every accumulator through an empty asm statement that is ordered
 * with the MFMAs: accumulator writes before it stay before it, reads after it stay after it.
 * Idle cycles for the hazards are placed explicitly next to it. */
template <int TM, int TN>
__device__ __forceinline__ void acc_fence(f32x4 (&acc)[TN][TM]) {
    static_assert(TN == 8 || TN == 7 || TN == 6 || TN == 5 || TN == 4, "one asm statement per accumulator column");
#pragma unroll
    for (int j = 0; j < TM; j++) {
        if constexpr (TN == 7)
            asm volatile("" : "+a"(acc[0][j]), "+a"(acc[1][j]), "+a"(acc[2][j]), "+a"(acc[3][j]),
                              "+a"(acc[4][j]), "+a"(acc[5][j]), "+a"(acc[6][j]));
        else if constexpr (TN == 8)
            asm volatile("" : "+a"(acc[0][j]), "+a"(acc[1][j]), "+a"(acc[2][j]), "+a"(acc[3][j]),
                              "+a"(acc[4][j]), "+a"(acc[5][j]), "+a"(acc[6][j]), "+a"(acc[7][j]));
        else if constexpr (TN == 6)
            asm volatile("" : "+a"(acc[0][j]), "+a"(acc[1][j]), "+a"(acc[2][j]), "+a"(acc[3][j]),
                              "+a"(acc[4][j]), "+a"(acc[5][j]));
        else if constexpr (TN == 5)
            asm volatile("" : "+a"(acc[0][j]), "+a"(acc[1][j]), "+a"(acc[2][j]), "+a"(acc[3][j]), "+a"(acc[4][j]));
        else
            asm volatile("" : "+a"(acc[0][j]), "+a"(acc[1][j]), "+a"(acc[2][j]), "+a"(acc[3][j]));
    }
}

/* whether a workgroup of gemm4w_kernel goes on to further tiles: the 4-wave form */
template <int WAVES> struct Walks4w { static constexpr bool value = WAVES == 4; };

template <int TM, int TN, int EPI, int WGM = 2, int WGN = 2>
__global__ __launch_bounds__(64 * WGM * WGN) void gemm4w_kernel(GemmArgs g) {
    constexpr int WM = 16 * TM, WN = 16 * TN, BM = WGM * WM, BN = WGN * WN;
    constexpr int RPP = 8 * WGM * WGN; /* tile rows one pass of the workgroup's loads covers: 8 per wave instruction */
    static_assert(BM % RPP == 0 && BN % RPP == 0, "tile rows must divide evenly over the waves' loads");
    constexpr int LA = BM / RPP, LB = BN / RPP;
    constexpr int NL = LA + LB;     /* global->LDS loads per wave and stage: 8 tile rows each */
    constexpr int NF = TM + TN;     /* fragments per K half-step: TN weight side, TM activation side */
    constexpr int NM = TM * TN;     /* MFMAs per K half-step */
    constexpr int RD = NM / NF;     /* one LDS read (and one load) every RD MFMAs */
    constexpr int STAGE = (BM + BN) * 128;
    static_assert((EPI != FLUX_HIP_EPI_SWIGLU && EPI != EPI_QKV_SWIGLU) || (TN % 2 == 0), "swiglu pairs 16-column blocks");
    static_assert(RD >= 2 && RD * (NF - 1) + 1 < NM, "reads and loads must fit between the MFMAs");
    extern __shared__ __attribute__((aligned(16))) char smem[];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WGN, wn = wave % WGN;
    const int lrow = tid >> 3, lchunk = tid & 7;
    const int l15 = lane & 15, lq = lane >> 4;
    const int swzl = lds_swz(l15);
    const int a_frag = (wm * WM + l15) * 128;
    const int b_frag = BM * 128 + (wn * WN + l15) * 128;
    const int coff0 = (lq ^ swzl) << 4, coff1 = ((4 + lq) ^ swzl) << 4;
    /* fragment q of a half-step: 0..TN-1 weight side (MFMA A operand), then activation side */
    auto frag = [&](const char *st, int coff, int q) -> bf16x8 {
        return q < TN ? *(const bf16x8 *)(st + b_frag + q * 2048 + coff) : *(const bf16x8 *)(st + a_frag + (q - TN) * 2048 + coff);
    };

    /* A launch has at most one workgroup per compute unit; each walks the tiles vb, vb + gridDim.x, ...
     * of the virtual grid, so that a tile's stores drain, and the next tile's first stage arrives,
     * while the matrix pipes already work again (with one workgroup per tile, the end of one and the
     * start of the next on a compute unit cost 5-14 us of a 60 us tile). */
    int vb = blockIdx.x;
    TileId t;
    if (!decode_tile<IsConv<EPI>::value>(g, vb, t)) return;

    /* Load i of a stage by this wave covers tile rows lrow + RPP i (8 rows of 128 bytes per wave
     * instruction): activation rows for i < LA, weight rows after. Rows RPP apart share a swizzle.
     * The K offset of this workgroup's slice is folded into the per-lane sources. */
    /* Sources are a uniform base per operand (tile's matrix + this workgroup's K slice + the K step, all scalar
     * arithmetic) plus a 32-bit byte offset per lane and load, so that stepping along K costs no vector work. */
    unsigned voff[NL];
    const char *baseA, *baseW;
    auto set_sources = [&](const TileId &tt) {
        const int M = g.M[tt.prob], m0 = tt.tml * BM;
        const int chunk = (lchunk ^ lds_swz(lrow)) << 3;
        baseA = (const char *)(g.A[tt.prob] + tt.ks * g.kt_per * 64);
        baseW = (const char *)(g.W[tt.prob] + tt.ks * g.kt_per * 64);
#pragma unroll
        for (int i = 0; i < LA; i++) voff[i] = ((unsigned)min(m0 + lrow + i * RPP, M - 1) * (unsigned)g.lda + chunk) * 2u;
#pragma unroll
        for (int i = 0; i < LB; i++) voff[LA + i] = ((unsigned)weight_row<BN, WN, EPI>(g, tt.tn, lrow + i * RPP) * (unsigned)g.ldw + chunk) * 2u;
    };
    auto issue1 = [&](int kt, int stage, int i) {
        const char *base = (i < LA ? baseA : baseW) + kt * 128;
        asm volatile("" : "+v"(voff[i])); /* keeps the load in its scalar base + 32-bit lane offset form, see gemm4d_kernel */
        __builtin_amdgcn_global_load_lds(GLOBAL_PTR(base + voff[i]), LDS_PTR(smem + stage * STAGE + (wave * 8 + i * RPP) * 128), 16, 0, 0);
    };
    set_sources(t);
#pragma unroll
    for (int i = 0; i < NL; i++) issue1(0, 0, i);

    for (;;) {
        const int kt_begin = t.ks * g.kt_per;
        const int KT = min(g.K >> 6, kt_begin + g.kt_per) - kt_begin;

        f32x4 acc[TN][TM];
#pragma unroll
        for (int i = 0; i < TN; i++)
#pragma unroll
            for (int j = 0; j < TM; j++)
#pragma unroll
                for (int e = 0; e < 4; e++) acc[i][j][e] = 0.0f;
        acc_fence<TM, TN>(acc); /* the zeroes are written, and a few cycles pass, before the first MFMA reads them */
        asm volatile("s_nop 7" ::: "memory");

        bf16x8 f0[NF], f1[NF];

        WAIT_VMCNT0();
        __syncthreads();
        if (KT > 1) {
#pragma unroll
            for (int i = 0; i < NL; i++) issue1(1, 1, i);
        }
#pragma unroll
        for (int q = 0; q < NF; q++) f0[q] = frag(smem, coff0, q);

        /* The blocks of a half-step are walked in serpentine order: exactly one MFMA operand changes from one
         * instruction to the next (the matrix pipes draw less power that way than when the weight fragment
         * wraps around together with a new activation fragment). */
        auto serp = [](int b) { return ((b / TN) & 1) ? TN - 1 - b % TN : b % TN; };
        auto step = [&](int kt, auto more_c, auto more2_c) {
            constexpr bool more = decltype(more_c)::value, more2 = decltype(more2_c)::value;
            auto &accr = acc;
            const int cur = kt & 1;
            const char *st = smem + cur * STAGE;
            const char *nx = smem + (cur ^ 1) * STAGE;
            /* first K half of the stage from f0, while the second half's fragments arrive in f1 */
#pragma unroll
            for (int b = 0; b < NM; b++) {
                MFMA_AGPR(accr[serp(b)][b / TN], f0[serp(b)], f0[TN + b / TN]);
                if (b % RD == 0 && b / RD < NF) f1[b / RD] = frag(st, coff1, b / RD);
            }
            if (more) {
                /* the next stage has landed for this wave; past the barrier it has for all, and
                 * everyone has finished reading this stage, which is refilled below */
                WAIT_VMCNT0();
                __syncthreads();
            }
            /* second half from f1, while the next stage's first fragments arrive in f0 and the stage
             * after next is requested; at most one other instruction between two MFMAs */
#pragma unroll
            for (int b = 0; b < NM; b++) {
                MFMA_AGPR(accr[serp(b)][b / TN], f1[serp(b)], f1[TN + b / TN]);
                if (more && b % RD == 0 && b / RD < NF) f0[b / RD] = frag(nx, coff0, b / RD);
                if (more2 && b % RD == 1 && b / RD < NL) issue1(kt + 2, cur, b / RD);
            }
        };
        int kt = 0;
        for (; kt < KT - 2; kt++) step(kt, BoolC<true>{}, BoolC<true>{});
        if (kt < KT - 1) {
            step(kt, BoolC<true>{}, BoolC<false>{});
            kt++;
        }
        step(kt, BoolC<false>{}, BoolC<false>{});

        /* The next tile's first stage is requested before this tile is stored: every wave has taken
         * its last fragments out of LDS once it is past this barrier. */
        const TileId done = t;
        vb += gridDim.x;
        const bool again = Walks4w<WGM * WGN>::value && vb < g.vgrid && decode_tile<IsConv<EPI>::value>(g, vb, t);
        if (again) {
            __syncthreads();
            set_sources(t);
#pragma unroll
            for (int i = 0; i < NL; i++) issue1(0, 0, i);
        }
        asm volatile("s_nop 15\n\ts_nop 15" ::: "memory"); /* the last MFMA results retire before they are read */
        acc_fence<TM, TN>(acc);

        /* The lane's position enters the epilogue through an empty asm statement: what the epilogue derives from it
         * (row and column offsets of every store, for the fused projection those of both store bodies) is then computed
         * per tile. Left visible, the compiler computes all of it once before the first tile and keeps it in registers
         * across the K loops, beyond what the register file holds beside the accumulators and fragments. */
        int l15e = l15, lqe = lq;
        asm volatile("" : "+v"(l15e), "+v"(lqe));
        store_tile<BN, WM, WN, EPI, WGM, true>(g, done, acc, done.tml * BM, g.M[done.prob], wm, wn, l15e, lqe, done.tm * WGM + wm);
        if (!again) break;
    }
}

/* The same tiles with deeper operand rings, for the transformer's epilogues. gemm4w_kernel holds two stages and
 * waits at its barrier for every load it has in flight (requested one to two half-steps earlier); operands that
 * come from HBM rather than from a cache arrive later than that now and then, and a wave that waits holds the
 * other three up at the barrier. Here the activation tile and the weight tile have rings of their own, NSA and NSW
 * slots of one K step (128-byte rows, the layout of gemm4w_kernel) each, as many as the 160 KB of LDS hold, and
 * the barrier waits with a count instead of a fence. The MFMA order is that of gemm4w_kernel: bit-identical results.
 *
 * Loads of a K step kt are spread over both of its halves (one load costs a lone wave 12 cycles of matrix-pipe
 * time at one load per eight MFMAs and 19 at one per four). The "first" operand - the one with three slots,
 * activations if both have three - is requested in the first half for step kt + 2, into the slot that step kt - 1
 * left at the last barrier; the "second" operand in the second half for step kt + NS2 (its ring's depth), into
 * the slot whose last reads completed at this step's barrier. The barrier in the middle of step kt needs step
 * kt + 1 in LDS: everything but the loads issued after it, which is a count (vector memory operations of a wave
 * complete in the order of their issue).
 *
 * Tiles follow each other without a gap in that pipeline: the last steps of a tile request the first steps of the
 * workgroup's next tile where they would request steps beyond their own K range, the last step reads the next
 * tile's first fragments, and the ring positions carry over. The finished tile is stored between the two K
 * loops, and nothing waits for those stores there: the first barrier of the next tile allows them (and the
 * loads behind them) to be in flight, the second one needs loads that were issued after them. Before that, a
 * tile began by waiting for every store of its predecessor to be acknowledged and for its own first steps,
 * requested only then, with the matrix pipes idle: 12 % of a 288 x 192 x 3072 tile's time. */
template <int EPI, int TM, int TN>
struct EpilogueOps { /* vector memory instructions a wave issues in the epilogue of a tile whose rows are all valid */
    static constexpr int value = EPI == FLUX_HIP_EPI_SWIGLU ? TM * (TN / 4 + TN / 2 % 2 + TN % 2) /* 16-byte stores + a last 8-byte and 4-byte one */
                                 : EPI == EPI_QKV_SWIGLU ? TM * (TN / 4 + TN / 2 % 2)
                                 : EPI == FLUX_HIP_EPI_BF16 || EPI == FLUX_HIP_EPI_CONV_BF16 || EPI == EPI_EXP ? TM * (TN / 2 + TN % 2) : EPI == FLUX_HIP_EPI_F32_T ? 4 * TM * TN : TM * TN;
};

template <int TM, int TN, int EPI, int NSA, int NSW>
__global__ __launch_bounds__(256) void gemm4d_kernel(GemmArgs g) {
    constexpr int WGM = 2, WGN = 2;
    constexpr int WM = 16 * TM, WN = 16 * TN, BM = WGM * WM, BN = WGN * WN;
    constexpr int RPP = 32; /* tile rows one pass of the workgroup's loads covers: 8 per wave instruction */
    static_assert(BM % RPP == 0 && BN % RPP == 0, "tile rows must divide evenly over the waves' loads");
    constexpr int LA = BM / RPP, LB = BN / RPP, NL = LA + LB;
    constexpr int NF = TM + TN, NM = TM * TN, RD = NM / NF;
    constexpr int ASZ = BM * 128, WSZ = BN * 128;
    static_assert((NSA == 2 || NSA == 3) && (NSW == 2 || NSW == 3) && (NSA == 3 || NSW == 3) && NSA * ASZ + NSW * WSZ <= 160 * 1024,
                  "rings of two or three slots within the LDS, one of them with three");
    static_assert((EPI != FLUX_HIP_EPI_SWIGLU && EPI != EPI_QKV_SWIGLU) || TN % 2 == 0 || (EPI == FLUX_HIP_EPI_SWIGLU && LaneCut<BN, WM>::value),
                  "swiglu pairs 16-column blocks");
    static_assert(RD >= 2 && RD * (NF - 1) + 1 < NM, "reads must fit between the MFMAs");
    constexpr bool FIRST_A = NSA == 3;
    constexpr int LF = FIRST_A ? LA : LB, LS = FIRST_A ? LB : LA, NS2 = FIRST_A ? NSW : NSA;
    constexpr int SF = (NM / LF) / RD * RD, SS = (NM / LS) / RD * RD; /* MFMAs between two loads of a half: a multiple of RD */
    static_assert(SF >= RD && SS >= RD && 1 + SF * (LF - 1) < NM && 1 + SS * (LS - 1) < NM, "the loads of a half fit between its MFMAs");
    constexpr int AHEAD = LF + (NS2 == 3 ? LS : 0); /* loads that may be in flight past the barrier */
    /* first barrier of a tile that follows another: also the stored tile's memory operations may be in flight (the wait
     * counter holds 63) */
    constexpr int AHEAD_STORES = AHEAD + EpilogueOps<EPI, TM, TN>::value < 63 ? AHEAD + EpilogueOps<EPI, TM, TN>::value : 63;
    extern __shared__ __attribute__((aligned(16))) char smem[];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6) & 3;
    const int wm = wave / WGN, wn = wave % WGN;
    const int lrow = tid >> 3, lchunk = tid & 7;
    const int l15 = lane & 15, lq = lane >> 4;
    const int swzl = lds_swz(l15);
    const int coff0 = (lq ^ swzl) << 4, coff1 = ((4 + lq) ^ swzl) << 4;
    const unsigned a_frag = (wm * WM + l15) * 128, w_frag = NSA * ASZ + (wn * WN + l15) * 128;

    int vb = blockIdx.x;
    TileId t;
    if (!decode_tile<IsConv<EPI>::value>(g, vb, t)) return;

    /* Sources of a tile's loads: a uniform base per operand (the tile's matrix + this workgroup's K slice) and a 32-bit
     * byte offset per lane and load, so that stepping along K is scalar work. Two sets: the tile being multiplied and
     * the workgroup's next one. */
    struct Src {
        unsigned voff[NL];
        const char *baseA, *baseW;
        int k0; /* convolutions: the first K step of the slice (the rows' offset is a function of the absolute step) */
    };
    Src cur, nxt;
    auto set_sources = [&](Src &sc, const TileId &tt) {
        const int M = g.M[tt.prob], m0 = tt.tml * BM;
        /* the lane's row enters through an empty asm statement, so that the per-load row numbers derived from it (two
         * sets of weight rows for the fused projection) are computed here, per tile, and not once before the first
         * tile, from where they would have to be kept in registers across every K loop */
        int lr = lrow;
        asm volatile("" : "+v"(lr));
        const int chunk = (lchunk ^ lds_swz(lr)) << 3;
        sc.k0 = IsConv<EPI>::value ? tt.ks * g.kt_per : 0;
        sc.baseA = (const char *)(g.A[tt.prob] + (IsConv<EPI>::value ? 0 : tt.ks * g.kt_per * 64));
        sc.baseW = (const char *)(g.W[tt.prob] + tt.ks * g.kt_per * 64);
#pragma unroll
        for (int i = 0; i < LA; i++) sc.voff[i] = ((unsigned)conv_in_row<EPI>(g, min(m0 + lr + i * RPP, M - 1)) * (unsigned)g.lda + chunk) * 2u;
#pragma unroll
        for (int i = 0; i < LB; i++) sc.voff[LA + i] = ((unsigned)weight_row<BN, WN, EPI>(g, tt.tn, lr + i * RPP) * (unsigned)g.ldw + chunk) * 2u;
    };
    /* where K step kt of an operand starts */
    auto step_a = [&](const Src &sc, int kt) { return sc.baseA + (IsConv<EPI>::value ? (ptrdiff_t)a_step_offset<EPI>(g, sc.k0 + kt) * 2 : (ptrdiff_t)kt * 128); };
    auto step_w = [&](const Src &sc, int kt) { return sc.baseW + (ptrdiff_t)kt * 128; };
    /* load i of the K step that starts at base: activation rows for i < LA (into slot sa
     * of their ring), weight rows after (slot sw). The offset passes through an empty asm statement where it is used: the
     * load is then selected in its "scalar base + 32-bit lane offset" form. Without it the compiler widens every offset
     * to 64 bits once, outside the K loop, keeps NL register pairs instead of NL registers, and adds the base with a
     * 64-bit vector addition in front of every load. */
    auto issue1 = [&](const char *base, unsigned &vo, int sa, int sw, int i) {
        const int dst = i < LA ? sa * ASZ + (wave * 8 + i * RPP) * 128 : NSA * ASZ + sw * WSZ + (wave * 8 + (i - LA) * RPP) * 128;
        asm volatile("" : "+v"(vo));
        __builtin_amdgcn_global_load_lds(GLOBAL_PTR(base + vo), LDS_PTR(smem + dst), 16, 0, 0);
    };
    auto k_steps = [&](const TileId &tt) { return min(g.K >> 6, tt.ks * g.kt_per + g.kt_per) - tt.ks * g.kt_per; };
    /* The first K steps of a tile that no predecessor requested, into slots 0, 1 (and 2): what the pipeline below has
     * in flight when it enters a tile's step 0, oldest first */
    auto prime = [&](Src &sc, int KTn) {
#pragma unroll
        for (int s = 0; s < 2; s++) {
            if (s < KTn) {
#pragma unroll
                for (int i = 0; i < NL; i++) issue1(i < LA ? step_a(sc, s) : step_w(sc, s), sc.voff[i], s, s, i);
            }
        }
        if (NS2 == 3 && KTn > 2) {
#pragma unroll
            for (int n = 0; n < LS; n++) issue1(FIRST_A ? step_w(sc, 2) : step_a(sc, 2), sc.voff[(FIRST_A ? LA : 0) + n], 2, 2, (FIRST_A ? LA : 0) + n);
        }
    };

    bf16x8 f0[NF], f1[NF];
    int ca = 0, cw = 0;                   /* ring slots of the step being multiplied */
    unsigned va = a_frag, vw = w_frag;    /* this lane's fragment rows in those slots */
    auto frag = [&](unsigned xa, unsigned xw, int coff, int q) -> bf16x8 {
        return q < TN ? *(const bf16x8 *)(smem + xw + coff + q * 2048) : *(const bf16x8 *)(smem + xa + coff + (q - TN) * 2048);
    };
    /* the first tile: its first steps are requested here, and its step 0 starts when that one has landed (a compute unit takes in 50 KB of cold
     * operands a microsecond: the other steps of the rings, 64 to 100 KB, are 1.3 to 2 us of every launch) */
    set_sources(cur, t);
    prime(cur, k_steps(t));
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(NL + (NS2 == 3 ? LS : 0)) : "memory");
#pragma unroll
    for (int q = 0; q < NF; q++) f0[q] = frag(va, vw, coff0, q);
    bool strict = true; /* the first barrier of the tile must not count on the operations of a stored tile */

    for (;;) {
        const int KT = k_steps(t); /* at least 4: the host sends shorter K ranges to gemm4w_kernel */

        f32x4 acc[TN][TM]; /* started by the MFMAs of step 0's first half (no pass over 4 TM TN registers to clear them) */

        auto serp = [](int b) { return ((b / TN) & 1) ? TN - 1 - b % TN : b % TN; };
        /* TAIL = false: steps kt + 1 .. kt + 3 belong to this tile. TAIL = true: one of the last three steps of a tile;
         * loads for steps beyond its K range request the first steps of the tile in nxt instead (every load is issued,
         * so the wait counts stay exact). WAIT: what may be in flight at the barrier. */
        auto step = [&](int kt, auto tail_c, auto wait_c, auto first_c) {
            constexpr bool TAIL = decltype(tail_c)::value;
            constexpr int WAIT = decltype(wait_c)::value;
            constexpr bool FIRST = decltype(first_c)::value; /* step 0: its first half starts the accumulators */
            auto &accr = acc;
            const int na = ca == NSA - 1 ? 0 : ca + 1, nw = cw == NSW - 1 ? 0 : cw + 1;
            const unsigned van = a_frag + na * ASZ, vwn = w_frag + nw * WSZ;
            const auto start = [&](int ks, bool a) {
                const bool over = TAIL && ks >= KT;
                const Src &sc = over ? nxt : cur;
                return a ? step_a(sc, over ? ks - KT : ks) : step_w(sc, over ? ks - KT : ks);
            };
            /* A convolution's offset of a K step is a dozen scalar instructions, so the bases of the two K steps requested in
             * this one are formed once. A projection forms the base at each load, from one byte offset for both operands:
             * bases carried across the halves and an offset for each operand were four more scalar instructions per step. */
            const char *first = nullptr, *second = nullptr;
            if constexpr (IsConv<EPI>::value) first = start(kt + 2, FIRST_A), second = start(kt + NS2, !FIRST_A);
            auto load = [&](const char *formed, int ks, int sa, int sw, int i) {
                const char *base = IsConv<EPI>::value ? formed : start(ks, i < LA);
                if (!TAIL) {
                    issue1(base, cur.voff[i], sa, sw, i);
                } else {
                    unsigned vo = ks >= KT ? nxt.voff[i] : cur.voff[i];
                    issue1(base, vo, sa, sw, i);
                }
            };
#pragma unroll
            for (int b = 0; b < NM; b++) {
                if (FIRST) MFMA_AGPR_NEW(accr[serp(b)][b / TN], f0[serp(b)], f0[TN + b / TN]);
                else MFMA_AGPR(accr[serp(b)][b / TN], f0[serp(b)], f0[TN + b / TN]);
                if (b % RD == 0 && b / RD < NF) f1[b / RD] = frag(va, vw, coff1, b / RD);
                /* step kt + 2 of the first operand, into the slot that step kt - 1 left */
                if (b % SF == 1 && b / SF < LF) load(first, kt + 2, ca == 0 ? 2 : ca - 1, cw == 0 ? 2 : cw - 1, (FIRST_A ? 0 : LA) + b / SF);
            }
            /* step kt + 1 has landed for this wave and its reads of step kt are complete; past the barrier both hold
             * for all */
            if (FIRST && strict) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(AHEAD) : "memory");
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(WAIT) : "memory");
#pragma unroll
            for (int b = 0; b < NM; b++) {
                MFMA_AGPR(accr[serp(b)][b / TN], f1[serp(b)], f1[TN + b / TN]);
                if (b % RD == 0 && b / RD < NF) f0[b / RD] = frag(van, vwn, coff0, b / RD);
                /* step kt + NS2 of the second operand, into the slot of step kt */
                if (b % SS == 1 && b / SS < LS) load(second, kt + NS2, ca, cw, (FIRST_A ? LA : 0) + b / SS);
            }
            ca = na;
            cw = nw;
            va = van;
            vw = vwn;
        };
        /* step 0: the stored tile's memory operations are older than anything its barrier needs */
        step(0, BoolC<false>{}, IntC<AHEAD_STORES>{}, BoolC<true>{});
        int kt = 1;
        for (; kt < KT - 3; kt++) step(kt, BoolC<false>{}, IntC<AHEAD>{}, BoolC<false>{});

        /* the workgroup's next tile: its first steps are requested by this tile's last ones. After the last tile they
         * request this tile's first steps once more, into slots that nobody reads again. */
        const TileId done = t;
        vb += gridDim.x;
        bool again;
        if constexpr (IsConv<EPI>::value) {
            const GemmArgs gd = conv_args_again();
            again = vb < gd.vgrid && decode_tile<true>(gd, vb, t);
        } else {
            again = vb < g.vgrid && decode_tile<IsConv<EPI>::value>(g, vb, t);
        }
        if (again) set_sources(nxt, t);
        else nxt = cur;
        for (; kt < KT; kt++) step(kt, BoolC<true>{}, IntC<AHEAD>{}, BoolC<false>{});

        asm volatile("s_nop 15\n\ts_nop 15" ::: "memory"); /* the last MFMA results retire before they are read */
        acc_fence<TM, TN>(acc);

        /* The lane's position enters the epilogue through an empty asm statement: what the epilogue derives from it
         * (row and column offsets of every store, for the fused projection those of both store bodies) is then computed
         * per tile. Left visible, the compiler computes all of it once before the first tile and keeps it in registers
         * across the K loops, beyond what the register file holds beside the accumulators and fragments. */
        int l15e = l15, lqe = lq;
        asm volatile("" : "+v"(l15e), "+v"(lqe));
        if constexpr (EPI == FLUX_HIP_EPI_CONV_BF16 || EPI == FLUX_HIP_EPI_CONV_F32) {
            const GemmArgs ge = conv_args_again();
            store_tile<BN, WM, WN, EPI, WGM, true>(ge, done, acc, done.tml * BM, ge.M[0], wm, wn, l15e, lqe, done.tm * WGM + wm);
        } else {
            store_tile<BN, WM, WN, EPI, WGM, true>(g, done, acc, done.tml * BM, g.M[done.prob], wm, wn, l15e, lqe, done.tm * WGM + wm);
        }
        if (!again) break;
        /* not every row of this wave's part of the stored tile was valid, or not every column: it issued fewer than
         * EpilogueOps operations */
        strict = done.tml * BM + wm * WM + WM > g.M[done.prob] || (CutTile<BN>::value && done.tn == g.ntiles - 1);
        cur = nxt;
    }
    /* the requests made in place of a next tile's land in this workgroup's LDS: not after it has gone */
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

/* Tiles with more accumulators than the 256 AGPRs hold (288 x 288, 384 x 224, 320 x 256 and the like; 16 x 16 blocks beyond the 64th
 * accumulate in VGPRs), for the fused projection of a single-stream block. What bounds the 4-wave tiles beside the matrix
 * pipes is LDS traffic and the issue of loads, both a matter of a wave tile's circumference: 144 x 144 takes 0.222 fragment reads and
 * 0.111 global->LDS loads per MFMA, 144 x 96 0.278 and 0.139; and more sizes leave fewer units idle in the last round (768 x 27648 is 432 tiles
 * of 256 x 192, two rounds, and 250 of 384 x 224, one). K = 3072 and N = 27648 with the weights from HBM, us, the best tile of up to 256
 * registers and this kernel's: 600 rows 108 -> 83, 768 109 -> 94, 1202 168 -> 159, 1536 194 -> 175, 2304 273 -> 260, 2560 324 -> 299,
 * 4608 544 -> 518 (1512 TFLOP/s), 5120 601 -> 576, 10000 1179 -> 1133, 13056 1525 -> 1497. What pays for the registers and the LDS (two slots
 * of one K step per operand):
 * activation fragments of the next half-step are read into the registers that this one has done with, a row of blocks behind the
 * MFMAs (the last SP rows, whose reads the barrier would have to wait for, have spare ones; the weights are double-buffered);
 * and with two slots for both operands the loads of a tile's last two steps all belong to the next tile, so that one set of source
 * offsets is enough.
 *
 * Step kt: half 0 multiplies (kt, first 32 of K) and reads (kt, second 32), weights first. Once all waves have read the weights (a
 * barrier behind LW MFMAs) their slot takes those of step kt + 2. At the barrier between the halves the same holds for the
 * activations, which follow in half 1, and step kt + 1 has landed: everything but the weights of step kt + 2. Reading the weights
 * two, three or four MFMAs apart and the barrier six or twelve behind them measured the same within 1 %. */
template <int TM, int TN, int SP, int RW, int RA>
struct WideReads { /* which fragment is read behind MFMA b of a half-step: of[b], or -1 */
    static constexpr int NF = TM + TN;
    signed char of[TM * TN];
    static constexpr int at(int q) {
        const int b = q < TN ? RW * q : RW * TN + RA * (q - TN), row = q - TN - SP;
        return row < 0 || b >= (row + 1) * TN ? b : (row + 1) * TN;
    }
    constexpr WideReads() : of() {
        for (int b = 0; b < TM * TN; b++) of[b] = -1;
        for (int q = 0; q < NF; q++) of[at(q)] = (signed char)q;
    }
    static constexpr int issued(int first, int b) {
        int n = 0;
        for (int q = first; q < NF; q++) n += at(q) <= b;
        return n;
    }
    static constexpr bool in_order() {
        for (int q = 1; q < NF; q++)
            if (at(q) <= at(q - 1)) return false;
        return true;
    }
};

template <int TM, int TN, int EPI>
__global__ __launch_bounds__(256) void gemm4x_kernel(GemmArgs g) {
    constexpr int WGM = 2, WGN = 2;
    constexpr int WM = 16 * TM, WN = 16 * TN, BM = WGM * WM, BN = WGN * WN;
    constexpr int RPP = 32;
    constexpr int LA = BM / RPP, LB = BN / RPP, NL = LA + LB;
    constexpr int NF = TM + TN, NM = TM * TN;
    constexpr int ASZ = BM * 128, WSZ = BN * 128;
    static_assert(2 * (ASZ + WSZ) <= 160 * 1024 && NM > 64 && IsWide<BN, WM>::value, "two slots per operand");
    constexpr int SP = 2;                       /* activation rows with spare registers */
    constexpr int AGPR_BLOCKS = 64;
    /* the MFMA behind which fragment q is read: weights, the last SP activation rows, the other activation rows, each when its MFMAs of
     * this half have been issued */
    constexpr int RW = 2, RA = (NM - 8 - RW * TN) / TM;
    constexpr int LW = RW * (TN - 1) + 6;   /* MFMAs in front of the barrier that frees the weights' slot */
    constexpr WideReads<TM, TN, SP, RW, RA> reads;
    constexpr int LATE = reads.issued(TN, LW - 1); /* reads behind the weights' by then */
    static_assert(RA >= 2 && reads.at(NF - 1) + 6 <= NM && reads.in_order(), "reads in order between the MFMAs, done before the barrier");
    constexpr int SW = (NM - LW) / LB, SA = NM / LA;
    static_assert(SW >= 2 && SA >= 2, "the loads of a half fit between its MFMAs");
    constexpr int E = EpilogueOps<EPI, TM, TN>::value;
    constexpr int AHEAD = LB, AHEAD_STORES = LB + E < 63 ? LB + E : 63;
    extern __shared__ __attribute__((aligned(16))) char smem[];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6) & 3;
    const int wm = wave / WGN, wn = wave % WGN;
    const int lrow = tid >> 3, lchunk = tid & 7;
    const int l15 = lane & 15, lq = lane >> 4;
    const int swzl = lds_swz(l15);
    const unsigned coff0 = (lq ^ swzl) << 4, coff1 = ((4 + lq) ^ swzl) << 4;
    const unsigned a_frag = (wm * WM + l15) * 128, w_frag = 2 * ASZ + (wn * WN + l15) * 128;

    int vb = blockIdx.x;
    TileId t;
    if (!decode_tile<false>(g, vb, t)) return;

    unsigned voff[NL];
    const char *baseA, *baseW;
    auto set_sources = [&](const TileId &tt) {
        const int M = g.M[tt.prob], m0 = tt.tml * BM;
        int lr = lrow;
        asm volatile("" : "+v"(lr));
        const int chunk = (lchunk ^ lds_swz(lr)) << 3;
        baseA = (const char *)g.A[tt.prob];
        baseW = (const char *)g.W[tt.prob];
#pragma unroll
        for (int i = 0; i < LA; i++) voff[i] = ((unsigned)min(m0 + lr + i * RPP, M - 1) * (unsigned)g.lda + chunk) * 2u;
#pragma unroll
        for (int i = 0; i < LB; i++) voff[LA + i] = ((unsigned)weight_row<BN, WN, EPI>(g, tt.tn, lr + i * RPP) * (unsigned)g.ldw + chunk) * 2u;
    };
    auto issue1 = [&](int ks, int slot, int i) { /* load i of K step ks: activation rows, then weight rows */
        const char *base = (i < LA ? baseA : baseW) + (ptrdiff_t)ks * 128;
        const int dst = i < LA ? slot * ASZ + (wave * 8 + i * RPP) * 128 : 2 * ASZ + slot * WSZ + (wave * 8 + (i - LA) * RPP) * 128;
        asm volatile("" : "+v"(voff[i]));
        __builtin_amdgcn_global_load_lds(GLOBAL_PTR(base + voff[i]), LDS_PTR(smem + dst), 16, 0, 0);
    };
    const int KT = g.K >> 6; /* at least 4 */

    bf16x8 w0[TN], w1[TN], fa[TM];
    f32x4 acc[TN][TM];
    int slot = 0;
    set_sources(t);
#pragma unroll
    for (int s = 0; s < 2; s++)
#pragma unroll
        for (int i = 0; i < NL; i++) issue1(s, s, i);
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(NL) : "memory"); /* step 0 has landed, as in gemm4d_kernel */
#pragma unroll
    for (int i = 0; i < TN; i++) w0[i] = *(const bf16x8 *)(smem + w_frag + coff0 + i * 2048);
#pragma unroll
    for (int j = 0; j < TM; j++) fa[j] = *(const bf16x8 *)(smem + a_frag + coff0 + j * 2048);
    bool strict = true;

    for (;;) {
        auto serp = [](int b) { return ((b / TN) & 1) ? TN - 1 - b % TN : b % TN; };
        /* a half-step: MFMAs of the fragments held, reads of the next half's from the rows at xa, xw, and `between` at every MFMA */
        auto half = [&](bf16x8 (&w)[TN], bf16x8 (&wn_)[TN], unsigned xa, unsigned xw, auto new_c, auto between) {
            bf16x8 sp[SP];
#pragma unroll
            for (int b = 0; b < NM; b++) {
                const int j = b / TN, i = serp(b);
                if (decltype(new_c)::value) {
                    if (b < AGPR_BLOCKS) MFMA_AGPR_NEW(acc[i][j], w[i], fa[j]);
                    else MFMA_VGPR_NEW(acc[i][j], w[i], fa[j]);
                } else {
                    if (b < AGPR_BLOCKS) MFMA_AGPR(acc[i][j], w[i], fa[j]);
                    else MFMA_VGPR(acc[i][j], w[i], fa[j]);
                }
                const int q = reads.of[b];
                if (q >= 0) {
                    if (q < TN) wn_[q] = *(const bf16x8 *)(smem + xw + q * 2048);
                    else if (q < TN + SP) sp[q - TN] = *(const bf16x8 *)(smem + xa + (TM - SP + q - TN) * 2048);
                    else fa[q - TN - SP] = *(const bf16x8 *)(smem + xa + (q - TN - SP) * 2048);
                }
                between(b);
            }
#pragma unroll
            for (int k = 0; k < SP; k++) fa[TM - SP + k] = sp[k];
        };
        /* ks: the K step that is requested, of the tile that voff and the bases belong to */
        auto step = [&](int ks, auto wait_c, auto first_c) {
            constexpr int WAIT = decltype(wait_c)::value;
            constexpr bool FIRST = decltype(first_c)::value;
            half(w0, w1, a_frag + slot * ASZ + coff1, w_frag + slot * WSZ + coff1, first_c, [&](int b) {
                if (b == LW - 1) asm volatile("s_waitcnt lgkmcnt(%0)\n\ts_barrier" ::"n"(LATE) : "memory"); /* all have their weights of this step */
                if (b >= LW && (b - LW) % SW == 0 && (b - LW) / SW < LB) issue1(ks, slot, LA + (b - LW) / SW);
            });
            if (FIRST && strict) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(AHEAD) : "memory");
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(WAIT) : "memory");
            const int ns = slot ^ 1;
            half(w1, w0, a_frag + ns * ASZ + coff0, w_frag + ns * WSZ + coff0, BoolC<false>{}, [&](int b) {
                if (b % SA == 1 && b / SA < LA) issue1(ks, slot, b / SA);
            });
            slot = ns;
        };
        step(2, IntC<AHEAD_STORES>{}, BoolC<true>{});
        for (int kt = 1; kt < KT - 2; kt++) step(kt + 2, IntC<AHEAD>{}, BoolC<false>{});
        /* the last two steps request the first two of the workgroup's next tile; after the last tile this tile's once more,
         * into slots that nobody reads again */
        const TileId done = t;
        vb += gridDim.x;
        const bool again = vb < g.vgrid && decode_tile<false>(g, vb, t);
        if (again) set_sources(t);
#pragma clang loop unroll(disable)
        for (int kt = 0; kt < 2; kt++) step(kt, IntC<AHEAD>{}, BoolC<false>{});

        asm volatile("s_nop 15\n\ts_nop 15" ::: "memory"); /* the last MFMA results retire before they are read */
#pragma unroll
        for (int b = 0; b < NM; b++) {
            if (b < AGPR_BLOCKS) asm volatile("" : "+a"(acc[serp(b)][b / TN]));
            else asm volatile("" : "+v"(acc[serp(b)][b / TN]));
        }
        int l15e = l15, lqe = lq;
        asm volatile("" : "+v"(l15e), "+v"(lqe));
        store_tile<BN, WM, WN, EPI, WGM, true>(g, done, acc, done.tml * BM, g.M[done.prob], wm, wn, l15e, lqe, done.tm * WGM + wm);
        if (!again) break;
        strict = done.tml * BM + wm * WM + WM > g.M[done.prob] || (CutTile<BN>::value && (done.tn == g.ntiles - 1 || done.tn == g.nq_tiles - 1));
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

/* 3x3 convolutions of images with too few 16 x 16 tiles for conv.hip's kernel: 128 positions x 64 channels per workgroup.
 * As a GEMM (the ring kernel's 128 x 128 tile) every K step fetches its 128 positions x 64 channels again, nine times what a chunk of channels
 * holds, and images this small need three to eight K slices with a second pass to give every compute unit work. This tile is half as wide: two to four
 * slices up to some 40 x 40 x 512, one piece beyond. Here the positions that a tile's nine taps touch
 * lie in LDS for a whole chunk (those of the next chunk arrive meanwhile), and the ring holds the weights alone: 11 to 14 KB a step.
 *
 * GEMM rows are interior positions in row-major order, so a tile is a run of positions whatever the image's sides. Its neighbourhood is one run
 * of the bordered image, from a row above the first position to a row below the last one, as long as that is at most 448 positions, and
 * otherwise (images wider than 156) three runs, one per tap row, CONVP_BAND apart in LDS: the LDS row of position p's tap (dy, dx) is
 * p - (the tile's first position) + dy * pitch + dx either way, pitch being the image's or CONVP_BAND. NPL: loads of eight LDS rows per wave
 * and chunk, 28, 40 or 56 KB twice; the weights have the rest.
 *
 * Four waves of 64 x 32 would read 1.5 times as many bytes of fragments as the LDS delivers during their MFMAs. So two waves share 64 x 64 and split
 * the K step, 32 channels each (32 KB of fragments for 256 cycles); their sums meet in LDS at the end. A step is one phase: its fragments are in
 * registers when it begins, those of the next one are read behind its first MFMAs, and the barrier in front of it waits for the weights of the next
 * step and leaves the slot of its own to those of SLOTS steps on.
 *
 * Alone, operands from the memory-side cache, bf16, us, against the best of the other tiles: 16 x 16 x 512 -> 512 15.9 -> 13.6 (four slices), 32 x 32 x 512 22.4 -> 16.3
 * (two), 42 x 42 x 512 24.2 -> 16.4, 64 x 64 x 512 29.3 -> 20.2 (two slices before), 84 x 84 x 512 -> 256 29.3 -> 18.4, 64 x 64 x 256 20.6 -> 11.2,
 * 128 x 128 x 128 13.8 -> 9.9. What bounds it: a unit takes in 12 KB of a step in 0.175 us, 70 KB a microsecond, which is 256 lines on their way
 * (loads return in order) at the memory-side cache's latency; the MFMAs are 0.11 us of it. 128 channels a tile (with and without the split of K) was 5 %
 * faster than the ring kernel's 128 x 128 where that has a round of tiles, which was not worth a second kernel. */
#define CONVP_BAND 144
template <int NPL> struct ConvP {
    static constexpr int PP = 3, LW = 2; /* a step's patch loads at most, and weight loads, of a wave */
    static constexpr int PATCH = NPL * 4096, WSZ = 64 * 128, LAST_TAP = (NPL + PP - 1) / PP - 1, ROOM = (160 * 1024 - 2 * PATCH) / WSZ;
    static constexpr int SLOTS = ROOM < 9 - LAST_TAP ? ROOM : 9 - LAST_TAP; /* the last patch load of a chunk is older than the weights that the next chunk waits for */
    static constexpr int LDS = 2 * PATCH + SLOTS * WSZ;
    static constexpr int patch_loads(int tap) { return tap < 0 || PP * tap >= NPL ? 0 : NPL - PP * tap < PP ? NPL - PP * tap : PP; }
    /* memory operations that a wave has issued, when it reaches the barrier in front of a tap, behind the weights of the tap after it: what
     * the steps since have requested, patch loads first (a chunk's last steps request none) */
    static constexpr int pending(int tap, bool last) {
        int n = LW * (last && 7 - tap < SLOTS - 2 ? 7 - tap : SLOTS - 2);
        for (int k = 1; k <= SLOTS - 2; k++) n += last ? 0 : patch_loads(tap - k);
        return n;
    }
    static_assert(SLOTS >= 3 && LDS <= 160 * 1024, "rings");
};

template <int NPL, int EPI>
__global__ __launch_bounds__(256) void convp_kernel(GemmArgs g) {
    using C = ConvP<NPL>;
    constexpr int BN = 64, TM = 4, TN = 4, NM = TM * TN, NF = TM + TN, SLOTS = C::SLOTS, W0 = 2 * C::PATCH;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6) & 3, kh = wave >> 1, half = wave & 1; /* half of the K step, half of the positions */
    const int l15 = lane & 15, lq = lane >> 4;
    TileId t;
    if (!decode_tile<true>(g, blockIdx.x, t)) return;
    const int M = g.M[0], m0 = t.tm * 128, wp = g.conv_wp;
    const int first = conv_row<FLUX_HIP_EPI_CONV_F32>(g, m0), last_pos = conv_row<FLUX_HIP_EPI_CONV_F32>(g, min(m0 + 127, M - 1));
    const int span = last_pos - first + 3;                      /* of a tap row's run */
    const bool bands = span + 2 * wp > NPL * 32;                /* (the host has made sure of 3 * CONVP_BAND <= 32 NPL then) */
    const int pitch = bands ? CONVP_BAND : wp;
    const int c0 = t.ks * (g.kt_per / 9), c1 = min(g.lda >> 6, c0 + g.kt_per / 9);

    unsigned prel[NPL], wrel[C::LW]; /* byte offsets of this lane's loads: positions (LDS row r), weights */
#pragma unroll
    for (int j = 0; j < NPL; j++) {
        const int r = 8 * (4 * j + wave) + (lane >> 3);
        const int b = r >= 2 * CONVP_BAND ? 2 : r >= CONVP_BAND ? 1 : 0;
        const int p = bands ? first + (b - 1) * wp - 1 + min(r - b * CONVP_BAND, span - 1) : first - wp - 1 + min(r, span + 2 * wp - 1);
        prel[j] = ((unsigned)p * (unsigned)g.lda + (((lane & 7) ^ lds_swz(r)) << 3)) * 2u;
    }
#pragma unroll
    for (int i = 0; i < C::LW; i++) {
        const int v = 8 * (4 * i + wave) + (lane >> 3);
        wrel[i] = ((unsigned)weight_row<BN, BN / 2, EPI>(g, t.tn, v) * (unsigned)g.ldw + (((lane & 7) ^ lds_swz(v)) << 3)) * 2u;
    }
    auto load_patch = [&](int chunk, int to, int j) {
        asm volatile("" : "+v"(prel[j]));
        __builtin_amdgcn_global_load_lds(GLOBAL_PTR((const char *)g.A[0] + chunk * 128 + prel[j]), LDS_PTR(smem + to + (4 * j + wave) * 1024), 16, 0, 0);
    };
    auto load_w = [&](int kt, int slot, int i) {
        asm volatile("" : "+v"(wrel[i]));
        __builtin_amdgcn_global_load_lds(GLOBAL_PTR((const char *)g.W[0] + (ptrdiff_t)kt * 128 + wrel[i]), LDS_PTR(smem + W0 + slot * C::WSZ + (4 * i + wave) * 1024), 16, 0, 0);
    };
    int kt = 9 * c0, slot = 0, to = C::PATCH; /* K step at work, its slot; where the next chunk's patch goes */
#pragma unroll
    for (int j = 0; j < NPL; j++) load_patch(c0, 0, j);
#pragma unroll
    for (int s = 0; s < SLOTS; s++)
#pragma unroll
        for (int i = 0; i < C::LW; i++) load_w(kt + s, s, i);

    unsigned pa[9][TM]; /* this lane's fragment addresses in the patch at work: a block's positions under each tap */
#pragma unroll
    for (int j = 0; j < TM; j++) {
        const int rel = conv_row<FLUX_HIP_EPI_CONV_F32>(g, min(m0 + half * 64 + j * 16 + l15, M - 1)) - first;
#pragma unroll
        for (int tap = 0; tap < 9; tap++) {
            const int r = rel + tap / 3 * pitch + tap % 3;
            pa[tap][j] = r * 128 + (((kh * 4 + lq) ^ lds_swz(r)) << 4);
        }
    }
    const unsigned wa = W0 + l15 * 128 + (((kh * 4 + lq) ^ lds_swz(l15)) << 4);
    auto frag = [&](int tap, int ws, int q) -> bf16x8 {
        return q < TN ? *(const bf16x8 *)(smem + wa + ws * C::WSZ + q * 2048) : *(const bf16x8 *)(smem + pa[tap][q - TN]);
    };

    /* Block (i, j) accumulates in a[4 (i TM + j)], by name (left to allocate them the compiler moves all accumulators at the joins of the paths
     * below); the compiler uses no AGPR (the tests look at its output for that) */
    asm volatile("" ::: "a255");
#pragma unroll
    for (int n = 0; n < 4 * NM; n++) asm volatile("v_accvgpr_write_b32 a[%0], 0" ::"i"(n));
    asm volatile("s_nop 7" ::: "memory");

    bf16x8 f[2][NF];
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(C::LW * (SLOTS - 1)) : "memory"); /* the patch and the first tap's weights */
#pragma unroll
    for (int q = 0; q < NF; q++) f[0][q] = frag(0, 0, q);

    auto serp = [](int b) { return ((b / TN) & 1) ? TN - 1 - b % TN : b % TN; };
    auto step = [&](int chunk, auto tap_c, auto last_c, auto set_c) {
        constexpr int TAP = decltype(tap_c)::value, SET = decltype(set_c)::value; /* the fragments' register set */
        constexpr bool LAST = decltype(last_c)::value, END = LAST && TAP == 8;    /* the slice's last chunk, and its last step */
        const int next = slot == SLOTS - 1 ? 0 : slot + 1;
        if (!END) { /* the next step's weights (and patch) have landed, and this step's have been read */
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(C::pending(TAP, LAST)) : "memory");
            if (TAP == 8) {
                const unsigned d = to - (C::PATCH - to);
#pragma unroll
                for (int k = 0; k < 9 * TM; k++) pa[k / TM][k % TM] += d;
                to = C::PATCH - to;
            }
        }
#pragma unroll
        for (int b = 0; b < NM; b++) {
            asm volatile("v_mfma_f32_16x16x32_bf16 a[%2:%3], %0, %1, a[%2:%3]" ::"v"(f[SET][serp(b)]), "v"(f[SET][TN + b / TN]),
                         "i"(4 * (serp(b) * TM + b / TN)), "i"(4 * (serp(b) * TM + b / TN) + 3));
            if (!END && b < NF) f[SET ^ 1][b] = frag((TAP + 1) % 9, next, b);
            if (!LAST && b >= NF && b - NF < C::patch_loads(TAP)) load_patch(chunk + 1, to, C::PP * TAP + b - NF);
            if ((!LAST || TAP + SLOTS <= 8) && b >= 12 && b % 2 == 0 && (b - 12) / 2 < C::LW) load_w(kt + SLOTS, slot, (b - 12) / 2);
        }
        slot = next;
        kt++;
    };
    auto taps = [&](int chunk, auto last_c, auto set_c) {
        constexpr int S = decltype(set_c)::value;
        step(chunk, IntC<0>{}, last_c, IntC<S>{}); step(chunk, IntC<1>{}, last_c, IntC<S ^ 1>{}); step(chunk, IntC<2>{}, last_c, IntC<S>{});
        step(chunk, IntC<3>{}, last_c, IntC<S ^ 1>{}); step(chunk, IntC<4>{}, last_c, IntC<S>{}); step(chunk, IntC<5>{}, last_c, IntC<S ^ 1>{});
        step(chunk, IntC<6>{}, last_c, IntC<S>{}); step(chunk, IntC<7>{}, last_c, IntC<S ^ 1>{}); step(chunk, IntC<8>{}, last_c, IntC<S>{});
    };
    for (int c = c0;; c += 2) {
        if (c == c1 - 1) { taps(c, BoolC<true>{}, IntC<0>{}); break; }
        taps(c, BoolC<false>{}, IntC<0>{});
        if (c + 1 == c1 - 1) { taps(c + 1, BoolC<true>{}, IntC<1>{}); break; }
        taps(c + 1, BoolC<false>{}, IntC<1>{});
    }

    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory"); /* the last MFMA results retire before they are read */
    /* The two halves of K: a wave keeps half of the channels of its 64 x 64 and hands the others to its partner */
    constexpr int KN = TN / 2;
    f32x4 sum[KN][TM];
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); /* nobody reads patches or weights any more */
    const auto hand = [&](auto kh_c) {
        constexpr int K = decltype(kh_c)::value;
        const auto block = [&](int keep, int i, int j) {
            const int n = (keep * KN + i) * TM + j;
            f32x4 a;
            asm volatile("v_accvgpr_read_b32 %0, a[%4]\n\tv_accvgpr_read_b32 %1, a[%5]\n\tv_accvgpr_read_b32 %2, a[%6]\n\tv_accvgpr_read_b32 %3, a[%7]"
                         : "=&v"(a[0]), "=&v"(a[1]), "=&v"(a[2]), "=&v"(a[3]) : "i"(4 * n), "i"(4 * n + 1), "i"(4 * n + 2), "i"(4 * n + 3));
            return a;
        };
#pragma unroll
        for (int i = 0; i < KN; i++)
#pragma unroll
            for (int j = 0; j < TM; j++) {
                *(f32x4 *)(smem + ((wave * KN + i) * TM + j) * 1024 + lane * 16) = block(K ^ 1, i, j);
                sum[i][j] = block(K, i, j);
            }
    };
    if (kh) hand(IntC<1>{});
    else hand(IntC<0>{});
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
    for (int i = 0; i < KN; i++)
#pragma unroll
        for (int j = 0; j < TM; j++) sum[i][j] += *(const f32x4 *)(smem + (((wave ^ 2) * KN + i) * TM + j) * 1024 + lane * 16);
    int l15e = l15, lqe = lq;
    asm volatile("" : "+v"(l15e), "+v"(lqe));
    const GemmArgs ge = conv_args_again();
    if constexpr (EPI == EPI_CONV_PARTIAL) store_tile<BN, 64, BN / 2, EPI, 2, true>(g, t, sum, m0, M, half, kh, l15e, lqe, t.tm * 2 + half);
    else store_tile<BN, 64, BN / 2, EPI, 2, true>(ge, t, sum, m0, ge.M[0], half, kh, l15e, lqe, t.tm * 2 + half);
}

/* ------------------------------------------------------------------ host side */

static int g_persistent = 1;
extern "C" void flux_hip_linear_persistent(int on) { g_persistent = on; }
static int compute_units() {
    static int n = 0;
    if (!n) {
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n < 8) n = 256;
    }
    return n;
}

static void set_row_tiles(GemmArgs &g, int BM) {
    int end = 0;
    for (int i = 0; i < GEMM_MAX_PARTS; i++) {
        end += (g.M[i] + BM - 1) / BM; /* empty parts (M = 0) add nothing */
        g.mt_end[i] = end;
    }
    g.mtiles = end;
}

template <int BM, int BN, int WGM, int WGN, int EPI>
static int launch_cfg(GemmArgs &g) {
    constexpr int T = WGM * WGN * 64;
    constexpr int LDS = 2 * (BM + BN) * 128;
    static bool attr_done = false;
    auto kern = gemm_kernel<BM, BN, WGM, WGN, EPI>;
    if (!attr_done) {
        HIP_OK(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, LDS));
        attr_done = true;
    }
    set_row_tiles(g, BM);
    g.ntiles = g.N / BN;
    g.nq_tiles = g.nq_cols / BN;
    g.total_tiles = g.mtiles * g.ntiles;
    int grid = (g.total_tiles * g.ksplit + 7) & ~7;
    g.vgrid = grid;
    hipLaunchKernelGGL(kern, dim3(grid), dim3(T), LDS, flux_hip_stream_handle(), g);
    HIP_OK(hipGetLastError());
    return 1;
}

template <int BN, int EPI>
static int launch_few(GemmArgs &g) {
    constexpr int STAGE = (128 + BN) * 128, LDS = (160 * 1024 / STAGE < 6 ? 160 * 1024 / STAGE : 6) * STAGE;
    static bool attr_done = false;
    auto kern = gemm_few_kernel<BN, EPI>;
    if (!attr_done) {
        HIP_OK(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, LDS));
        attr_done = true;
    }
    set_row_tiles(g, 128);
    g.nq_tiles = (g.nq_cols + BN - 1) / BN; /* both sides of the fused projection end in a tile that may be cut off */
    g.ntiles = g.nq_tiles + (g.N - g.nq_cols + BN - 1) / BN;
    g.total_tiles = g.mtiles * g.ntiles;
    g.vgrid = (g.total_tiles * g.ksplit + 7) & ~7;
    hipLaunchKernelGGL(kern, dim3(g.vgrid), dim3(512), LDS, flux_hip_stream_handle(), g);
    HIP_OK(hipGetLastError());
    return 1;
}

template <int TM, int TN, int EPI, int WGM = 2, int WGN = 2>
static int launch_4w(GemmArgs &g) {
    constexpr int BM = 16 * TM * WGM, BN = 16 * TN * WGN, LDS = 2 * (BM + BN) * 128;
    static bool attr_done = false;
    auto kern = gemm4w_kernel<TM, TN, EPI, WGM, WGN>;
    if (!attr_done) {
        HIP_OK(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, LDS));
        attr_done = true;
    }
    set_row_tiles(g, BM);
    g.ntiles = g.N / BN;
    g.nq_tiles = g.nq_cols / BN;
    g.total_tiles = g.mtiles * g.ntiles;
    /* the kernel addresses operand rows with 32-bit byte offsets from the matrix base */
    size_t span = ((size_t)max(max(g.w_row0, g.w_row1), g.w_row2) + g.N) * g.ldw * 2;
    for (int i = 0; i < GEMM_MAX_PARTS; i++) span = max(span, (size_t)g.M[i] * g.lda * 2);
    if (span >= ((size_t)1 << 32)) return g.N % 128 == 0 ? launch_cfg<128, 128, 2, 2, EPI>(g) : launch_cfg<64, 64, 2, 2, EPI>(g);
    /* one workgroup fits on a compute unit (registers, LDS): launch at most that many, each walks its share of the tiles */
    g.vgrid = (g.total_tiles * g.ksplit + 7) & ~7;
    const int grid = g_persistent && Walks4w<WGM * WGN>::value ? min(g.vgrid, compute_units() & ~7) : g.vgrid;
    hipLaunchKernelGGL(kern, dim3(grid), dim3(64 * WGM * WGN), LDS, flux_hip_stream_handle(), g);
    HIP_OK(hipGetLastError());
    return 1;
}

static int g_ring = 1;
extern "C" void flux_hip_linear_ring(int on) { g_ring = on; }

/* The deep-ring form of the 4-wave tiles: one workgroup per compute unit at most, each walks its share of the tiles. */
template <int TM, int TN, int EPI, int NSA, int NSW>
static int launch_4d(GemmArgs &g) {
    constexpr int BM = 32 * TM, BN = 32 * TN, LDS = (NSA * BM + NSW * BN) * 128;
    static bool attr_done = false;
    auto kern = gemm4d_kernel<TM, TN, EPI, NSA, NSW>;
    if (!attr_done) {
        HIP_OK(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, LDS));
        attr_done = true;
    }
    set_row_tiles(g, BM);
    g.ntiles = (g.N + BN - 1) / BN; /* (a last tile that is cut off: CutTile) */
    g.nq_tiles = g.nq_cols / BN;
    g.total_tiles = g.mtiles * g.ntiles;
    size_t span = ((size_t)max(max(g.w_row0, g.w_row1), g.w_row2) + g.N) * g.ldw * 2;
    for (int i = 0; i < GEMM_MAX_PARTS; i++) span = max(span, (size_t)g.M[i] * g.lda * 2);
    if constexpr (!IsConv<EPI>::value && EPI != EPI_EXP) /* (conv_launch and flux_hip_linear_exp have looked) */
        if (span >= ((size_t)1 << 32)) return g.N % 128 == 0 ? launch_cfg<128, 128, 2, 2, EPI>(g) : launch_cfg<64, 64, 2, 2, EPI>(g);
    g.vgrid = (g.total_tiles * g.ksplit + 7) & ~7;
    const int grid = min(g.vgrid, compute_units() & ~7);
    hipLaunchKernelGGL(kern, dim3(grid), dim3(256), LDS, flux_hip_stream_handle(), g);
    HIP_OK(hipGetLastError());
    return 1;
}

template <int TM, int TN, int EPI>
static int launch_4x(GemmArgs &g) {
    constexpr int BM = 32 * TM, BN = 32 * TN, LDS = 2 * (BM + BN) * 128;
    static bool attr_done = false;
    auto kern = gemm4x_kernel<TM, TN, EPI>;
    if (!attr_done) {
        HIP_OK(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, LDS));
        attr_done = true;
    }
    set_row_tiles(g, BM);
    g.nq_tiles = (g.nq_cols + BN - 1) / BN; /* both sides of the fused projection end in a tile that may be cut off */
    g.ntiles = g.nq_tiles + (g.N - g.nq_cols + BN - 1) / BN;
    g.total_tiles = g.mtiles * g.ntiles;
    size_t span = ((size_t)max(max(g.w_row0, g.w_row1), g.w_row2) + g.N) * g.ldw * 2;
    for (int i = 0; i < GEMM_MAX_PARTS; i++) span = max(span, (size_t)g.M[i] * g.lda * 2);
    if (span >= ((size_t)1 << 32)) return g.N % 128 == 0 ? launch_cfg<128, 128, 2, 2, EPI>(g) : launch_cfg<64, 64, 2, 2, EPI>(g);
    g.vgrid = (g.total_tiles + 7) & ~7;
    const int grid = min(g.vgrid, compute_units() & ~7);
    hipLaunchKernelGGL(kern, dim3(grid), dim3(256), LDS, flux_hip_stream_handle(), g);
    HIP_OK(hipGetLastError());
    return 1;
}

template <int EPI>
static int launch_epi(GemmArgs &g, int tile) {
    /* the ring kernel runs its tiles as one pipeline and wants at least four K steps in every K slice (the last slice
     * may be shorter than the others); shorter ones go to the two-stage kernel */
    const int kt_total = g.K >> 6, kt_last = kt_total - (g.ksplit - 1) * g.kt_per;
    if (g_ring && g_persistent && g.kt_per >= 4 && kt_last >= 4) {
        /* three weight slots, two activation slots: in a denoising step the weights always come from HBM, the
         * activations mostly from the memory-side cache (measured per kernel in a step, this split beat the other
         * one by 0 - 10 %); the 192 x 192 tile has room for three of each */
        switch (tile) {
            case 2: return launch_4d<8, 8, EPI, 2, 3>(g);
            case 5: return launch_4d<9, 6, EPI, 2, 3>(g);
            case 6: return launch_4d<6, 6, EPI, 3, 3>(g);
            case 7: return launch_4d<8, 6, EPI, 2, 3>(g);
            case 12: return launch_4d<8, 4, EPI, 3, 3>(g);
            case 13: return launch_4d<4, 4, EPI, 3, 3>(g);
            case 14: return launch_4d<6, 8, EPI, 2, 3>(g);
            case 17: if constexpr (EPI == EPI_QKV_SWIGLU) return launch_4x<9, 9, EPI>(g); break;
            case 18: if constexpr (EPI == EPI_QKV_SWIGLU) return launch_4x<12, 7, EPI>(g); break;
            case 19: if constexpr (EPI == EPI_QKV_SWIGLU) return launch_4x<10, 7, EPI>(g); break;
            case 20: if constexpr (EPI == EPI_QKV_SWIGLU) return launch_4x<10, 8, EPI>(g); break;
            case 21: if constexpr (EPI == EPI_QKV_SWIGLU) return launch_4x<9, 8, EPI>(g); break;
            case 22: if constexpr (EPI == EPI_QKV_SWIGLU) return launch_4x<11, 7, EPI>(g); break;
            case 23: if constexpr (EPI == FLUX_HIP_EPI_SWIGLU) return launch_4d<8, 5, EPI, 3, 3>(g); break;
            case 11:
                if constexpr (EPI == FLUX_HIP_EPI_RESID || EPI == FLUX_HIP_EPI_BF16) return launch_4d<8, 7, EPI, 2, 3>(g);
                break;
            default: break;
        }
    }
    if ((tile >= 11 && tile < 15) || (tile > 16 && tile < 24)) tile = g.N % 256 == 0 ? 2 : 1; /* (the dispatch offers these only where the ring kernel takes them) */
    switch (tile) {
        case 2: return launch_4w<8, 8, EPI>(g);
        case 5: return launch_4w<9, 6, EPI>(g);
        case 6: return launch_4w<6, 6, EPI>(g);
        case 7: return launch_4w<8, 6, EPI>(g);
        case 4: return launch_4w<8, 4, EPI, 2, 4>(g); /* 8 waves, two per SIMD, on the 256x256 tile */
        case 1: return launch_cfg<128, 128, 2, 2, EPI>(g);
        case 3: return launch_cfg<64, 64, 2, 2, EPI>(g);
        case 8: return launch_few<80, EPI>(g);
        case 9: return launch_few<128, EPI>(g);
        case 10: return launch_few<112, EPI>(g);
        case 16: return launch_few<96, EPI>(g);
        case 24: return launch_few<144, EPI>(g);
        default: return launch_cfg<64, 128, 2, 2, EPI>(g);
    }
}

/* Second pass of a split-K GEMM: sums the K slices ws[s][moff + m][n] in a fixed order and
 * applies the epilogue to the sum (for the residual form the same arithmetic as gated_add,
 * flux_transformer.c:90-97). For SwiGLU the workspace holds plain columns - gate features in
 * [0, N/2), up features in [N/2, N) - and thread n4 combines column n with column N/2 + n. */
template <int EPI>
__global__ __launch_bounds__(256) void splitk_finish_kernel(GemmArgs g) {
    const int ncols = EPI == FLUX_HIP_EPI_SWIGLU ? g.N >> 1 : g.N;
    const int n4 = ncols >> 2;
    const size_t total = (size_t)g.ws_rows * n4;
    size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= total) return;
    int row = (int)(idx / n4), n = (int)(idx - (size_t)row * n4) << 2;
    if (EPI == FLUX_HIP_EPI_F32_T) { /* neighbouring threads write neighbouring rows */
        n = (int)(idx / g.ws_rows) << 2;
        row = (int)(idx - (size_t)(n >> 2) * g.ws_rows);
    }
    /* moff[i] = first workspace row of part i; unused parts start at ws_rows */
    int prob = (row >= g.moff[1]) + (row >= g.moff[2]) + (row >= g.moff[3]);
    int m = row - g.moff[prob];
    f32x4 sum = {0.0f, 0.0f, 0.0f, 0.0f}, sum2 = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int s = 0; s < g.ksplit; s++) {
        const float *w = g.ws + ((size_t)s * g.ws_rows + g.moff[prob] + m) * g.N + n;
        f32x4 v = *(const f32x4 *)w;
#pragma unroll
        for (int e = 0; e < 4; e++) sum[e] += v[e];
        if (EPI == FLUX_HIP_EPI_SWIGLU) {
            f32x4 u = *(const f32x4 *)(w + ncols);
#pragma unroll
            for (int e = 0; e < 4; e++) sum2[e] += u[e];
        }
    }
    if (EPI == FLUX_HIP_EPI_RESID) {
        float *p = (float *)g.C[prob] + (size_t)m * g.ldc + n;
        f32x4 x = *(f32x4 *)p;
        f32x4 gt = *(const f32x4 *)(g.gate[prob] + n);
#pragma unroll
        for (int e = 0; e < 4; e++) x[e] += gt[e] * sum[e];
        *(f32x4 *)p = x;
    } else if (EPI == FLUX_HIP_EPI_F32) {
        *(f32x4 *)((float *)g.C[prob] + (size_t)m * g.ldc + n) = sum;
    } else if (EPI == FLUX_HIP_EPI_F32_T) {
#pragma unroll
        for (int e = 0; e < 4; e++) ((float *)g.C[prob])[(size_t)(n + e) * g.ldc + m] = sum[e];
    } else {
        bf16x4 o;
#pragma unroll
        for (int e = 0; e < 4; e++) o[e] = (bf16)(EPI == FLUX_HIP_EPI_SWIGLU ? silu_f(sum[e]) * sum2[e] : sum[e]);
        *(bf16x4 *)((bf16 *)g.C[prob] + (size_t)m * g.ldc + n) = o;
    }
}

/* Second pass of a convolution that ran as K slices: sums the slices of 32 positions x 64 channels in slice order, adds bias and
 * residual, writes the interior and the zero border, and leaves the sums for the group norm that follows, one row of
 * them per 32 positions. ksplit = 0 (an image without interior) writes zeros. */
template <int EPI>
__global__ __launch_bounds__(256) void conv_finish_kernel(GemmArgs g) {
    __shared__ float sh[4 * 16 * 2];
    constexpr bool F32 = EPI == FLUX_HIP_EPI_CONV_F32;
    const int q = threadIdx.x & 15, r = threadIdx.x >> 4, n = blockIdx.y * 64 + q * 4, wp = g.conv_wp;
    const size_t slice = (size_t)g.M[0] * g.N;
    float s1 = 0.0f, s2 = 0.0f;
    const f32x4 bv = *(const f32x4 *)(g.bias + n);
#pragma unroll
    for (int it = 0; it < 2; it++) {
        const int p = blockIdx.x * 32 + it * 16 + r;
        if (p >= g.conv_rows) break;
        int m = p;
        bool inside = g.ksplit > 0;
        if (wp > 0) {
            const int y = p / wp, x = p - y * wp;
            inside = inside && y >= 1 && p < g.conv_rows - wp && x >= 1 && x < wp - 1;
            m = (y - 1) * (wp - 2) + x - 1;
        }
        f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
        if (inside) {
            f32x4 a = v;
            if (g.res) v = *(const f32x4 *)(g.res + (size_t)p * g.ldc + n);
            const float *w = g.ws + (size_t)m * g.N + n;
#pragma unroll 8
            for (int s = 0; s < g.ksplit; s++) {
                const f32x4 t = *(const f32x4 *)(w + s * slice);
#pragma unroll
                for (int e = 0; e < 4; e++) a[e] += t[e];
            }
#pragma unroll
            for (int e = 0; e < 4; e++) {
                v[e] = v[e] + a[e] + bv[e];
                s1 += v[e];
                s2 += v[e] * v[e];
            }
        }
        if (g.conv_packed_out && !inside) continue;
        const size_t at = (size_t)(g.conv_packed_out ? m : p) * g.ldc + n;
        if (F32) {
            *(f32x4 *)((float *)g.C[0] + at) = v;
        } else {
            bf16x4 o;
#pragma unroll
            for (int e = 0; e < 4; e++) o[e] = (bf16)v[e];
            *(bf16x4 *)((bf16 *)g.C[0] + at) = o;
        }
    }
    if (g.stats) {
        s1 += __shfl_xor(s1, 16); s2 += __shfl_xor(s2, 16);
        s1 += __shfl_xor(s1, 32); s2 += __shfl_xor(s2, 32);
        const int wave = threadIdx.x >> 6;
        if ((threadIdx.x & 63) < 16) { sh[(wave * 16 + q) * 2] = s1; sh[(wave * 16 + q) * 2 + 1] = s2; }
        __syncthreads();
        if (threadIdx.x < 16) {
            const float *c = sh + q * 2;
            const f32x2 o = {(c[0] + c[32]) + (c[64] + c[96]), (c[1] + c[33]) + (c[65] + c[97])};
            *(f32x2 *)(g.stats + ((size_t)blockIdx.x * (g.N >> 2) + (n >> 2)) * 2) = o;
        }
    }
}

/* What follows a residual projection in every block is the AdaLN of the updated rows
 * (apply_adaln, flux_transformer.c:979-1048). When the projection ran as K slices, this kernel is
 * its second pass and that normalisation in one: a workgroup owns one row, sums the slices in
 * the fixed order, updates x (as splitk_finish_kernel<RESID> does), and while the row is still in
 * registers computes mean and biased variance (two passes) and writes
 * (1 + scale) * (x - mean) / sqrt(var + eps) + shift as bf16. One read of the partial sums, one
 * read and write of x, one write of the normalised row. N <= 4096. */
struct AdalnArgs {
    bf16 *out[GEMM_MAX_PARTS];
    const float *shift[GEMM_MAX_PARTS], *scale[GEMM_MAX_PARTS]; /* RMS form: scale = the norm's weight, shift unused */
    int ldo;
    float eps;
};

/* v summed over the workgroup's waves */
__device__ __forceinline__ float block_sum(float v, float *red, int waves) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    __syncthreads(); /* red is free again */
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    float sum = 0.0f;
    for (int w = 0; w < waves; w++) sum += red[w];
    return sum;
}

/* RMS = true: the norm that follows is x / sqrt(mean(x^2) + eps) * weight instead (qwen3_rms_norm,
 * flux_qwen3.c:177-197). A thread owns Q quads of columns, blockDim.x quads apart. Everything the row needs is requested at once - the first U
 * slices, then x, gate, scale and shift - so that it costs one round trip to memory beside the further slices. With 256 threads of
 * four quads, four slices at a time and scale and shift behind them / now, us: three slices of 3072, 80 rows 5.9 / 4.2, 200 6.4 / 4.9, 512 9.0 / 8.0, 768 10.9 / 10.2,
 * 1202 17.5 / 14.9, 2498 31.0 / 26.4; four slices 768 rows 12.2 / 11.4, 2498 34.1 / 33.2; four slices of 2560, 80 rows 4.5 / 4.1, 512 7.8 / 7.5. */
template <bool RMS, int Q, int U>
__global__ __launch_bounds__(1024 / Q) void splitk_finish_adaln_kernel(GemmArgs g, AdalnArgs a) {
    __shared__ float red[16];
    const int row = blockIdx.x, threads = blockDim.x, waves = threads >> 6;
    const int prob = (row >= g.moff[1]) + (row >= g.moff[2]) + (row >= g.moff[3]);
    const int m = row - g.moff[prob];
    const int N = g.N;
    float *xr = (float *)g.C[prob] + (size_t)m * g.ldc;
    const float *gate = g.gate[prob], *scale = a.scale[prob], *shift = RMS ? nullptr : a.shift[prob];
    f32x4 v[Q], x0[Q], gt0[Q], sc0[Q], sh0[Q];
    int c[Q];
    bool mine[Q];
#pragma unroll
    for (int i = 0; i < Q; i++) {
        const int at = (i * threads + threadIdx.x) * 4;
        mine[i] = at < N;
        c[i] = mine[i] ? at : 0;
        v[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    /* slices U at a time, the additions in slice order */
    const size_t slice = (size_t)g.ws_rows * N;
    const float *w0 = g.ws + (size_t)row * N;
    f32x4 t[U][Q];
    const auto request = [&](int s) {
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int i = 0; i < Q; i++)
                if (s + u < g.ksplit) t[u][i] = *(const f32x4 *)(w0 + (size_t)(s + u) * slice + c[i]);
    };
    request(0);
#pragma unroll
    for (int i = 0; i < Q; i++) {
        x0[i] = *(const f32x4 *)(xr + c[i]);
        gt0[i] = *(const f32x4 *)(gate + c[i]);
        sc0[i] = *(const f32x4 *)(scale + c[i]);
        if (!RMS) sh0[i] = *(const f32x4 *)(shift + c[i]);
    }
    for (int s = 0;;) {
#pragma unroll
        for (int u = 0; u < U; u++)
            if (s + u < g.ksplit) {
#pragma unroll
                for (int i = 0; i < Q; i++)
#pragma unroll
                    for (int e = 0; e < 4; e++) v[i][e] += t[u][i][e];
            }
        s += U;
        if (s >= g.ksplit) break;
        request(s);
    }
    float s1 = 0.0f;
#pragma unroll
    for (int i = 0; i < Q; i++) {
        f32x4 x = x0[i];
#pragma unroll
        for (int e = 0; e < 4; e++) x[e] += gt0[i][e] * v[i][e];
        v[i] = x;
        if (mine[i]) {
            *(f32x4 *)(xr + c[i]) = x;
            s1 += (x[0] + x[1]) + (x[2] + x[3]);
        }
    }
    const float mean = RMS ? 0.0f : block_sum(s1, red, waves) / (float)N;
    float q = 0.0f;
#pragma unroll
    for (int i = 0; i < Q; i++)
        if (mine[i]) {
#pragma unroll
            for (int e = 0; e < 4; e++) { const float d = v[i][e] - mean; q += d * d; }
        }
    const float inv = 1.0f / sqrtf(block_sum(q, red, waves) / (float)N + a.eps);
    bf16 *o = a.out[prob] + (size_t)m * a.ldo;
#pragma unroll
    for (int i = 0; i < Q; i++) {
        bf16x4 r;
#pragma unroll
        for (int e = 0; e < 4; e++) r[e] = (bf16)(RMS ? v[i][e] * inv * sc0[i][e] : (1.0f + sc0[i][e]) * ((v[i][e] - mean) * inv) + sh0[i][e]);
        if (mine[i]) *(bf16x4 *)(o + c[i]) = r;
    }
}

static int launch_exp(GemmArgs &g, int tile) {
    switch (tile) {
        case 2: return launch_4d<8, 8, EPI_EXP, 2, 3>(g);
        case 12: return launch_4d<8, 4, EPI_EXP, 3, 3>(g);
        default: return launch_4d<4, 4, EPI_EXP, 3, 3>(g);
    }
}

template <int EPI>
static int launch_split(GemmArgs &g, int tile) {
    if (!launch_epi<EPI_PARTIAL>(g, tile)) return 0;
    const size_t total = (size_t)g.ws_rows * ((EPI == FLUX_HIP_EPI_SWIGLU ? g.N >> 1 : g.N) >> 2);
    hipLaunchKernelGGL(splitk_finish_kernel<EPI>, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, flux_hip_stream_handle(), g);
    return hipGetLastError() == hipSuccess ? 1 : flux_hip_fail("split-K reduction launch failed");
}

static int launch_split_adaln(GemmArgs &g, int tile, const AdalnArgs &a) {
    if (!launch_epi<EPI_PARTIAL>(g, tile)) return 0;
    /* Few rows wait for memory: a quad a thread, four slices on their way. With more rows than units it is the bytes (768 rows in four slices: 61 MB), and
     * small workgroups win. Whole passes, us, a quad a thread / four: prompts of 67 tokens 2633 / 2690, 128 3172 / 3227, 200 3748 / 3784,
     * 300 4345 / 4343, 512 5167 / 5168; denoising steps of 80 tokens 2478 / 2507, 208 3313 / 3305, 320 3743 / 3720, 640 5051 / 5000. */
    const bool few = g.ws_rows <= 200;
    const int quads = g.N >> 2, threads = few ? (quads + 63) / 64 * 64 : (quads + 255) / 256 * 64;
    auto kern = few ? (a.shift[0] ? splitk_finish_adaln_kernel<false, 1, 4> : splitk_finish_adaln_kernel<true, 1, 4>)
                    : (a.shift[0] ? splitk_finish_adaln_kernel<false, 4, 2> : splitk_finish_adaln_kernel<true, 4, 2>);
    hipLaunchKernelGGL(kern, dim3((unsigned)g.ws_rows), dim3(threads), 0, flux_hip_stream_handle(), g, a);
    return hipGetLastError() == hipSuccess ? 1 : flux_hip_fail("split-K reduction + AdaLN launch failed");
}

/* Workspace of flux_hip_linear_static: the K slices' partial sums live in this array instead of in
 * memory from hipMalloc. Each GPU that loads the library holds its own copy until the process ends.
 * In host code the array's name is only a handle for hipGetSymbolAddress; the address a kernel can
 * use is asked for once per device (static_ws_for_current_device) and kept. */
#define STATIC_WS_BYTES ((size_t)FLUX_HIP_LINEAR_STATIC_BYTES)
static __device__ __align__(256) float g_static_ws[STATIC_WS_BYTES / sizeof(float)];
#define STATIC_WS_MAX_DEVICES 64
static float *g_static_ws_ptr[STATIC_WS_MAX_DEVICES];

static float *static_ws_for_current_device() {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= STATIC_WS_MAX_DEVICES) {
        flux_hip_fail("flux_hip_linear_static: no current device (or a device number beyond %d)", STATIC_WS_MAX_DEVICES - 1);
        return nullptr;
    }
    if (!g_static_ws_ptr[dev]) {
        float *p = nullptr;
        const hipError_t e = hipGetSymbolAddress((void **)&p, HIP_SYMBOL(g_static_ws));
        if (e != hipSuccess || !p) {
            flux_hip_fail("flux_hip_linear_static: hipGetSymbolAddress failed: %s", hipGetErrorString(e));
            return nullptr;
        }
        g_static_ws_ptr[dev] = p;
    }
    return g_static_ws_ptr[dev];
}

/* called by flux_hip_init with its device current */
extern "C" int flux_hip_linear_static_init(void) { return static_ws_for_current_device() != nullptr; }

extern "C" void flux_hip_linear_release(void);
static float *g_ws = nullptr;
static size_t g_ws_bytes = 0;
static int ensure_ws(size_t bytes) {
    if (bytes <= g_ws_bytes) return 1;
    HIP_OK(hipStreamSynchronize(flux_hip_stream_handle()));
    if (g_ws) (void)hipFree(g_ws);
    g_ws = nullptr;
    g_ws_bytes = 0;
    HIP_OK(hipMalloc((void **)&g_ws, bytes));
    g_ws_bytes = bytes;
    return 1;
}

/* Whether K slices can have their partial sums in the growing workspace: not where the memory cannot be had, and not under stream
 * capture (the graph would keep the address of memory that a later call may free to grow it, and growing it fails there). Slices
 * are a choice of speed, so no call fails for that: a projection takes the static array instead, a convolution runs in
 * one piece. */
static bool workspace_for_slices(size_t bytes) {
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(flux_hip_stream_handle(), &capture) != hipSuccess || capture != hipStreamCaptureStatusNone) {
        (void)hipGetLastError();
        return false;
    }
    if (ensure_ws(bytes)) return true;
    (void)hipGetLastError(); /* the next launch is not to report this one */
    return false;
}

extern "C" void flux_hip_linear_release(void) {
    if (g_ws) (void)hipFree(g_ws);
    g_ws = nullptr;
    g_ws_bytes = 0;
}

static int g_force_tile = -1;
#define TILE_MASK_ALL 0x1FF7FEFu /* tiles the automatic choice may use: all but the 8-wave form of 256 x 256 */
static unsigned g_tile_mask = TILE_MASK_ALL;
static int g_splitk_enabled = 1;
extern "C" void flux_hip_linear_force_tile(int tile) { g_force_tile = tile; }
extern "C" void flux_hip_linear_tile_mask(unsigned mask) { g_tile_mask = mask ? mask : TILE_MASK_ALL; }
extern "C" void flux_hip_linear_enable_splitk(int on) { g_splitk_enabled = on; }
static int g_force_split = 0; /* > 1: every projection that can run as K slices runs as this many (comparison runs and tests) */
extern "C" void flux_hip_linear_force_split(int slices) { g_force_split = slices > 1 ? slices : 0; }

/* Launch probe: HIP events around every launch with one chosen epilogue, so a benchmark can
 * read that kernel's average duration inside its timed region. */
#define PROBE_MAX 4096
static int g_probe_epi = -1, g_probe_n = 0;
static hipEvent_t g_probe_ev[PROBE_MAX][2];
static unsigned char g_probe_tile[PROBE_MAX];
static int g_probe_created = 0;

extern "C" int flux_hip_linear_probe(int epilogue) {
    g_probe_epi = epilogue;
    g_probe_n = 0;
    return 1;
}

/* Count and summed duration of the recorded launches that used `tile` (-1: all of them). The
 * record is kept until the next flux_hip_linear_probe call. */
extern "C" int flux_hip_linear_probe_read_tile(int tile, int *launches, float *total_ms) {
    float sum = 0.0f;
    int n = 0;
    for (int i = 0; i < g_probe_n; i++) {
        if (tile >= 0 && g_probe_tile[i] != tile) continue;
        float ms = 0.0f;
        HIP_OK(hipEventSynchronize(g_probe_ev[i][1]));
        HIP_OK(hipEventElapsedTime(&ms, g_probe_ev[i][0], g_probe_ev[i][1]));
        sum += ms;
        n++;
    }
    if (launches) *launches = n;
    if (total_ms) *total_ms = sum;
    return 1;
}

extern "C" int flux_hip_linear_probe_read(int *launches, float *total_ms) {
    return flux_hip_linear_probe_read_tile(-1, launches, total_ms);
}

/* Duration and tile id of each recorded launch, in launch order; returns how many were written. */
extern "C" int flux_hip_linear_probe_read_launches(int max, int *tiles, float *ms) {
    int n = 0;
    for (int i = 0; i < g_probe_n && n < max; i++, n++) {
        float t = 0.0f;
        if (hipEventSynchronize(g_probe_ev[i][1]) != hipSuccess || hipEventElapsedTime(&t, g_probe_ev[i][0], g_probe_ev[i][1]) != hipSuccess) return -1;
        if (tiles) tiles[n] = g_probe_tile[i];
        if (ms) ms[n] = t;
    }
    return n;
}

static int probe_slot(int epilogue) {
    const bool conv = epilogue == FLUX_HIP_EPI_CONV_BF16 || epilogue == FLUX_HIP_EPI_CONV_F32;
    if ((g_probe_epi == -2 ? !conv : epilogue != g_probe_epi) || g_probe_n >= PROBE_MAX) return -1;
    while (g_probe_created <= g_probe_n) {
        if (hipEventCreate(&g_probe_ev[g_probe_created][0]) != hipSuccess) return -1;
        if (hipEventCreate(&g_probe_ev[g_probe_created][1]) != hipSuccess) return -1;
        g_probe_created++;
    }
    return g_probe_n++;
}

/* for the convolutions of conv.hip that are not launched from here */
int conv_probe_begin(int epilogue, int tile) {
    const int slot = probe_slot(epilogue);
    if (slot >= 0) {
        g_probe_tile[slot] = (unsigned char)tile;
        (void)hipEventRecord(g_probe_ev[slot][0], flux_hip_stream_handle());
    }
    return slot;
}
void conv_probe_end(int slot) {
    if (slot >= 0) (void)hipEventRecord(g_probe_ev[slot][1], flux_hip_stream_handle());
}

/* Tile and K-split choice, then the launch; `allowed` has bit t set for every tile id that may be used. */
static int gemm_dispatch(GemmArgs &g, int np, int epilogue, unsigned allowed, int *tile_out = nullptr, const AdalnArgs *adaln = nullptr,
                         int *adaln_done = nullptr, float *fixed_ws = nullptr, size_t fixed_ws_bytes = 0, int *leave_slices = nullptr) {
    /* Choose tile and K split with a small cost model: workgroups run in rounds over
     * 256 CUs x occupancy; a workgroup's time is its FLOPs at the tile's measured rate plus a
     * fixed prologue/epilogue cost; the launch cannot beat the time to stream its operands,
     * which depends on how many bytes the resident workgroups keep in flight. */
    /* tile ids: 0..3 the small tiles and 256 x 256, 4 = the 8-wave form of 256 x 256 (only when
     * forced, for comparison runs), 5 = 288 x 192, 6 = 192 x 192, 7 = 256 x 192, 8, 16, 10, 9 and 24 = gemm_few_kernel's, 80, 96, 112, 128 and 144
     * columns wide, for parts of at most 128 rows, 11 = 256 x 224 (4096 + 512 rows x 3072 columns are 252 such tiles, one round of workgroups on 256
     * compute units of which each does 7/8 of a 256 x 256 tile's work; 216 tiles of 256 x 256 are one round as well),
     * 12 = 256 x 128, 13 = 128 x 128 and 14 = 192 x 256 in the ring kernel, for launches of about one round: the two-stage 128 x 128
     * tile waits for memory in every K step when it has a compute unit to itself. With the weights coming from HBM, as in a
     * forward: 512 x 6144 x 2560 39 us, in the ring 30; 1202 x 3072 x 3072: 49 and 34; 512 x 19456 x 2560 on 228 tiles of 192 x 256 52,
     * on 152 of 256 x 256 60. (The rates of 12 to 14 below are those of cached operands and up to 40 % above these launches; over
     * 133 shapes of 67 to 16384 rows with cold weights the chosen form took 0.8 % more than the best of seven on average.)
     * 17 to 22 = gemm4x_kernel's, for the fused projection: 288 x 288, 384 x 224, 320 x 224, 320 x 256, 288 x 256, 352 x 224. Over 29 row counts
     * from 300 to 13056 the chosen tile takes 0.3 % more than the best on average; 256 x 288 was never the best, 352 x 256 (two row
     * counts, 3 %) spills. */
    constexpr int NT = 25;
    static const int bm[NT] = {64, 128, 256, 64, 256, 288, 192, 256, 128, 128, 128, 256, 256, 128, 192, 0, 128, 288, 384, 320, 320, 288, 352, 256, 128}, bn[NT] = {128, 128, 256, 64, 256, 192, 192, 192, 80, 128, 112, 224, 128, 128, 256, 1, 96, 288, 224, 224, 256, 256, 224, 160, 144};
    static const int occ[NT] = {3, 2, 1, 4, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1};
    static const double rate[NT] = {2.0e12, 2.9e12, 6.05e12, 1.5e12, 4.6e12, 6.0e12, 5.7e12, 5.75e12, 0, 0, 0, 5.9e12, 5.3e12, 4.4e12, 5.5e12, 1.0, 0, 6.3e12, 6.1e12, 6.15e12, 6.4e12, 6.3e12, 6.15e12, 5.4e12, 0}; /* FLOP/s of one CU running this tile; 0: gemm_few_kernel */
    const int kt_total = g.K >> 6;
    int tile = -1, best_split = 1;
    {
        double best = 1e30;
        static const int splits[] = {1, 2, 3, 4, 6, 8, 12, 16, 24, 32};
        /* every epilogue can run as K slices + a finishing pass; for SwiGLU the gate and up rows must be one contiguous block of the
         * weight matrix. The transposed store (the final layer's 128 columns: 8 tiles of 64 x 64 at 256 rows) does up to 8192 rows. Weights from HBM and
         * activations just written, as in a step, us in one piece / in slices: 16 rows 24 / 13, 256 37 / 17, 2048 39 / 19, 2304 39 / 32, 4096 42 / 24, 4864 43 / 36,
         * 6912 46 / 40, 7936 46 / 44, 8192 47 / 32, never slower over 37 row counts; beyond, a gain or none as
         * the count falls: 8448 50 / 50, 9216 51 / 35, 11008 54 / 54, 12032 55 / 56, 12544 55 / 57. (With weights that a cache holds one piece takes 26 to 28 us
         * and slices up to 39 from 2304 rows on; in a step 7 GB of other weights have passed.) */
        const int N = g.N, K = g.K, w_row0 = g.w_row0, w_row1 = g.w_row1;
        double rows = 0.0;
        int most = 0;
        for (int i = 0; i < np; i++) rows += g.M[i], most = max(most, g.M[i]);
        const bool can_split = g_splitk_enabled &&
                               (epilogue == FLUX_HIP_EPI_RESID || epilogue == FLUX_HIP_EPI_BF16 || epilogue == FLUX_HIP_EPI_F32 ||
                                (epilogue == FLUX_HIP_EPI_F32_T && rows <= 8192) ||
                                (epilogue == FLUX_HIP_EPI_SWIGLU && w_row1 == w_row0 + N / 2));
        int weights = 0; /* matrices of weights: sequences share them, streams do not */
        for (int i = 0; i < np; i++) {
            weights++;
            for (int j = 0; j < i; j++)
                if (g.W[j] == g.W[i]) { weights--; break; }
        }
        for (int t = 0; t < NT; t++) {
            const bool few = rate[t] == 0;
            if (few && most > 128) continue; /* they stream the weights once: every part in one row tile */
            /* 256 x 224 (tile 11) divides no width and cuts its last column tile off: for the outputs whose stores can do
             * that, through the ring kernel only, never in K slices */
            const bool cut = t == 11;
            if (cut && !((epilogue == FLUX_HIP_EPI_RESID || epilogue == FLUX_HIP_EPI_BF16) && g_ring && g_persistent && kt_total >= 4)) continue;
            /* bf16 outputs leave in pairs of 16-column blocks: the cut must fall between two pairs of a wave's 112 columns */
            if (cut && epilogue == FLUX_HIP_EPI_BF16 && (N % 224) % 112 % 32 != 0) continue;
            const bool wide = t >= 17 && t < 23;
            /* 256 x 160 (tile 23) likewise, at a multiple of eight features: for SwiGLU alone. The text encoder's gate and up rows (19456 x
             * 2560) are 244 tiles of it at 512 rows, of which 256 units run all at once; with the weights from HBM, us, 23 / the best other: 260 rows
             * 43.8 / 45.8, 300 44.7 / 46.0, 384 47.0 / 46.8, 400 47.2 / 52.4, 512 47.4 / 53.8; 200 45.2 / 40.4 and 256 44.5 / 40.3,
             * where the model takes 256 x 128. */
            const bool cut160 = t == 23;
            if (cut160 && !(epilogue == FLUX_HIP_EPI_SWIGLU && N % 64 == 0 && g_ring && g_persistent && kt_total >= 4)) continue;
            if (wide && !(epilogue == EPI_QKV_SWIGLU && g_ring && g_persistent && kt_total >= 4)) continue;
            if (wide && bn[t] == 256 && (g.nq_cols & 255 || N & 255)) continue; /* (CutTile) */
            if (!cut && !cut160 && !wide && !few && (N % bn[t] || g.nq_cols % bn[t])) continue;
            if (!((allowed >> t) & 1)) continue;
            if (t >= 12 && t < 15 && !(g_ring && g_persistent && kt_total >= 4)) continue;
            long tiles = 0;
            for (int i = 0; i < np; i++) tiles += (g.M[i] + bm[t] - 1) / bm[t];
            tiles *= (g.nq_cols + bn[t] - 1) / bn[t] + (N - g.nq_cols + bn[t] - 1) / bn[t];
            for (int si = 0; si < 10; si++) {
                const int sp = splits[si];
                if (sp > 1 && (cut || cut160 || wide || !can_split || kt_total / sp < 4)) break;
                if (g_force_split && can_split && sp != g_force_split && kt_total / g_force_split >= 4) continue;
                if (sp > 1 && fixed_ws && (double)sp * rows * N * sizeof(float) > (double)fixed_ws_bytes) {
                    /* the slices must fit the given workspace: fewer slices then, down to none - unless this number
                     * of slices was demanded, which is the one request the fixed workspace refuses */
                    if (sp == g_force_split)
                        return flux_hip_fail("flux_hip_linear_static: %d K slices of %.0f rows x %d columns need %.1f MiB of partial sums, beyond the maximum "
                                             "of %zu MiB of the static workspace", sp, rows, N, sp * rows * N * 4.0 / 1048576.0, fixed_ws_bytes >> 20);
                    break;
                }
                const int per = (kt_total + sp - 1) / sp;
                const long blocks = tiles * ((kt_total + per - 1) / per);
                const long slots = 256L * occ[t];
                const long rounds = (blocks + slots - 1) / slots;
                const long resident = blocks < slots ? blocks : slots;
                const long per_cu = (resident + 255) / 256;          /* workgroups sharing one CU */
                const double t_block = 2.0 * bm[t] * bn[t] * 64.0 * per / (rate[t] / per_cu) + 2.5e-6;
                double t_compute = rounds * t_block;
                const double bytes = (rows + (most <= 128 ? weights : 1) * (double)N) * K * 2.0;
                /* what a launch that only streams its operands has been seen to reach with two LDS stages (every step waits for the loads it
                 * has just requested): 3.2-3.5 TB/s */
                const double bw_cap = 3.4e12;
                double bw = 5.5e12 * (double)(resident * (bm[t] + bn[t]) * 128) / 12.0e6;
                if (bw > bw_cap) bw = bw_cap;
                double est = t_compute > bytes / bw ? t_compute : bytes / bw;
                /* What all tiles together fetch through the L2s, over the rate at which that ties the tiles with fewer bytes to those with
                 * fewer rounds (no hard limit: 128 x 128 tiles whose activations the memory-side cache held have been seen at 16 TB/s).
                 * In the step, over 26 token counts from 219 to 10709, six prompt lengths and 20 image sizes, 12.9 TB/s
                 * kept tiles with too few rounds' worth of them: out1 at 5993 rows 406 us on 256 x 192 in two slices, 342 on 192 x 192
                 * (a step 1.9 % longer), 270 prompt tokens 3 % longer, P V of 5332 positions 58 us against 47. 14.5 and
                 * none send 790 to 1300 tokens to 128 x 128 and 192 x 192, 1.2 to 3 % longer. Activations beyond the 256 MB of the
                 * memory-side cache come from HBM and the rate is lower: P V of 14580 positions 220 us on 256 x 128, which
                 * 13.5 chooses, and 183 on 256 x 256 in two slices. */
                const double l2_rate = rows * K * 2.0 > 256.0e6 ? 12.9e12 : 13.5e12;
                const double l2 = (double)tiles * (bm[t] + bn[t]) * K * 2.0 / l2_rate;
                if (l2 > est) est = l2;
                if (few) {
                    /* See gemm_few_kernel: round by round a workgroup's intake (or its LDS reads), or the round's weights from HBM. 62 launches of 16 to
                     * 128 rows: the chosen width and slices take 1 % more than the best of up to 20 on average. */
                    const double intake = ((most + 7) / 8 * 8 + bn[t]) * 128 / 54.0e9, lds = (most + 15) / 16 * (1 + bn[t] / 16) * 2048 / (128 * 2.1e9);
                    const double wg = per * (intake > lds ? intake : lds), hbm = (rows + (double)weights * N) * K * 2.0 / 6.0e12;
                    est = 3.5e-6 + 0.2 * rounds * wg;
                    for (long left = blocks; left > 0; left -= 256) {
                        const double part = hbm * (left < 256 ? left : 256) / blocks;
                        est += (wg > part ? wg : part) + 2.0e-6;
                    }
                } else if (most <= 128) {
                    est += 4.0e-6; /* their launches of few rows take that much longer than this model has them */
                }
                /* Slices cost their partial sums, and beyond 128 MB of those the stores of every round as well: the K = 12288 projection at
                 * 6148 to 6912 rows (151 to 170 MB) in two slices of 288 x 192 takes 379 + 78 us, in one piece of 256 x 192 430 and
                 * 27 for the norm, and the step around it is 0.5 to 1.2 % longer; at 2132 to 2560 rows (52 to 63 MB) two slices
                 * make it 1 % shorter. */
                if (sp > 1) est += 3.0e-6 + (sp + 2.0) * rows * N * 4.0 / (few ? 8.0e12 : sp * rows * N * 4.0 > 128.0e6 ? 2.6e12 : 4.0e12);
                else if (adaln) est += 3.0e-6 + rows * N * 6.0 / 4.0e12; /* the norm that the second pass would have taken along */
                if (est < best) { best = est; tile = t; best_split = sp; }
            }
        }
    }
    if (tile < 0) tile = g.N % 128 == 0 ? 1 : 3; /* no permitted tile divides N (a forced tile that does not fit): 128 x 128, else 64 x 64 */
    g.ksplit = 1;
    g.kt_per = kt_total;
    if (best_split > 1) {
        g.kt_per = (kt_total + best_split - 1) / best_split;
        g.ksplit = (kt_total + g.kt_per - 1) / g.kt_per;
        g.ws_rows = 0;
        for (int i = 0; i < GEMM_MAX_PARTS; i++) {
            g.moff[i] = g.ws_rows;
            g.ws_rows += g.M[i];
        }
        if (fixed_ws) {
            g.ws = fixed_ws;
        } else {
            if (!workspace_for_slices((size_t)g.ksplit * g.ws_rows * g.N * sizeof(float))) { /* once more, with as many slices as fit the static array */
                float *ws = static_ws_for_current_device();
                return ws ? gemm_dispatch(g, np, epilogue, allowed, tile_out, adaln, adaln_done, ws, STATIC_WS_BYTES, leave_slices) : 0;
            }
            g.ws = g_ws;
        }
    }

    if (tile_out) *tile_out = tile;
    /* the launch probe creates events: never on the path that promises to allocate nothing */
    const int slot = fixed_ws ? -1 : probe_slot(epilogue);
    if (slot >= 0) g_probe_tile[slot] = (unsigned char)tile;
    if (slot >= 0) (void)hipEventRecord(g_probe_ev[slot][0], flux_hip_stream_handle());
    int ok;
    const bool split = g.ksplit > 1;
    switch (epilogue) {
        case FLUX_HIP_EPI_BF16:
            if (leave_slices) *leave_slices = split ? g.ksplit : 0;
            ok = split && leave_slices ? launch_epi<EPI_PARTIAL>(g, tile) : split ? launch_split<FLUX_HIP_EPI_BF16>(g, tile) : launch_epi<FLUX_HIP_EPI_BF16>(g, tile); break;
        case EPI_EXP: ok = launch_exp(g, tile); break;
        case FLUX_HIP_EPI_F32:
            if (leave_slices) *leave_slices = split ? g.ksplit : 0;
            ok = split && leave_slices ? launch_epi<EPI_PARTIAL>(g, tile) : split ? launch_split<FLUX_HIP_EPI_F32>(g, tile) : launch_epi<FLUX_HIP_EPI_F32>(g, tile); break;
        case FLUX_HIP_EPI_F32_T: ok = split ? launch_split<FLUX_HIP_EPI_F32_T>(g, tile) : launch_epi<FLUX_HIP_EPI_F32_T>(g, tile); break;
        case FLUX_HIP_EPI_RESID:
            if (split && adaln) {
                ok = launch_split_adaln(g, tile, *adaln);
                if (adaln_done) *adaln_done = ok;
            } else {
                ok = split ? launch_split<FLUX_HIP_EPI_RESID>(g, tile) : launch_epi<FLUX_HIP_EPI_RESID>(g, tile);
            }
            break;
        case FLUX_HIP_EPI_SWIGLU: ok = split ? launch_split<FLUX_HIP_EPI_SWIGLU>(g, tile) : launch_epi<FLUX_HIP_EPI_SWIGLU>(g, tile); break;
        case EPI_QKV_SWIGLU: ok = launch_epi<EPI_QKV_SWIGLU>(g, tile); break;
        default: return flux_hip_fail("flux_hip_linear: unknown epilogue %d", epilogue);
    }
    if (slot >= 0) (void)hipEventRecord(g_probe_ev[slot][1], flux_hip_stream_handle());
    return ok;
}

static int linear_impl(int epilogue, int nparts, const flux_hip_linear_part *parts, int N, int K, int lda, int ldw, int ldc, int w_row0,
                       int w_row1, const flux_hip_adaln_part *norm, float eps, int *fused, float *fixed_ws = nullptr, size_t fixed_ws_bytes = 0,
                       const char *who = "flux_hip_linear") {
    if (epilogue < FLUX_HIP_EPI_BF16 || epilogue > FLUX_HIP_EPI_SWIGLU) return flux_hip_fail("%s: unknown epilogue %d", who, epilogue);
    if (nparts < 1 || nparts > GEMM_MAX_PARTS) return flux_hip_fail("%s: nparts=%d (1 to %d)", who, nparts, GEMM_MAX_PARTS);
    if (K <= 0 || (K & 63)) return flux_hip_fail("%s: K=%d must be a positive multiple of 64", who, K);
    if (N <= 0 || (N & 127)) return flux_hip_fail("%s: N=%d must be a positive multiple of 128", who, N);
    if (lda < K || ldw < K || (lda & 7) || (ldw & 7))
        return flux_hip_fail("%s: lda=%d ldw=%d must be >= K and multiples of 8", who, lda, ldw);
    if (epilogue != FLUX_HIP_EPI_F32_T && (ldc & 3)) return flux_hip_fail("%s: ldc=%d must be a multiple of 4", who, ldc);
    GemmArgs g = {};
    AdalnArgs a = {};
    int maxm = 0;
    for (int i = 0; i < nparts; i++) {
        if (parts[i].M < 0) return flux_hip_fail("flux_hip_linear: negative row count");
        if (parts[i].M > 0 && (!parts[i].A || !parts[i].W || !parts[i].C))
            return flux_hip_fail("flux_hip_linear: NULL operand");
        if (epilogue == FLUX_HIP_EPI_RESID && parts[i].M > 0 && !parts[i].gate)
            return flux_hip_fail("flux_hip_linear: residual epilogue needs a gate vector");
        if (parts[i].M > 0 && ((((uintptr_t)parts[i].A | (uintptr_t)parts[i].W | (uintptr_t)parts[i].gate) & 15) ||
                               ((uintptr_t)parts[i].C & (epilogue == FLUX_HIP_EPI_F32_T ? 3 : epilogue == FLUX_HIP_EPI_BF16 || epilogue == FLUX_HIP_EPI_SWIGLU ? 7 : 15))))
            return flux_hip_fail("flux_hip_linear: operands must be 16-byte aligned (bf16 outputs 8-byte)");
    }
    /* drop empty parts */
    int np = 0;
    for (int i = 0; i < nparts; i++) {
        if (parts[i].M == 0) continue;
        g.A[np] = (const bf16 *)parts[i].A;
        g.W[np] = (const bf16 *)parts[i].W;
        g.C[np] = parts[i].C;
        g.gate[np] = parts[i].gate;
        g.M[np] = parts[i].M;
        if (norm) {
            a.out[np] = (bf16 *)norm[i].out_bf16;
            a.shift[np] = norm[i].shift;
            a.scale[np] = norm[i].scale;
        }
        if (parts[i].M > maxm) maxm = parts[i].M;
        np++;
    }
    if (np == 0) return 1;
    g.N = N; g.K = K; g.lda = lda; g.ldw = ldw; g.ldc = ldc; g.w_row0 = w_row0; g.w_row1 = w_row1;
    a.ldo = N;
    a.eps = eps;
    return gemm_dispatch(g, np, epilogue, (g_force_tile >= 0 ? 1u << g_force_tile : g_tile_mask) & 0x1817FFFu, nullptr, norm ? &a : nullptr, fused,
                         fixed_ws, fixed_ws_bytes);
}

extern "C" int flux_hip_linear(int epilogue, int nparts, const flux_hip_linear_part *parts,
                               int N, int K, int lda, int ldw, int ldc, int w_row0, int w_row1) {
    return linear_impl(epilogue, nparts, parts, N, K, lda, ldw, ldc, w_row0, w_row1, nullptr, 0.0f, nullptr);
}

/* A bf16 projection of one row range whose reader can sum K slices itself: *slices = 0 and C is written as by flux_hip_linear, or
 * *slices partial sums are left at *ws, fp32 [*slices][M][N], to be added in slice order (what the second pass would do), and C is
 * untouched. The sums are valid until the next projection. */
extern "C" int flux_hip_linear_slices(const void *A, const void *W, void *C, int M, int N, int K, const float **ws, int *slices) {
    *slices = 0;
    if (M <= 0) return 1;
    if (K <= 0 || (K & 63) || N <= 0 || (N & 127)) return flux_hip_fail("flux_hip_linear_slices: N=%d must be a multiple of 128, K=%d of 64", N, K);
    if (!A || !W || !C || ((((uintptr_t)A | (uintptr_t)W) & 15) || ((uintptr_t)C & 7))) return flux_hip_fail("flux_hip_linear_slices: NULL or unaligned operand");
    GemmArgs g = {};
    g.A[0] = (const bf16 *)A; g.W[0] = (const bf16 *)W; g.C[0] = C; g.M[0] = M;
    g.N = N; g.K = K; g.lda = K; g.ldw = K; g.ldc = N;
    const int ok = gemm_dispatch(g, 1, FLUX_HIP_EPI_BF16, (g_force_tile >= 0 ? 1u << g_force_tile : g_tile_mask) & 0x1017FFFu, nullptr, nullptr, nullptr, nullptr, 0, slices);
    *ws = g.ws;
    return ok;
}

/* Attention scores as unnormalised probabilities, P[m][n] = 2^(scale * A[m] . W[n] - ref[m]) in bf16 for n < keys and 0 for keys <= n < N, and
 * their fp32 sums over pieces of each row, sums [M][*pieces] (at most N / 64 of them). N a multiple of 256, K of 64 and at least 256. In the
 * ring kernel's epilogue, where they cost a multiply-add, an exponential and half a store of 16 bytes per eight: 16384 x 16384 scores
 * written as fp32 and read by a softmax took 395 + 348 us. Not to be had where that kernel is switched off, which its caller asks first:
 * everything that fails here is an error. */
extern "C" int flux_hip_linear_exp_available(void) { return g_ring && g_persistent; }
extern "C" int flux_hip_linear_exp(const void *A, const void *W, void *P, int M, int N, int K, int lda, int ldw, const float *ref, float scale, int keys,
                                   float *sums, int *pieces) {
    *pieces = 0;
    if (!flux_hip_linear_exp_available()) return flux_hip_fail("flux_hip_linear_exp: the ring kernel is switched off");
    if (M <= 0 || N <= 0 || (N & 255) || K < 256 || (K & 63) || lda < K || ldw < K || (lda & 7) || (ldw & 7) || ((size_t)M * lda | (size_t)N * ldw) >= ((size_t)1 << 31))
        return flux_hip_fail("flux_hip_linear_exp: bad shape (M=%d, N=%d, K=%d, lda=%d, ldw=%d)", M, N, K, lda, ldw);
    if (!A || !W || !P || !ref || !sums || (((uintptr_t)A | (uintptr_t)W | (uintptr_t)P) & 15))
        return flux_hip_fail("flux_hip_linear_exp: NULL or unaligned operand");
    GemmArgs g = {};
    g.A[0] = (const bf16 *)A; g.W[0] = (const bf16 *)W; g.C[0] = P; g.M[0] = M;
    g.N = N; g.K = K; g.lda = lda; g.ldw = ldw; g.ldc = N;
    g.bias = ref; g.stats = sums; g.exp_scale = scale; g.exp_keys = keys;
    const int ok = gemm_dispatch(g, 1, EPI_EXP, 1u << 2 | 1u << 12 | 1u << 13);
    *pieces = 2 * g.ntiles;
    return ok;
}

/* C = A W^T in fp32 for a reader that sums K slices itself, as flux_hip_linear_slices: *slices = 0 and C is written, or *slices partial sums
 * are left at *ws. */
extern "C" int flux_hip_linear_f32_slices(const void *A, const void *W, float *C, int M, int N, int K, const float **ws, int *slices) {
    *slices = 0;
    if (M <= 0) return 1;
    if (K <= 0 || (K & 63) || N <= 0 || (N & 127)) return flux_hip_fail("flux_hip_linear_f32_slices: N=%d must be a multiple of 128, K=%d of 64", N, K);
    if (!A || !W || !C || (((uintptr_t)A | (uintptr_t)W | (uintptr_t)C) & 15)) return flux_hip_fail("flux_hip_linear_f32_slices: NULL or unaligned operand");
    GemmArgs g = {};
    g.A[0] = (const bf16 *)A; g.W[0] = (const bf16 *)W; g.C[0] = C; g.M[0] = M;
    g.N = N; g.K = K; g.lda = K; g.ldw = K; g.ldc = N;
    const int ok = gemm_dispatch(g, 1, FLUX_HIP_EPI_F32, (g_force_tile >= 0 ? 1u << g_force_tile : g_tile_mask) & 0x1017FFFu, nullptr, nullptr, nullptr, nullptr, 0, slices);
    *ws = g.ws;
    return ok;
}

/* One launch for the fused projection of a single-stream block, see the header. Never split along K. */
extern "C" int flux_hip_linear_qkv_swiglu(const void *A, const void *W, void *qkv_out, void *mlp_out, int M, int qkv_cols, int mlp, int K,
                                          int lda, int ldw, int ld_qkv, int ld_mlp) {
    if (M <= 0) return 1;
    if (K <= 0 || (K & 63)) return flux_hip_fail("flux_hip_linear_qkv_swiglu: K=%d must be a positive multiple of 64", K);
    if (qkv_cols <= 0 || (qkv_cols & 127) || mlp <= 0 || (mlp & 63))
        return flux_hip_fail("flux_hip_linear_qkv_swiglu: qkv_cols=%d must be a multiple of 128, mlp=%d of 64", qkv_cols, mlp);
    if (lda < K || ldw < K || (lda & 7) || (ldw & 7) || (ld_qkv & 3) || (ld_mlp & 3))
        return flux_hip_fail("flux_hip_linear_qkv_swiglu: bad leading dimensions");
    if (!A || !W || !qkv_out || !mlp_out) return flux_hip_fail("flux_hip_linear_qkv_swiglu: NULL operand");
    if ((((uintptr_t)A | (uintptr_t)W) & 15) || (((uintptr_t)qkv_out | (uintptr_t)mlp_out) & 7))
        return flux_hip_fail("flux_hip_linear_qkv_swiglu: operands must be 16-byte aligned (outputs 8-byte)");
    GemmArgs g = {};
    g.A[0] = (const bf16 *)A; g.W[0] = (const bf16 *)W; g.C[0] = qkv_out; g.C2 = mlp_out; g.M[0] = M;
    g.N = qkv_cols + 2 * mlp; g.K = K; g.lda = lda; g.ldw = ldw; g.ldc = ld_qkv; g.ldc2 = ld_mlp;
    g.w_row0 = 0; g.w_row1 = qkv_cols; g.w_row2 = qkv_cols + mlp; g.nq_cols = qkv_cols;
    int tile = -1;
    const int saved = g_splitk_enabled;
    g_splitk_enabled = 0;
    const int ok = gemm_dispatch(g, 1, EPI_QKV_SWIGLU, (g_force_tile >= 0 ? 1u << g_force_tile : g_tile_mask) & 0x17F7FFFu, &tile);
    g_splitk_enabled = saved;
    return ok;
}

/* flux_hip_linear for callers that must not allocate: the partial sums of the K slices go to the
 * static device array above. Nothing here or below it calls hipMalloc, hipFree or an allocating
 * library routine. Every partial sum the second pass reads has been written by the first pass of the
 * same call, so the array needs no clearing between calls; calls that overlap on one GPU (two
 * streams, two host threads) would share it and race. */
extern "C" int flux_hip_linear_static(int epilogue, int nparts, const flux_hip_linear_part *parts,
                                      int N, int K, int lda, int ldw, int ldc, int w_row0, int w_row1) {
    float *ws = static_ws_for_current_device();
    if (!ws) return 0;
    return linear_impl(epilogue, nparts, parts, N, K, lda, ldw, ldc, w_row0, w_row1, nullptr, 0.0f, nullptr, ws, STATIC_WS_BYTES,
                       "flux_hip_linear_static");
}

/* The residual projection, and - when it runs as K slices - the AdaLN of the updated rows in its
 * second pass, see the header. */
extern "C" int flux_hip_linear_resid_adaln(int nparts, const flux_hip_linear_part *parts, int N, int K, int lda, int ldw, int ldc,
                                           const flux_hip_adaln_part *norm, float eps, int *fused) {
    if (!fused) return flux_hip_fail("flux_hip_linear_resid_adaln: fused must not be NULL");
    *fused = 0;
    if (norm) {
        if (N > 4096) return flux_hip_fail("flux_hip_linear_resid_adaln: N=%d (at most 4096 columns per row)", N);
        for (int i = 0; i < nparts && i < GEMM_MAX_PARTS; i++)
            if (parts[i].M > 0 && (!norm[i].out_bf16 || !norm[i].scale || (!norm[i].shift) != (!norm[0].shift) ||
                                   (((uintptr_t)norm[i].out_bf16 | (uintptr_t)norm[i].shift | (uintptr_t)norm[i].scale) & 15)))
                return flux_hip_fail("flux_hip_linear_resid_adaln: NULL or unaligned norm operand (shift must be given for all parts or for none)");
    }
    return linear_impl(FLUX_HIP_EPI_RESID, nparts, parts, N, K, lda, ldw, ldc, 0, 0, norm, eps, fused);
}



/* Tiles of a convolution: 15 = conv.hip's kernel for 3x3 without stride; ids 0 to 3 as above (64 x 128, 128 x 128, 256 x 256, 64 x 64), 12 = 256 x 128, 13 =
 * 128 x 128 in the ring kernel, as is 2: 128 x 128 in two stages reached 700 to 870 TFLOP/s on 3x3 layers of 128 to 512 channels over
 * 128 x 128 to 1024 x 1024 positions, 256 x 128 reaches 920 to 1230 and 256 x 256 1200 to 1390 (bf16 output). */
#define CONV_PATCH 15 /* 16 x 16 positions x 128 channels, conv.hip */
#define CONV_RUN 14   /* 128 consecutive positions x 64 channels, convp_kernel */
/* LDS rows that the largest neighbourhood of 128 consecutive positions takes, see convp_kernel */
static int convp_rows(int width) {
    const int run = 128 + 2 * ((127 + width - 1) / width) + 2, one = run + 2 * (width + 2);
    return one <= 448 ? one : run <= CONVP_BAND ? 3 * CONVP_BAND : 1 << 30;
}
template <int NPL, int EPI>
static int launch_convp(GemmArgs &g) {
    constexpr int LDS = ConvP<NPL>::LDS;
    static bool attr_done = false;
    auto kern = convp_kernel<NPL, EPI>;
    if (!attr_done) {
        HIP_OK(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, LDS));
        attr_done = true;
    }
    set_row_tiles(g, 128);
    g.ntiles = g.N / 64;
    g.total_tiles = g.mtiles * g.ntiles;
    g.vgrid = (g.total_tiles * g.ksplit + 7) & ~7;
    hipLaunchKernelGGL(kern, dim3(g.vgrid), dim3(256), LDS, flux_hip_stream_handle(), g);
    HIP_OK(hipGetLastError());
    return 1;
}

template <int EPI>
static int conv_tile_launch(GemmArgs &g, int tile) {
    if (tile == CONV_RUN) {
        const int rows = convp_rows(g.conv_wp - 2);
        return rows <= 224 ? launch_convp<7, EPI>(g) : rows <= 320 ? launch_convp<10, EPI>(g) : launch_convp<14, EPI>(g);
    }
    switch (tile) {
        case 2: return launch_4d<8, 8, EPI, 2, 3>(g);
        case 12: return launch_4d<8, 4, EPI, 3, 3>(g);
        case 13: return launch_4d<4, 4, EPI, 3, 3>(g);
        case 1: return launch_cfg<128, 128, 2, 2, EPI>(g);
        case 3: return launch_cfg<64, 64, 2, 2, EPI>(g);
        default: return launch_cfg<64, 128, 2, 2, EPI>(g);
    }
}

#define CONV_TILES 16
static const int conv_bm[CONV_TILES] = {64, 128, 256, 64, 0, 0, 0, 0, 0, 0, 0, 0, 256, 128, 128, 256}, conv_bn[CONV_TILES] = {128, 128, 256, 64, 0, 0, 0, 0, 0, 0, 0, 0, 128, 128, 64, 128};

template <int EPI>
static int conv_finish(GemmArgs &g) {
    hipLaunchKernelGGL(conv_finish_kernel<EPI>, dim3((g.conv_rows + 31) / 32, g.N / 64), dim3(256), 0, flux_hip_stream_handle(), g);
    HIP_OK(hipGetLastError());
    return 1;
}

/* Tile and K split of a convolution by the same kind of model as gemm_dispatch's: rounds of workgroups, each a tile's time at
 * its measured rate plus the bytes of its epilogue at a compute unit's share of the memory rate (nothing overlaps those where one
 * workgroup owns the unit). K slices add a second pass and its partial sums; images that leave most units idle take them. 512 -> 512 channels with residual, us between events, operands
 * from the memory-side cache: 16 x 16 positions are 16 run tiles in one piece, 20.1, in four slices 15.6; 32 x 32 20.4, 18.6 in two and 19.2 in four (128 x 128 tiles 36 and
 * 23 in four); at 56 x 56 one piece wins, 22.3 against 30.2. conv.hip's kernel is ahead from about a round of its tiles on (96 x 96: 57.7, 59.4 of
 * 256 x 128; 88 x 136 60.4 and 61.9) as long as the image's sides do not leave a second, nearly empty round (90 x 162: 264 of its tiles, 99.6 us; 228 of
 * 256 x 128, 66.5). */
static int conv_launch(GemmArgs &g, int epilogue, int *stats_rows, void *enlarged = nullptr) {
    static const int occ[CONV_TILES] = {3, 2, 1, 4, 0, 0, 0, 0, 0, 0, 0, 0, 1, 1, 1, 1};
    static const double rate[CONV_TILES] = {2.0e12, 3.3e12, 5.4e12, 1.5e12, 0, 0, 0, 0, 0, 0, 0, 0, 4.8e12, 4.2e12, 5.0e12, 6.2e12}; /* FLOP/s of one CU */
    static const int splits[] = {1, 2, 3, 4, 6, 8, 12, 16};
    const int M = g.M[0], N = g.N, kt_total = g.K >> 6, f = g_force_tile;
    const bool forced = f >= 0 && f < CONV_TILES && conv_bm[f] && N % conv_bn[f] == 0; /* a forced tile that this layer cannot use is ignored */
    const bool ring_ok = g_ring && (size_t)g.conv_rows * (g.conv_stride == 2 ? 4 : 1) * g.lda * 2 < ((size_t)1 << 32) && (size_t)N * g.ldw * 2 < ((size_t)1 << 32) &&
                         (size_t)g.conv_rows * N < ((size_t)1 << 32);
    const int width = g.conv_wp - 2, height = g.conv_wp > 0 ? g.conv_rows / g.conv_wp - 2 : 0;
    const bool patch_ok = g_ring && g.conv_taps == 9 && g.conv_stride == 1 && !g.conv_packed_out && conv3_takes(height, width, g.lda, N);
    const bool run_ok = ring_ok && g.conv_taps == 9 && g.conv_stride == 1 && !g.conv_packed_out && M > 0 && convp_rows(width) <= 448;
    /* Where CONV_RUN in one piece is a round at most, slices take longer against it than the model below has them: over 504 forms of 36 image sizes (8 x 8 to
     * 128 x 128 and 24 x 320 positions) and seven pairs of channel counts the choice takes 0.8 % more than the best of up to 26 forms on average and 9 % at most; without
     * the term for that 1.7 and 16 %, and a decode from a 4 x 4 latent 590 us of convolutions for 569. With more positions the same term took 128 x 128 in one piece where slices of
     * 256 x 128 are faster: 32 x 132 x 512 in a decode 46 us and 37. */
    const bool run_round = run_ok && (long)((M + 127) / 128) * (N / 64) <= 256;
    int tile = -1, split = 1;
    const auto choose = [&](bool slices) {
        double best = 1e30;
        tile = -1;
        split = 1;
        for (int t = 0; t < CONV_TILES; t++) {
            const bool ring = t == 2 || t >= 12;
            if (!conv_bm[t] || N % conv_bn[t] || (forced && t != f)) continue;
            if (t == 0 && !forced) continue; /* (for comparison runs) */
            if (ring && (!ring_ok || kt_total < 4)) continue;
            if (t == CONV_PATCH && !patch_ok) continue;
            const bool run = t == CONV_RUN;
            if (run && !run_ok) continue;
            const long tiles = t == CONV_PATCH ? conv3_tiles(height, width, N) : (long)((M + conv_bm[t] - 1) / conv_bm[t]) * (N / conv_bn[t]);
            for (int sp : splits) {
                /* a slice of runs is whole chunks of channels, two at least (of one it is mostly its first loads: 17.3 us against 15.6 at 16 x 16 x 512) */
                const int unit = run ? 9 : 1;
                const int per = (kt_total / unit + sp - 1) / sp * unit, used = (kt_total + per - 1) / per, last = kt_total - (used - 1) * per;
                if (sp > 1 && (t == CONV_PATCH || !slices || per < 4 || last < 4 || used != sp || N % 64 || (run && per < 18 && !forced))) continue;
                if (slices && g_force_split && kt_total / g_force_split >= 4 && sp != g_force_split) continue;
                const double ws = (double)sp * M * N * 4.0;
                if (sp > 1 && ws > 256e6) continue;
                const long blocks = tiles * sp, slots = 256L * occ[t], rounds = (blocks + slots - 1) / slots;
                if (run && rounds > 2 && !forced) continue; /* (72 x 276 x 512 in five rounds: 98 us, in conv.hip's 16 x 16 tiles 90) */
                const long per_cu = (min(blocks, slots) + 255) / 256;
                double est = rounds * (2.0 * conv_bm[t] * conv_bn[t] * 64.0 * per / (rate[t] / per_cu) + 2.5e-6 +
                                       (double)conv_bm[t] * conv_bn[t] * (sp > 1 ? 0 : (epilogue == FLUX_HIP_EPI_CONV_BF16 ? 2 : 4) + (g.res ? 4 : 0)) / 2.0e10);
                if (t == CONV_PATCH) /* the epilogue lies under the next tile and costs it half of its bytes' time, the last one's all */
                    est = rounds * (2.0 * conv_bm[t] * conv_bn[t] * 64.0 * per / rate[t] + (double)conv_bm[t] * conv_bn[t] * ((epilogue == FLUX_HIP_EPI_CONV_BF16 ? 2 : 4) + (g.res ? 4 : 0)) / 4.0e10) + 6.0e-6;
                if (run) est += 0.5e-6 + (rounds - 1) * 3.5e-6;           /* (a second round's first loads meet the first one's stores) */
                if (sp > 1) est += 4.0e-6 + 2.0 * ws / 4.0e12;
                if (sp > 1 && run_round) est += run ? 1.5e-6 : 3.0e-6;
                if (est < best) { best = est; tile = t; split = sp; }
            }
        }
        if (tile < 0) tile = N % 128 == 0 ? 1 : 3; /* (a forced ring tile that cannot run) */
    };
    choose(g_splitk_enabled);
    if (split > 1 && M > 0 && !workspace_for_slices((size_t)split * M * N * sizeof(float))) choose(false);
    g.kt_per = tile == CONV_RUN ? (kt_total / 9 + split - 1) / split * 9 : (kt_total + split - 1) / split;
    g.ksplit = M == 0 ? 0 : split; /* 0: nothing but border */
    const bool bf = epilogue == FLUX_HIP_EPI_CONV_BF16;
    if (g.ksplit > 1) {
        g.ws = g_ws;
        g.ws_rows = M;
    }
    const bool direct = g.ksplit == 1 && tile == CONV_PATCH;
    if (enlarged && !direct) {
        if (!flux_hip_vae_upsample2x_bf16(enlarged, g.A[0], height / 2 + 2, width / 2 + 2, g.lda)) return 0;
        g.A[0] = (const bf16 *)enlarged;
    }
    /* one record per convolution: K slices and their second pass together */
    const int slot = conv_probe_begin(epilogue, tile);
    int ok = 1;
    if (direct) {
        ok = conv3_launch(!bf, enlarged != nullptr, g.A[0], g.W[0], g.bias, g.res, g.C[0], height, width, g.lda, N, g.stats, stats_rows, compute_units() & ~7);
    } else if (g.ksplit == 1) {
        if (stats_rows) *stats_rows = 2 * ((M + conv_bm[tile] - 1) / conv_bm[tile]);
        ok = bf ? conv_tile_launch<FLUX_HIP_EPI_CONV_BF16>(g, tile) : conv_tile_launch<FLUX_HIP_EPI_CONV_F32>(g, tile);
    } else {
        if (stats_rows) *stats_rows = (g.conv_rows + 31) / 32;
        if (g.ksplit > 1) ok = conv_tile_launch<EPI_CONV_PARTIAL>(g, tile);
        ok = ok && (bf ? conv_finish<FLUX_HIP_EPI_CONV_BF16>(g) : conv_finish<FLUX_HIP_EPI_CONV_F32>(g));
    }
    conv_probe_end(slot);
    return ok;
}

extern "C" int flux_hip_conv_image(int epilogue, const void *in, int in_wp, int packed, const void *w, const float *bias, const float *res, void *out,
                                   int rows, int wp, int cin, int cout, int taps, float *stats, int *stats_rows);

/* Convolution over a zero-bordered channels-last image as one GEMM, see the header. */
extern "C" int flux_hip_conv_stats(int epilogue, const void *in, const void *w, const float *bias, const float *res, void *out, int rows,
                                   int wp, int cin, int cout, int taps, float *stats, int *stats_rows);

extern "C" int flux_hip_conv(int epilogue, const void *in, const void *w, const float *bias, const float *res,
                             void *out, int rows, int wp, int cin, int cout, int taps) {
    return flux_hip_conv_stats(epilogue, in, w, bias, res, out, rows, wp, cin, cout, taps, nullptr, nullptr);
}

static GemmArgs conv_args(const void *in, const void *w, void *out, int rows, int wp, int cin, int cout, int taps) {
    GemmArgs g = {};
    g.A[0] = (const bf16 *)in;
    g.W[0] = (const bf16 *)w;
    g.C[0] = out;
    g.N = cout; g.K = taps * cin; g.lda = cin; g.ldw = taps * cin; g.ldc = cout;
    g.conv_taps = taps; g.conv_wp = wp; g.conv_rows = rows;
    g.M[0] = rows;
    if (wp > 0) {
        g.M[0] = wp > 2 && rows / wp > 2 ? (rows / wp - 2) * (wp - 2) : 0;
        g.conv_magic = wp > 2 ? 0xFFFFFFFFu / (unsigned)(wp - 2) : 0;
    }
    return g;
}

/* The same, and (stats != NULL) the sums for the group norm that follows, see the header. */
extern "C" int flux_hip_conv_stats(int epilogue, const void *in, const void *w, const float *bias, const float *res, void *out, int rows,
                                   int wp, int cin, int cout, int taps, float *stats, int *stats_rows) {
    if (epilogue != FLUX_HIP_EPI_CONV_BF16 && epilogue != FLUX_HIP_EPI_CONV_F32)
        return flux_hip_fail("flux_hip_conv: epilogue %d is not a convolution epilogue", epilogue);
    if (taps != 1 && taps != 9) return flux_hip_fail("flux_hip_conv: taps=%d (1 or 9)", taps);
    if (rows <= 0 || cin <= 0 || (cin & 63) || cout <= 0 || (cout & 63))
        return flux_hip_fail("flux_hip_conv: rows=%d cin=%d cout=%d (channels must be multiples of 64)", rows, cin, cout);
    if (taps == 9 && (wp < 3 || rows % wp || rows / wp < 3 || cin > 64 * 227))
        return flux_hip_fail("flux_hip_conv: a 3x3 convolution needs a bordered image (rows=%d wp=%d cin=%d)", rows, wp, cin);
    if (wp > 0 && rows % wp) return flux_hip_fail("flux_hip_conv: rows=%d is not a multiple of the image width %d", rows, wp);
    if (!in || !w || !bias || !out) return flux_hip_fail("flux_hip_conv: NULL operand");
    if ((((uintptr_t)in | (uintptr_t)w | (uintptr_t)bias | (uintptr_t)res | (uintptr_t)out) & 15))
        return flux_hip_fail("flux_hip_conv: operands must be 16-byte aligned");
    if (res && epilogue != FLUX_HIP_EPI_CONV_F32) return flux_hip_fail("flux_hip_conv: only the fp32 epilogue adds a residual");
    return flux_hip_conv_image(epilogue, in, 0, 0, w, bias, res, out, rows, wp, cin, cout, taps, stats, stats_rows);
}

/* flux_hip_conv_stats to fp32 over the nearest-neighbour 2x enlargement of the bordered image `in`; rows and wp are the enlargement's. conv.hip's kernel
 * reads the source in place of it; for the tiles of smaller images it is written to `enlarged` first. Writing it took 104 us at 1024 x 1024 x 256, 53
 * at 512 x 512 x 512 and 14 at 256 x 256 x 512, and the convolution read four times the bytes. */
extern "C" int flux_hip_conv_enlarged(const void *in, void *enlarged, const void *w, const float *bias, float *out, int rows, int wp, int cin, int cout,
                                      float *stats, int *stats_rows) {
    if (!in || !enlarged || !w || !bias || !out || wp < 4 || rows % wp || rows / wp < 4 || ((rows / wp | wp) & 1) || cin <= 0 || cin & 63 || cout <= 0 || cout & 63)
        return flux_hip_fail("flux_hip_conv_enlarged: bad argument (rows=%d wp=%d cin=%d cout=%d)", rows, wp, cin, cout);
    if ((((uintptr_t)in | (uintptr_t)enlarged | (uintptr_t)w | (uintptr_t)bias | (uintptr_t)out) & 15) || (stats && (!stats_rows || ((uintptr_t)stats & 7))))
        return flux_hip_fail("flux_hip_conv_enlarged: unaligned operand");
    GemmArgs g = conv_args(in, w, out, rows, wp, cin, cout, 9);
    g.conv_stride = 1; g.conv_in_wp = wp;
    g.bias = bias; g.stats = stats;
    return conv_launch(g, FLUX_HIP_EPI_CONV_F32, stats_rows, enlarged);
}

/* flux_hip_conv_stats without its argument checks, for the VAE's own layers: the bf16 output takes a residual as well, and
 * in_wp > 0 makes it the stride-2 3x3 convolution of a bordered image in_wp wide, rows and wp being the output's. For 1x1
 * convolutions without residual or statistics on that side, packed & 1: `in`, packed & 2: `out` hold the (rows / wp - 2) * (wp - 2)
 * interior positions only. */
extern "C" int flux_hip_conv_image(int epilogue, const void *in, int in_wp, int packed, const void *w, const float *bias, const float *res, void *out,
                                   int rows, int wp, int cin, int cout, int taps, float *stats, int *stats_rows) {
    GemmArgs g = conv_args(in, w, out, rows, wp, cin, cout, taps);
    g.conv_packed_out = packed >> 1 & 1;
    g.conv_stride = packed & 1 ? 0 : in_wp > 0 ? 2 : 1; g.conv_in_wp = in_wp > 0 ? in_wp : wp;
    g.bias = bias; g.res = res; g.stats = stats;
    if (stats && (!stats_rows || ((uintptr_t)stats & 7))) return flux_hip_fail("flux_hip_conv_stats: stats needs stats_rows and 8-byte alignment");
    return conv_launch(g, epilogue, stats_rows);
}
