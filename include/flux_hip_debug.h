/*
 * flux_hip_debug.h - test and measurement switches of libflux_hip.so.
 *
 * None of these has a counterpart in the reference and none is needed to use the library; an
 * application includes flux_hip.h only. They are process-wide mutable state (like the reference's
 * own globals, flux_kernels.c:32-45): set one, run, and restore the default. tests/conftest.py
 * restores all of them before every test module.
 */
#ifndef FLUX_HIP_DEBUG_H
#define FLUX_HIP_DEBUG_H

#include "flux_hip.h"

#ifdef __cplusplus
extern "C" {
#endif

/* force_tile: 0/1/2/3/5/6/7 pins the GEMM tile of flux_hip_linear (64x128, 128x128, 256x256, 64x64,
 * 288x192, 192x192, 256x192; 4 = 256x256 in its 8-wave form, never chosen automatically; 8 / 16 / 10 / 9 / 24 = 80 / 96 / 112 /
 * 128 / 144 columns for row ranges of at most 128 rows, whose last column tile is cut off at N and whose ring is 6 / 5 / 5 / 5 / 4
 * LDS stages; 11 = 256x224, whose last column
 * tile is cut off at N: for the residual and bf16 epilogues with at least four 64-wide K steps and no K slices; 12 / 13 / 14 =
 * 256x128 / 128x128 / 192x256 in the ring kernel, at least four K steps; 17 to 22 = 288x288, 384x224, 320x224, 320x256, 288x256,
 * 352x224 for the fused [Q|K|V|gate|up] launch alone, at least four K steps; 23 = 256x160 in the ring kernel for the SwiGLU epilogue
 * alone, whose last column tile is cut off at N, a multiple of 64, at least four K steps), -1
 * restores the automatic choice (a tile that cuts no columns off and whose width does not divide N is skipped; if none is left the
 * 128x128 tile runs). Convolutions know tiles 0 to 3, 12, 13, 14 (128 consecutive positions x 64 channels, their neighbourhood in LDS:
 * 3x3 without stride; K slices of whole 64-channel chunks) and 15 (16x16 positions x 128 channels, likewise, at least 128 input channels) and
 * ignore one that does not fit the layer. */
void flux_hip_linear_force_tile(int tile);
/* bit t set = the automatic choice may use tile t (default 0x1FF7FEF: all but tile 4; 0 restores it) */
void flux_hip_linear_tile_mask(unsigned mask);
/* 0 turns the split-K path off (default 1) */
void flux_hip_linear_enable_splitk(int on);
/* slices > 1: projections whose epilogue and K length allow it run as exactly that many K slices (one of 2, 3, 4, 6,
 * 8, 12, 16, 24, 32; at least four 64-wide K steps per slice), whatever the cost model would choose; 0 (default):
 * the cost model chooses. With flux_hip_linear_static a demanded number of slices whose partial sums do not fit the
 * static workspace is refused. */
void flux_hip_linear_force_split(int slices);
/* 1 (default): the 4-wave GEMM launches at most one workgroup per compute unit and each walks several
 * tiles; 0: one workgroup per tile */
void flux_hip_linear_persistent(int on);
/* 1 (default): the 4-wave tiles run as gemm4d_kernel (operand rings of two or three LDS slots, count-based waits at
 * the barrier); 0: as gemm4w_kernel (two stages, everything in flight awaited at the barrier). Bit-identical results. */
void flux_hip_linear_ring(int on);
/* attention kernel: -1 and 15 = automatic (default: 64-query waves, block lengths chosen per sequence length);
 * 0 / 1 = the 32-query-per-wave kernel with 128 / 256 queries per workgroup; 11..14 = 16, 32, 48, 64 queries per wave
 * throughout */
void flux_hip_attention_force_variant(int v);
/* 1 (default): a CFG step runs its two forwards as one batch of two sequences; 0: one after the other.
 * Takes effect at the next flux_hip_session_begin. */
void flux_hip_set_batched_cfg(int on);
/* The fused projection of a single-stream block: 1 (default) = one launch (flux_hip_linear_qkv_swiglu), 0 = two
 * (QKV, then gate/up). */
void flux_hip_set_fused_qkv_mlp(int on);
/* VAE attention: at most `rows` query rows per chunk (0 = default: 512 MB of bf16 probabilities per chunk). */
void flux_hip_vae_set_attention_chunk(int rows);

/* Launch probe: probe(epilogue) records HIP events around every later flux_hip_linear launch with
 * that epilogue (-2: every convolution, K slices and their second pass as one; -1 stops); probe_read waits for them and returns
 * their count and summed duration, probe_read_tile the same for the launches that used one tile id,
 * probe_read_launches copies out, in launch order, the tile id and duration (ms) of up to `max`
 * recorded launches and returns their number (-1 on error). */
int flux_hip_linear_probe(int epilogue);
int flux_hip_linear_probe_read(int *launches, float *total_ms);
int flux_hip_linear_probe_read_tile(int tile, int *launches, float *total_ms);
int flux_hip_linear_probe_read_launches(int max, int *tiles, float *ms);

/* What the matrix pipes sustain on their own: a register-resident loop of independent bf16 MFMAs on every
 * compute unit (one workgroup each, waves_per_simd = 1 or 2 waves per SIMD; `iters` x 16 MFMAs per wave),
 * run launches + 1 times; the best launch's rate in TFLOP/s goes to *tflops. shape 0 =
 * v_mfma_f32_16x16x32_bf16, 1 = v_mfma_f32_32x32x16_bf16; pattern 0 = all-zero operands, 1 = values in
 * [1, 2) with a random low byte, 2 = random bit patterns. `bench.py --workload mfma_peak` prints the table. */
int flux_hip_mfma_peak(int shape, int pattern, int waves_per_simd, int iters, int launches, float *tflops);
/* What an instruction between a lone wave's MFMAs costs the matrix pipe (csrc/microbench.hip): mode 0 nothing,
 * 1 global_load_lds_dwordx4, 2 ds_read_b128, 3 v_exp_f32, 4 three v_fma_f32, 5 global_load_dwordx4 + ds_write_b128; one
 * such instruction behind every `every`-th MFMA (1, 2, 4, 8, 16). Returns clock cycles per MFMA (16 = no loss) and
 * the core clock of the run. */
int flux_hip_mfma_issue_cost(int mode, int every, int iters, float *cycles_per_mfma, float *ghz);

#ifdef __cplusplus
}
#endif
#endif /* FLUX_HIP_DEBUG_H */
