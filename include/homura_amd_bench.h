/* Measurement and test-support entry points of libhomura_amd.so. They are not part of the drop-in
 * boundary (include/homura_amd.h): nothing here has a counterpart in the reference's FFI. */
#ifndef HOMURA_AMD_BENCH_H
#define HOMURA_AMD_BENCH_H

#include "homura_amd.h"

#ifdef __cplusplus
extern "C" {
#endif
#pragma GCC visibility push(default)

/* Timed decode for benchmarking: runs `n_steps` decode steps starting from token `first_id`
 * (greedy feedback on device), returns total milliseconds measured with HIP events on the
 * context stream. */
int hm_model_bench_decode(hm_model *m, int64_t first_id, int n_steps, float *ms_out,
                          int32_t *h_tokens_out);

/* Per-kernel profile of one decode step (HOMURA_PROFILE analogue, reference
 * src/runtime.rs:1849-1873): HIP events around every device launch; one record per device
 * kernel name. Fills up to `cap` records; returns the number written. */
typedef struct {
    char label[32]; /* "gemv_bf16[qkv]", "gqa_decode_attn", "gemv_bf16[lm_head+argmax]", ... */
    float ms;       /* summed over the launches */
    int launches;
    double bytes;   /* algorithmic bytes moved by these launches */
} hm_kernel_profile;
int hm_model_profile_step(hm_model *m, int64_t token_id, hm_kernel_profile *out, int cap);
/* Roofline timing: per device kernel name, all of the step's launches of that kernel (one per
 * layer, different weights each) back to back, `rounds` times, between two HIP events.
 * Disturbs activations and the current cache row: call after the decode. */
int hm_model_time_kernels(hm_model *m, int rounds, hm_kernel_profile *out, int cap);

/* ── deterministic synthetic data (host side, no GPU needed) ─────────────────
 * Counter-based generator shared by tests and benchmarks: sample i of stream `seed` uses
 * outputs 3i..3i+2 of the splitmix64 sequence seeded with `seed`; a normal variate is the
 * centred sum of the twelve 16-bit fields of those outputs (Irwin-Hall, unit variance),
 * computed in integers so that every platform produces the same bits. */
void hm_synth_normal_f32(uint64_t seed, uint64_t first, size_t n, float scale, float *out);
void hm_synth_normal_bf16(uint64_t seed, uint64_t first, size_t n, float scale, uint16_t *out);
void hm_synth_token_ids(uint64_t seed, size_t n, int vocab, int64_t *out);
/* n_blocks Q8_0 blocks: q uniform in [-127,127], d = f16(|N(0,1)| * d_scale) */
void hm_synth_q8_0(uint64_t seed, size_t n_blocks, float d_scale, uint8_t *out);
/* n_blocks Q4_0 blocks: nibbles uniform in [0,15], d = f16(|N(0,1)| * d_scale) */
void hm_synth_q4_0(uint64_t seed, size_t n_blocks, float d_scale, uint8_t *out);

/* Floor of a step made of dependent launches: a HIP graph of `n_kernels` one-wavefront kernels that do
 * nothing (chained = 0) or that each read 4 bytes their predecessor wrote and write 4 bytes (chained = 1),
 * replayed `replays` times between two events; microseconds per replay. */
int hm_bench_launch_floor(hm_ctx *ctx, int n_kernels, int chained, int replays, float *us_per_replay);

/* Test support: writes `word` over the whole LDS of every CU (a grid of workgroups that each take a CU's LDS).
 * LDS keeps its contents from one kernel to the next, and from one process to the next: a kernel that reads
 * LDS it did not write works or fails by what ran before it. Filled with 0xFFFFFFFF (a NaN), any such read
 * that reaches a result shows. Device allocations can be pre-filled the same way with the environment
 * variable HOMURA_ALLOC_FILL=<byte>, read when the first buffer is allocated. */
int hm_test_fill_lds(hm_ctx *ctx, uint32_t word);

/* Test support: the floats that the prompt pass sets aside for the product of up to `rows` rows with an [n][k] matrix of a
 * weight format on a chip of `cus` CUs, and the most that the product of m <= rows rows writes (all its K slices). Host only. */
int hm_test_prompt_product(int hm_dtype, int rows, int m, int k, int n, int cus, long long *floats_held, long long *floats_written);

/* Test support: a group of splits that folds on its die (die_fold.h) finds one arrival from each of two dies that were not there. */
int hm_test_die_arrivals(hm_ctx *ctx, int group);
/* Test support: counts[3] of what went which way in this context so far: attention launches whose splits fold on their die; gate rows of scans and
 * recurrences (layers of a prompt's portions) straight from their projection, and through the convolution. */
int hm_test_routes(hm_ctx *ctx, long long *counts);

/* Test support: the rows that the decode attention's grid covers in a step of `live` live rows over a cache of max_len, the rows of a split, and
 * the rows that its splits ask for without having looked at the live length. Host only. */
int hm_test_attn_rows(int live, int max_len, int *span, int *chunk, int *sure);

/* Test support: the tile and K slices (at most max_parts) of a product of gemm_tiles_mfma.hip on a chip of `cus` CUs; the few-rows kernel's
 * tile of 32 or 64 rows by 32 or 64 columns where that takes it. kind 0: two f16 pieces with column factors, 1: with block scales, 2: one bf16 piece.
 * k a multiple of 64. Host only. */
int hm_test_product_tiles(int kind, int m, int k, int n, int cus, int max_parts, int *tile_m, int *tile_n, int *slices);

/* Test support: one product of the prompt pass with the row kernel ahead of it. front 0: x [m][k] f32 through RMSNorm (weights norm_w
 * [k], eps 1e-6); front 1: x [m][2 k] f32 as (gate, up) pairs through SiLU(gate) * up; front 2: x [m][k] bf16 rows as one piece. w: bf16
 * rows [n][k], or the raw blocks of Q8_0 / Q4_0. half 0: three bf16 pieces, 1: two f16 pieces (HM_ERR_STATE where the weights do not take
 * that). All pointers are device memory. The result comes as *parts <= 8 slices out [parts][m][n] to be added, row r then times
 * row_factor[r]. */
int hm_test_prompt_rows(hm_ctx *ctx, int front, const void *x, const float *norm_w, int dtype, const void *w, int half, int m, int k,
                        int n, float *out, float *row_factor, int *parts);

/* Test support: the gate|up product of the prompt pass and its gated rows with column factors: x [m][k] f32 through RMSNorm (norm_w [k], eps
 * 1e-6), w [2 inter][k] bf16 rows or Q8_0 / Q4_0 blocks as (gate, up) pairs of rows. fused 1: the product's workgroups write the rows, 0: its
 * slices go through the row kernel. out [m][2][inter] f16 pieces of silu(gate) up times scale [inter]. *pays: what the prompt pass would take. */
int hm_test_gated_rows(hm_ctx *ctx, const void *x, const float *norm_w, int dtype, const void *w, int fused, int m, int k, int inter,
                       uint16_t *out, float *scale, int *pays);

/* Test support: those rows through the down product: down [k][inter], the same dtype (inter a multiple of 64), out [m][k] f32. */
int hm_test_gated_down(hm_ctx *ctx, const void *x, const float *norm_w, int dtype, const void *w, const void *down, int fused, int m, int k,
                       int inter, float *out);

/* Test support: the q|k|v projection of the prompt pass in f16 pieces and its tail: x [S][k] f32 through RMSNorm (norm_w [k], eps), w
 * [(H + 2 kvh) hd][k] bf16 rows or Q8_0 / Q4_0 blocks; bias, and qw with kw, may be NULL. fused 1: the product's workgroups do the tail, 0: its slices go
 * through the row kernel. q [S][(H + 2 kvh) hd] (its q columns), caches [kvh][max_len][hd] rows past .. *pays: what the prompt pass would take. */
int hm_test_qkv_product(hm_ctx *ctx, const void *x, const float *norm_w, int dtype, const void *w, int fused, int S, int k, int H, int kvh, int hd,
                        const float *bias, const float *qw, const float *kw, const float *cos, const float *sin, float *q, uint16_t *kcache,
                        uint16_t *vcache, int max_len, int past, float eps, int *pays);

/* Test support: the latents' rows of a prompt: down [parts][n][ld] f32 (q latent, padded to a multiple of 32 | kv latent | rotated key), norms, tables
 * [past + n][rot], to q_split [n][pieces * q_rank padded] and ring [past + n][pieces * (rank padded + rot padded)]. Rows that are no
 * whole vectors (an odd ld) take the kernel of a workgroup a row. */
int hm_test_latent_rows(hm_ctx *ctx, const float *down, int ld, int parts, const float *q_norm, const float *kv_norm, const float *cos_tab,
                        const float *sin_tab, int q_rank, int rank, int rot, int pieces, int n, int past, float eps, uint16_t *q_split, uint16_t *ring);

/* Test support: a gate|up product of one bf16 piece with its activation, a [m][k], b [n][k] as (gate, up) pairs of rows, out [m][n / 2] bf16; kind 0
 * silu(g) u, 1 the clamped sigmoid gate. *pays: whether the prompt pass of a list-of-layers model would take it. */
int hm_test_gated_product(hm_ctx *ctx, const uint16_t *a, const uint16_t *b, uint16_t *out, int m, int k, int n, int kind, float limit, float slope,
                          int *pays);

/* Test support: the bytes of f16 weight copies that a transformer's prompt pass holds, and how many of its groups of projections
 * (q|k|v, o, gate|up, down of every layer) multiply with them. */
int hm_test_prefill_f16_copies(hm_model *m, size_t *bytes, int *groups);

/* Test support: the tail of the prompt pass's q|k|v projection for S rows [S][(H + 2 kvh) * hd] at positions past ..: q rotated in
 * place, k and v into caches [kvh][max_len][hd]. d_qw and d_kw [hd], or both NULL. hd 64 or 128. */
int hm_test_qkv_tail(hm_ctx *ctx, float *d_qkv, const float *d_qw, const float *d_kw, const float *d_cos, const float *d_sin,
                     uint16_t *d_kcache, uint16_t *d_vcache, int S, int H, int kvh, int hd, int max_len, int past, float eps);

/* Phase trace of the latest whole-step decode launch: device-clock ticks (100 MHz) taken by workgroup
 * 0 at 11 points per layer (both workgroup barriers of the Q|K|V, attention, O, gate|up and down
 * phases; the end of the fold follows attention's second barrier) and one at the end of the kernel, then
 * a word that is 1 when the step found its workgroups dealt round-robin to the dies and used die-local
 * exchanges. The first call switches recording on and stores 0 in *n_out; later calls copy
 * layers * 11 + 2 entries of the step that ran last (workgroup 0's), or, when cap has room for 256
 * times as many, one such row per workgroup (256 rows; those of workgroups the grid lacks stay 0). */
int hm_model_whole_step_trace(hm_model *m, unsigned long long *h_out, int cap, int *n_out);

/* Test support for block-quantised models with K-quant projections: keep the f32 activation rows that the
 * prompt pass hands to the Q8_K quantiser (reference emit_quant.rs:422-466) for the next `rows` cache
 * positions (0 = stop, free the buffer), and copy them to the host afterwards. Per layer: [rows][hidden]
 * (input of q|k|v), [rows][heads * head_dim] (o), [rows][hidden] (gate|up), [rows][intermediate] (down);
 * rows of groups whose matrices are not K-quants stay zero. A checker can then quantise the very values
 * the GPU quantised, so that a rounding decision taken differently on the two sides is counted instead of
 * being seen as an error. */
int hm_model_prefill_capture_q8k_inputs(hm_model *m, int rows);
int hm_model_prefill_captured_q8k_inputs(hm_model *m, float *h_out, size_t n_floats);

/* Test support for list-of-layers models: keep the residual rows behind every layer run (one entry per pass where
 * layers are looped) of the prompt-pass chunks from now on, and copy out those of the latest chunk, [runs][rows][width]. */
int hm_model_capture_residuals(hm_model *m, int on);
int hm_model_captured_residuals(hm_model *m, float *h_out, size_t n_floats);

#pragma GCC visibility pop
#ifdef __cplusplus
}
#endif
#endif
