// Internal launch interface of the MFMA GEMM used by the prefill path.
#pragma once

#include <cstdint>

#include "gated_act.h"
#include "grouped_tiles.h"
#include "hm_common.h"

namespace homura {

// C[M][N] f32 = (sum of the pieces of A)[M][K] x B[N][K]^T. d_a_split is [M][pieces * K] bf16: piece p
// of every f32 activation in columns [p K, (p+1) K) (what the kernels of prefill.hip write). B is the
// K-contiguous stream layout of the model weights. K % 32 == 0, pieces 1..3.
// With parts != NULL the product may be cut along K into up to max_parts slices when M x N alone
// leaves most of the chip idle: slice s lands in d_c + s * M * N, *parts says how many there are, and
// the caller adds them up in index order. A product comes in more than one slice only while slices times
// its 128 x 128 tiles stay within gemm_sliced_tiles(): d_c holds M * N floats, and that many tiles at least.
inline long long gemm_sliced_tiles(int cus) { return 2LL * cus; }
int gemm_split_nk(hm_ctx *ctx, const uint16_t *d_a_split, int pieces, const uint16_t *d_b_nk, float *d_c, int M, int K,
                  int N, int max_parts = 1, int *parts = nullptr);

// The same sum of piece products against B in the reference's layout [K][N] (N contiguous; N % 8 == 0, K % 32 == 0).
int gemm_split_kn(hm_ctx *ctx, const uint16_t *d_a_split, int pieces, const uint16_t *d_b_kn, float *d_c, int M, int K,
                  int N);

// C = A x B^T for two f32 matrices, each given as three bf16 pieces per element: d_a_split [M][3 K],
// d_b_split [N][3 K] (piece p in columns [p K, (p+1) K)). The six products of an A piece and a B piece
// whose indices add up to at most 2 are accumulated; what is left out is below 2^-24 of the result.
// K % 64 == 0. Row r of C starts at d_c + r * ldc (ldc = 0: N); slices as in gemm_split_nk, slice s at
// d_c + s * M * ldc.
int gemm_split_split_nk(hm_ctx *ctx, const uint16_t *d_a_split, const uint16_t *d_b_split, float *d_c, int M, int K,
                        int N, int max_parts = 1, int *parts = nullptr, int ldc = 0);

// The same products with every tile loaded once (gemm_pieces_mfma.hip): a_pieces x b_pieces = 2 x 1 or 3 x 1
// (d_b_split is then the plain [N][K] bf16 matrix) or 3 x 3. K % 32 == 0. Slices and ldc as above.
int gemm_pieces_nk(hm_ctx *ctx, const uint16_t *d_a_split, int a_pieces, const uint16_t *d_b_split, int b_pieces,
                   float *d_c, int M, int K, int N, int max_parts = 1, int *parts = nullptr, int ldc = 0);

// A batch of 3 x 1 products of one shape (block-diagonal matrices): problem z reads d_a_split + z * a_batch ([M][3 K])
// and d_b_nk + z * b_batch ([N][K]), writes row r at d_c + z * c_batch + r * ldc. K % 32 == 0.
int gemm_pieces_batched(hm_ctx *ctx, const uint16_t *d_a_split, size_t a_batch, const uint16_t *d_b_nk, size_t b_batch,
                        float *d_c, size_t c_batch, int batch, int M, int K, int N, int ldc);

// Products of one B [N][K] per group (a mixture of experts) over the rows that the groups' lists name: d_list
// [groups][list_cap] entries, d_count [groups], `entries` of them in all. Entry e reads row e % a_rows of the split matrix
// and writes row e of d_c [.][N]. 1 or 3 pieces; K % 32 == 0.
// With act (gemm_gated_fits): neighbouring columns are (gate, up) pairs, and act(w gate, w up) with the entry's weight w
// leaves as bf16, d_c being [.][N / 2] of them.
// (gemm_grouped_dma: the same for one piece and K % 64 == 0, behind gemm_grouped_nk's checks.)
inline bool gemm_gated_fits(int pieces, int K, int N) { return pieces == 1 && K % 64 == 0 && N % 4 == 0; }
int gemm_grouped_dma(hm_ctx *ctx, const uint16_t *d_a, const uint16_t *d_b_nk, float *d_c, const GroupLists &lists, unsigned tiles,
                     int K, int N, const GatedAct *act, const float *d_weight);
int gemm_grouped_nk(hm_ctx *ctx, const uint16_t *d_a_split, int pieces, int a_rows, const uint16_t *d_b_nk, float *d_c,
                    const int *d_list, const int *d_count, int groups, int list_cap, int entries, int K, int N,
                    const GatedAct *act = nullptr, const float *d_weight = nullptr);

// 3 x 1 pieces against a block-scaled integer matrix: d_b_ints [N][K] bf16 holds the integers of a Q8_0 / Q4_0
// matrix (exact), d_scales [K / 32][npad] f32 the scale of every 32-wide block of every row (npad >= N rounded
// up to 128). C = sum over blocks of scale * (A x ints^T over the block). Slices and ldc as above.
int gemm_pieces_scaled_nk(hm_ctx *ctx, const uint16_t *d_a_split, const uint16_t *d_b_ints, const float *d_scales, int npad,
                          float *d_c, int M, int K, int N, int max_parts = 1, int *parts = nullptr, int ldc = 0);
// The same products with f16 operands (half_weights.h): two f16 pieces per activation, B [N][K] f16, column n of the result times
// unscale[n]; block-scaled integers (d_scales) carry their factors in the scales, unscale is NULL then, and npad >= half_scale_cols(N). K % 64 == 0.
// (gemm_half_wide: its widest tiles, gemm_pieces_mfma.hip; stages of 32 k)
// gated (gate_scale with it): neighbouring columns are (gate, up) pairs, and silu(gate) up times gate_scale [N / 2] leaves as two f16
// pieces, the second times HALF_LOW (row_pieces.h), gated [M][2 (N / 2)], instead of d_c: one slice, N % 2 == 0. gemm_half_gated_pays: whether that is the quicker way, or slices and
// silu_mul_half_launch behind them.
// low: the second pieces come so, as the gated rows hold them.
// tail (with head_dim 64 or 128): the product is a q|k|v projection of M = tail->S rows, and its workgroups hand their head rows on as
// qkv_post_launch does: q [M][N] at tail->qkv, k and v in the caches, nothing to d_c. One slice. gemm_half_tail_pays as above.
struct QkvPostArgs;
struct HalfProduct {
    const float *unscale;
    const float *gate_scale = nullptr;
    uint16_t *gated = nullptr;
    const QkvPostArgs *tail = nullptr;
    bool low = false;
};
bool gemm_half_tail_pays(bool scaled, int head_dim, int M, int K, int N, int cus, int max_parts);
bool gemm_half_gated_pays(bool scaled, int M, int K, int N, int cus, int max_parts);
int gemm_half_nk(hm_ctx *ctx, const uint16_t *d_a_half, const uint16_t *d_b_half, const HalfProduct &half, const float *d_scales,
                 int npad, float *d_c, int M, int K, int N, int max_parts = 1, int *parts = nullptr);
inline int half_scale_cols(int N) { return (N + 191) / 192 * 192 > (N + 127) / 128 * 128 ? (N + 191) / 192 * 192 : (N + 127) / 128 * 128; }
int gemm_half_wide(hm_ctx *ctx, const uint16_t *d_a_half, const uint16_t *d_b_half, const HalfProduct &half, float *d_c, int M, int K, int N,
                   int slices, int stages_per_split);
// One bf16 piece by the same kernel (its operands checked by the caller: 16-byte aligned, K % 64 == 0)
// gemm_tiles_square: its choice is one slice of 128 x 128 tiles, which gemm_dma_kernel (gemm_bf16_mfma.hip) multiplies faster
bool gemm_tiles_square(int M, int K, int N, int cus, int max_parts);
int gemm_tiles_bf16(hm_ctx *ctx, const uint16_t *d_a, const uint16_t *d_b_nk, float *d_c, int M, int K, int N, int max_parts, int *parts);
// The gate|up product of one bf16 piece with its activation: act(gate, up) of neighbouring columns as bf16, d_out [M][N / 2]; K % 64 == 0.
// gemm_gated_pays: whether that is the quicker way (not where the few-rows kernel multiplies).
int gemm_gated_nk(hm_ctx *ctx, const uint16_t *d_a, const uint16_t *d_b_nk, uint16_t *d_out, int M, int K, int N, const GatedAct &act);
bool gemm_gated_pays(int M, int K, int N, int cus, int max_parts);
// The product of one bf16 piece that expands latents into the keys and values of all heads: columns [head * dim ..) go as bf16 to the rows
// of k [heads][cap][kw], columns [v_at + head * vdim ..) to those of v [heads][cap][vw]; columns that are no head's go nowhere, and what a row has
// behind dim and vdim stays as it was. gemm_heads_fits: not where the few-rows kernel multiplies.
struct HeadRows {
    int heads = 0, dim = 0, vdim = 0, v_at = 0, kw = 0, vw = 0, cap = 0;
    uint16_t *k = nullptr, *v = nullptr;
};
int gemm_heads_nk(hm_ctx *ctx, const uint16_t *d_a, const uint16_t *d_b_nk, int M, int K, int N, const HeadRows &h);
bool gemm_heads_fits(int M, int K, int N, int cus);
int gemm_half_slices(bool scaled, int M, int K, int N, int cus, int max_parts);
// The K slices that a product of activation pieces with b_pieces (1 or 3) pieces of B, or with a block-scaled B, comes in
int gemm_pieces_slices(int b_pieces, bool scaled, int M, int K, int N, int cus, int max_parts);
int gemm_pieces_any(hm_ctx *ctx, const uint16_t *d_a_split, int a_pieces, const uint16_t *d_b_split, int b_pieces,
                    const float *d_scales, int npad, float *d_c, int M, int K, int N, int max_parts, int *parts, int ldc);

}  // namespace homura
