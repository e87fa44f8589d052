// The prompt pass's products on f16 matrix instructions: every f32 activation as two f16 pieces against weights that are f16
// without loss, two matrix instructions where three bf16 pieces take three.
//
// x 2^e = p0 + p1, p0 = f16(x 2^e), p1 = f16(x 2^e - p0). p1 ends at 2^-24, f16's last subnormal: 23 to 24 significant bits of a
// scaled value of 2^-1 and more, which is 2^15 below the bound, and a bit less with every binade below that (three bf16 pieces hold all 24 at
// any size). Rows with outliers of 2^13 times their other values, brought down by their weights, come out as with three bf16 pieces
// (errors 0.9 of theirs); of 2^16 1.2 to 1.6 times, of 2^18 4 to 6 times as far off. The exponents e keep p0 in range whatever the finite
// input: a bound on |x| is known where the weights are, and x 2^e stays below 2^15.
//   a norm's output       |x_k| <= sqrt(dim) |w_k|                      one e per column, folded into the norm's weights
//   attention's output    a mean of value rows, |v_j| <= sqrt(dim) |W_v[j] o w|_2 + |b_j| (Cauchy-Schwarz)   one e per value column
//   SiLU(gate) up         |g_j u_j| <= dim |W_g[j] o w|_2 |W_u[j] o w|_2   one e per column, so that the gate|up product can write the
//                         rows itself. Rows of normal values lie 2^10 to 2^12 below that, and rows of small gates anywhere below those, so the
//                         second pieces are held 2^12 higher (HALF_LOW, row_pieces.h): 23 to 24 bits of values down to 2^-18 of a normal
//                         row's, gates near -15; below, a bit less a binade. Where the row kernel writes the rows there is a factor per row
//                         on top, from its largest value, and where a column's factor would cost the down weights bits, that one alone.
//                         (Down product, error of a row relative to itself, gates at -12 / -20, from the product and from the row kernel: 4e-7 / 4e-6 to
//                         1.2e-5, and 4e-7 / 1e-6. Second pieces as they are and no row factors: 1e-5 / 2e-2.)
// What is multiplied into a column of the activations is divided out of that column of the weights, so a product needs one
// factor per output row of the weights, 2^-r, which also puts the row's largest weight at 2^14 .. 2^15. All factors are powers
// of two. A matrix takes this way only if every one of its weights is then an f16 exactly (bf16 weights: 31 binades of a row,
// Q8_0 / Q4_0 integers: 24 binades of a block's columns); otherwise it keeps the three bf16 pieces.
#pragma once

#include <cstdint>

#include "hm_common.h"

namespace homura {

// w [dim] f32 norm weights -> w_scaled = w 2^e and the exponents e. *d_flag |= 1 where a weight has no exponent.
int half_norm_scales(hm_ctx *ctx, const float *d_w, int dim, float *d_w_scaled, int *d_exps, int *d_flag);

// The value rows' exponents: rows [N][K] of W_v (hm_dtype bf16: [N][K], or raw blocks), the norm weights ahead of it and its bias
// (or NULL). d_scale [N] = 2^e, and d_exps [H * hd]: the exponents by column of the attention's output, row n = (KV head, dim).
int half_value_scales(hm_ctx *ctx, int hm_dtype, const void *d_wv, const float *d_norm_w, const float *d_bias, int N, int K, int H,
                      int hd, float *d_scale, int *d_exps, int *d_flag);

// The gated rows' exponents: rows_bound [2 inter] = sqrt(dim) |W[n] o w|_2 of the gate (even) and up (odd) rows, row n of the matrix in
// place n * mult + off; then scale [inter] = 2^e and the exponents e by column.
int half_row_bounds(hm_ctx *ctx, int hm_dtype, const void *d_w, const float *d_norm_w, int N, int K, float *d_bounds, int mult, int off);
int half_gated_scales(hm_ctx *ctx, const float *d_bounds, int inter, float *d_scale, int *d_exps, int *d_flag);

// bf16 rows [N][K] -> f16(w 2^(r - e)) and unscale[n] = 2^-r. d_exps [K] or NULL (all 0).
int half_rows(hm_ctx *ctx, const uint16_t *d_w, const int *d_exps, int N, int K, uint16_t *d_out, float *d_unscale, int *d_flag);

// Q8_0 / Q4_0 blocks [N][K / 32]: the integers times 2^(m - e) as f16, m the least e of a block's columns, and the block scales
// times 2^-m, laid out as quant_ints_launch does (prefill.h).
int half_ints(hm_ctx *ctx, int hm_dtype, const uint8_t *d_blocks, const int *d_exps, int N, int K, uint16_t *d_ints, float *d_scales,
              int npad, int row_mult, int row_off, int *d_flag);

}  // namespace homura
