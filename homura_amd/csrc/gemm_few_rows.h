// Matrix products of at most 64 activation rows.
#pragma once

#include <cstdint>

#include "hm_common.h"

namespace homura {

constexpr int FEW_ROWS = 64;

// 32-row tiles of B a workgroup takes: two where single ones would be more than three quarters of a round of workgroups
// (24 rows: 1024 -> 4096 5.4 us with one and 6.2 with two, 1024 -> 6144 7.3 and 6.5)
inline int few_rows_tiles(int N, int cus) { return (N + 31) / 32 * 4 > 3 * (long long)cus ? 2 : 1; }

// Whether a product goes this way: always up to 32 rows, up to 64 while its workgroups are one round (64 rows, 1536 -> 17920:
// 40 us in two rounds, 32 in 128-row tiles)
inline bool few_rows_pays(int M, int N, int cus) {
    const int nt = few_rows_tiles(N, cus);
    return M <= 32 || (M <= FEW_ROWS && (N + 32 * nt - 1) / (32 * nt) <= cus);
}

// K slices of such a product, at most max_parts: while the workgroups still fit the chip at once, a group for every wavefront
int few_rows_slices(int M, int K, int N, int cus, int max_parts);

// C[M][N] f32 (row stride ldc) = (sum of the pieces of A [M][pieces K])  x  B [N][K]^T, M <= FEW_ROWS, K % 32 == 0; with d_scales
// (pieces = 3) B holds the integers of a block format and d_scales [K / 32][npad] the scale of every 32-wide block, npad >= N
// rounded up to 128. With parts the result may come as up to max_parts K slices, slice s at d_c + s * M * ldc.
int gemm_few_rows(hm_ctx *ctx, const uint16_t *d_a_split, int pieces, const uint16_t *d_b_nk, const float *d_scales, int npad,
                  float *d_c, int M, int K, int N, int max_parts, int *parts, int ldc);

}  // namespace homura
