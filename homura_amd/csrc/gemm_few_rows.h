// Matrix products of at most 64 activation rows.
#pragma once

#include <cstdint>

#include "gemm_bf16_mfma.h"
#include "hm_common.h"

namespace homura {

constexpr int FEW_ROWS = 64;

// 32-row tiles of B a workgroup takes: two where single ones would be more than three quarters of a round of workgroups
// (24 rows: 1024 -> 4096 5.4 us with one and 6.2 with two, 1024 -> 6144 7.3 and 6.5)
inline int few_rows_tiles(int N, int cus) { return (N + 31) / 32 * 4 > 3 * (long long)cus ? 2 : 1; }

// Whether a product goes this way: up to 64 rows while its workgroups are one round (64 rows, 1536 -> 17920: 40 us in two
// rounds, 32 in 128-row tiles); more rounds with up to 32 rows, always with two or three pieces and with one where the last
// round is nearly full. Weights cold, 24 rows, us here / in 128-row tiles, three pieces: 1536 -> 17920 26.7 / 34.3, 1024 ->
// 65536 41.2 / 56.1, 1536 -> 151936 132 / 191, 3072 -> 24576 46.7 / 65.4; one piece: 1536 -> 17920 (1.1 rounds) 17.8 / 17.5,
// 3072 -> 24576 (1.5) 34.2 / 33.0, 2048 -> 32000 (1.95) 30.9 / 34.4, 1024 -> 65536 (4) 30.9 / 36.4, 1536 -> 151936 (9.3) 104 / 104.
inline bool few_rows_pays(int pieces, int M, int N, int cus) {
    const int nt = few_rows_tiles(N, cus);
    const long long wgs = (N + 32 * nt - 1) / (32 * nt), rounds = (wgs + cus - 1) / cus;
    if (rounds <= 1) return M <= FEW_ROWS;
    return M <= 32 && (pieces > 1 || 10 * wgs >= 9 * rounds * cus);
}

// K slices of such a product, at most max_parts: while the workgroups still fit the chip at once, a group for every wavefront
int few_rows_slices(int M, int K, int N, int cus, int max_parts);

// C[M][N] f32 (row stride ldc) = (sum of the pieces of A [M][pieces K])  x  B [N][K]^T, M <= FEW_ROWS, K % 32 == 0; with d_scales
// (pieces = 3, or 2 with half) B holds the integers of a block format and d_scales [K / 32][npad] the scale of every 32-wide block, npad >= N
// rounded up to 128. With parts the result may come as up to max_parts K slices, slice s at d_c + s * M * ldc.
// half: f16 operands (gemm_half_nk).
int gemm_few_rows(hm_ctx *ctx, const uint16_t *d_a_split, int pieces, const uint16_t *d_b_nk, const float *d_scales, int npad,
                  float *d_c, int M, int K, int N, int max_parts, int *parts, int ldc, const HalfProduct *half = nullptr);

}  // namespace homura
