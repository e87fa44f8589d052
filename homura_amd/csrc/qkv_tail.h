// The tail of the q|k|v projection for one thread's share of a head row: bias, the head's norm and the rotation for q and k, then q to
// where it belongs in the f32 rows and k and v to the cache (QkvPostArgs, prefill.h). A thread holds four neighbouring low dims i .. i + 3
// and their partners half a head above; HD / 8 threads in a row of lanes make a head, and all of them take part.
#pragma once
#include "hm_common.h"
#include "prefill.h"

namespace homura {

struct QkvAngles {
    f32x4 c0, c1, s0, s1;
};
template <int HD>
__device__ __forceinline__ QkvAngles qkv_angles(const QkvPostArgs &a, int pos, int i) {
    const float *c = a.cos_tab + (size_t)pos * HD + i, *s = a.sin_tab + (size_t)pos * HD + i;
    return QkvAngles{*reinterpret_cast<const f32x4 *>(c), *reinterpret_cast<const f32x4 *>(c + HD / 2), *reinterpret_cast<const f32x4 *>(s),
                     *reinterpret_cast<const f32x4 *>(s + HD / 2)};
}

// row `s` of the chunk, head `j` of q | k | v; live: the row and the head exist
template <int HD>
__device__ __forceinline__ void qkv_tail(const QkvPostArgs &a, int s, int j, int i, bool live, f32x4 lo, f32x4 hi, const QkvAngles &t) {
    constexpr int LANES = HD / 8, HALF = HD / 2;
    const bool is_q = j < a.H, turns = j < a.H + a.kvh;
    if (a.bias) {
        const float *b = a.bias + (size_t)j * HD;
        lo += *reinterpret_cast<const f32x4 *>(b + i);
        hi += *reinterpret_cast<const f32x4 *>(b + i + HALF);
    }
    if (a.kw) {
        // In the order of the decode kernels' wave_sum over the pairs of a row, to the bit: a thread's four dims are one of its quads.
        float ss;
        {
#pragma clang fp contract(off)
            float d[4];
#pragma unroll
            for (int k = 0; k < 4; k++) d[k] = fmaf(lo[k], lo[k], hi[k] * hi[k]);
            ss = (d[0] + d[1]) + (d[2] + d[3]);
        }
        ss += dpp_move<0xB1, 0xF>(ss, 0.f);
        ss += dpp_move<0x4E, 0xF>(ss, 0.f);
        ss += dpp_move<0x141, 0xF>(ss, 0.f);
        if (LANES == 16) ss += dpp_move<0x140, 0xF>(ss, 0.f);
        if (turns) {
            const float inv = 1.0f / sqrtf(ss / (float)HD + a.eps);
            const float *nw = is_q ? a.qw : a.kw;
            const f32x4 w0 = *reinterpret_cast<const f32x4 *>(nw + i), w1 = *reinterpret_cast<const f32x4 *>(nw + i + HALF);
#pragma unroll
            for (int k = 0; k < 4; k++) {
                lo[k] = (lo[k] * inv) * w0[k];
                hi[k] = (hi[k] * inv) * w1[k];
            }
        }
    }
    if (!live) return;
    if (turns) {
        const f32x4 l = lo, h = hi;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            lo[k] = l[k] * t.c0[k] + (-h[k]) * t.s0[k];
            hi[k] = h[k] * t.c1[k] + l[k] * t.s1[k];
        }
    }
    if (is_q) {
        float *q = a.qkv + ((size_t)s * (a.H + 2 * a.kvh) + j) * HD + i;
        *reinterpret_cast<f32x4 *>(q) = lo;
        *reinterpret_cast<f32x4 *>(q + HALF) = hi;
        return;
    }
    typedef uint16_t u16x4 __attribute__((ext_vector_type(4)));
    u16x4 blo, bhi;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        blo[k] = f32_to_bf16_rne_dev(lo[k]);
        bhi[k] = f32_to_bf16_rne_dev(hi[k]);
    }
    const int g = turns ? j - a.H : j - a.H - a.kvh;
    uint16_t *dst = (turns ? a.kcache : a.vcache) + ((size_t)g * a.max_len + a.past + s) * HD;
    *reinterpret_cast<u16x4 *>(dst + i) = blo;
    *reinterpret_cast<u16x4 *>(dst + i + HALF) = bhi;
}

// The same for a tile of ROWS x COLS sums in LDS (rows `ld` floats apart), row m0 and column n0 first: THREADS threads, two head rows of
// each at a time, if it is an even number, so that the second one's tables are on their way.
template <int HD, int ROWS, int COLS, int THREADS>
__device__ __forceinline__ void qkv_tail_tile(const QkvPostArgs &a, const float *tile, int ld, int m0, int n0) {
    constexpr int LANES = HD / 8, ITEMS = ROWS * (COLS / HD) * LANES / THREADS, AT = ITEMS % 2 ? 1 : 2;
    static_assert(COLS % HD == 0 && ROWS * (COLS / HD) * LANES % THREADS == 0, "whole heads, as many head rows for every thread");
    const int heads = a.H + 2 * a.kvh;
#pragma unroll 1
    for (int it = 0; it < ITEMS; it += AT) {
        QkvAngles t[AT];
        int row[AT], head[AT];
        const int i = (int)threadIdx.x % LANES * 4;
#pragma unroll
        for (int o = 0; o < AT; o++) {
            const int r = ((it + o) * THREADS + (int)threadIdx.x) / LANES;
            row[o] = r % ROWS;
            head[o] = r / ROWS;
            t[o] = qkv_angles<HD>(a, a.past + min(m0 + row[o], a.S - 1), i);
        }
#pragma unroll
        for (int o = 0; o < AT; o++) {
            const float *at = tile + row[o] * ld + head[o] * HD + i;
            const int j = n0 / HD + head[o];
            qkv_tail<HD>(a, m0 + row[o], min(j, heads - 1), i, m0 + row[o] < a.S && j < heads, *reinterpret_cast<const f32x4 *>(at),
                         *reinterpret_cast<const f32x4 *>(at + HD / 2), t[o]);
        }
    }
}

}  // namespace homura
