// Entry points that tests drive single steps of the prompt and decode passes with (homura_amd_bench.h). Those that look into a file's own choices
// stand there.
#include "../../include/homura_amd_bench.h"

#include <algorithm>
#include <vector>

#include "die_fold.h"
#include "gemm_bf16_mfma.h"
#include "half_weights.h"
#include "latent_attention.h"
#include "prefill.h"
#include "quant_formats.h"
#include "row_pieces.h"

using namespace homura;

namespace {

struct Scratch {
    std::vector<void *> all;
    ~Scratch() {
        for (void *p : all) (void)hipFree(p);
    }
    template <class T>
    T *get(size_t count) {
        void *p = nullptr;
        if (hipMalloc(&p, count * sizeof(T)) != hipSuccess) return nullptr;
        all.push_back(p);
        return static_cast<T *>(p);
    }
};

}  // namespace

extern "C" int hm_test_prompt_rows(hm_ctx *ctx, int front, const void *x, const float *norm_w, int dtype, const void *w, int half, int m,
                                   int k, int n, float *out, float *row_factor, int *parts) {
    HM_CHECK_CTX(ctx);
    HM_REQUIRE(ctx, x && w && out && row_factor && parts && (front != 0 || norm_w), "hm_test_prompt_rows: NULL pointer");
    const bool bf16 = dtype == HM_DTYPE_BF16;
    HM_REQUIRE(ctx, (bf16 || dtype == HM_DTYPE_Q8_0 || dtype == HM_DTYPE_Q4_0) && front >= 0 && front <= 2 && half >= 0 && half <= 1 &&
                        (front != 2 || (bf16 && !half)) && m > 0 && n > 0 && k > 0 && k % (half ? 64 : 32) == 0,
               "hm_test_prompt_rows: bad arguments");
    Scratch mem;
    const int npad = half ? half_scale_cols(n) : (n + 127) / 128 * 128;
    uint16_t *rows = mem.get<uint16_t>((size_t)m * k * 3), *wh = mem.get<uint16_t>((size_t)n * k);
    float *scaled = mem.get<float>(k), *factors = mem.get<float>(std::max<size_t>((size_t)(k / 32) * npad, n));
    int *exps = mem.get<int>(k), *flag = mem.get<int>(1);
    HM_REQUIRE(ctx, rows && wh && scaled && factors && exps && flag, "hm_test_prompt_rows: out of memory");
    HM_HIP(ctx, hipMemsetAsync(flag, 0, 4, ctx->stream));
    std::vector<float> ones((size_t)m, 1.f);
    int rc = hm_upload(ctx, row_factor, ones.data(), (size_t)m * 4);
    const uint16_t *b = bf16 && !half ? static_cast<const uint16_t *>(w) : wh, *a = rows;
    const int *cols = nullptr;
    if (rc == HM_OK && half && front == 0) {
        rc = half_norm_scales(ctx, norm_w, k, scaled, exps, flag);
        cols = exps;
    }
    if (rc == HM_OK && half)
        rc = bf16 ? half_rows(ctx, static_cast<const uint16_t *>(w), cols, n, k, wh, factors, flag)
                  : half_ints(ctx, dtype, static_cast<const uint8_t *>(w), cols, n, k, wh, factors, npad, 1, 0, flag);
    else if (rc == HM_OK && !bf16)
        rc = quant_ints_launch(ctx, dtype, static_cast<const uint8_t *>(w), n, k, wh, factors, npad);
    const float *xf = static_cast<const float *>(x);
    if (front == 2) a = static_cast<const uint16_t *>(x);
    else if (rc == HM_OK && front == 0)
        rc = rmsnorm_split_launch(ctx, xf, nullptr, 1, half ? scaled : norm_w, rows, half ? 2 : 3, nullptr, m, k, 1e-6f, false, nullptr, nullptr,
                                  nullptr, half == 1);
    else if (rc == HM_OK)
        rc = half ? silu_mul_half_launch(ctx, xf, 1, rows, row_factor, m, k) : silu_mul_split_launch(ctx, xf, 1, rows, 3, m, k);
    int bad = 0;
    if (rc == HM_OK) rc = hm_download(ctx, &bad, flag, 4);
    if (rc == HM_OK) rc = hm_sync(ctx);
    if (rc != HM_OK) return rc;
    if (bad) return hm_set_error(ctx, HM_ERR_STATE, "hm_test_prompt_rows: the weights are not f16 without loss");
    HalfProduct product{bf16 ? factors : nullptr};
    product.low = front == 1;
    if (half) rc = gemm_half_nk(ctx, a, b, product, bf16 ? nullptr : factors, npad, out, m, k, n, 8, parts);
    else if (!bf16) rc = gemm_pieces_scaled_nk(ctx, a, b, factors, npad, out, m, k, n, 8, parts);
    else rc = gemm_split_nk(ctx, a, front == 2 ? 1 : 3, b, out, m, k, n, 8, parts);
    return rc == HM_OK ? hm_sync(ctx) : rc;
}

namespace {

// The gate|up product of the test hooks below and its gated rows in two f16 pieces, out of the product or of the row kernel
struct GatedTest {
    Scratch mem;
    int *gate_exps = nullptr, *flag = nullptr;
    float *scale = nullptr, *row_unscale = nullptr;  // by column; by row (row kernel)
    uint16_t *gated = nullptr;                       // [m][2][inter], guarded words behind them if the caller has any
    int run(hm_ctx *ctx, const void *x, const float *norm_w, int dtype, const void *w, int fused, int m, int k, int inter, int *pays) {
        const bool bf16 = dtype == HM_DTYPE_BF16;
        HM_REQUIRE(ctx, (bf16 || dtype == HM_DTYPE_Q8_0 || dtype == HM_DTYPE_Q4_0) && m > 0 && inter > 0 && (fused || inter % 4 == 0) && k > 0 &&
                            k % 64 == 0, "gated rows: bad arguments");
        const int n = 2 * inter, npad = half_scale_cols(n);
        uint16_t *rows = mem.get<uint16_t>((size_t)m * k * 2), *wh = mem.get<uint16_t>((size_t)n * k);
        float *scaled = mem.get<float>(k), *factors = mem.get<float>(std::max<size_t>((size_t)(k / 32) * npad, n)), *bounds = mem.get<float>(n);
        float *c = mem.get<float>(8 * (size_t)m * n);
        int *exps = mem.get<int>(k);
        gate_exps = mem.get<int>(inter);
        flag = mem.get<int>(1);
        row_unscale = mem.get<float>(m);
        if (!scale) scale = mem.get<float>(inter);
        if (!gated) gated = mem.get<uint16_t>((size_t)m * n);
        HM_REQUIRE(ctx, rows && wh && scaled && factors && bounds && c && exps && gate_exps && flag && row_unscale && scale && gated, "gated rows: out of memory");
        HM_HIP(ctx, hipMemsetAsync(flag, 0, 4, ctx->stream));
        if (pays) *pays = gemm_half_gated_pays(!bf16, m, k, n, ctx->num_cus, 8);
        int rc = half_norm_scales(ctx, norm_w, k, scaled, exps, flag);
        if (rc == HM_OK)
            rc = bf16 ? half_rows(ctx, static_cast<const uint16_t *>(w), exps, n, k, wh, factors, flag)
                      : half_ints(ctx, dtype, static_cast<const uint8_t *>(w), exps, n, k, wh, factors, npad, 1, 0, flag);
        if (rc == HM_OK) rc = half_row_bounds(ctx, dtype, w, norm_w, n, k, bounds, 1, 0);
        if (rc == HM_OK) rc = half_gated_scales(ctx, bounds, inter, scale, gate_exps, flag);
        if (rc == HM_OK)
            rc = rmsnorm_split_launch(ctx, static_cast<const float *>(x), nullptr, 1, scaled, rows, 2, nullptr, m, k, 1e-6f, false, nullptr, nullptr,
                                      nullptr, true);
        int parts = 1;
        if (rc == HM_OK) rc = exact(ctx);
        if (rc != HM_OK) return rc;
        HalfProduct half{bf16 ? factors : nullptr};
        if (fused) {
            half.gate_scale = scale;
            half.gated = gated;
        }
        rc = gemm_half_nk(ctx, rows, wh, half, bf16 ? nullptr : factors, npad, fused ? nullptr : c, m, k, n, 8, &parts);
        if (rc == HM_OK && !fused) rc = silu_mul_half_launch(ctx, c, parts, gated, row_unscale, m, inter, scale);
        return rc == HM_OK ? hm_sync(ctx) : rc;
    }
    // that the weights so far are f16 without loss
    int exact(hm_ctx *ctx) {
        int bad = 0, rc = hm_download(ctx, &bad, flag, 4);
        if (rc == HM_OK) rc = hm_sync(ctx);
        if (rc != HM_OK) return rc;
        return bad ? hm_set_error(ctx, HM_ERR_STATE, "gated rows: the weights are not f16 without loss") : HM_OK;
    }
};

}  // namespace

extern "C" int hm_test_gated_rows(hm_ctx *ctx, const void *x, const float *norm_w, int dtype, const void *w, int fused, int m, int k,
                                  int inter, uint16_t *out, float *scale, int *pays) {
    HM_CHECK_CTX(ctx);
    HM_REQUIRE(ctx, x && norm_w && w && out && scale && pays, "hm_test_gated_rows: NULL pointer");
    GatedTest t;
    t.scale = scale;
    t.gated = out;
    int rc = t.run(ctx, x, norm_w, dtype, w, fused, m, k, inter, pays);
    if (rc != HM_OK) return rc;
    // without the row kernel's factors and HALF_LOW, as the two f16 nearest to what the pieces add up to
    std::vector<uint16_t> p((size_t)m * 2 * inter);
    std::vector<float> rows((size_t)m, 1.f);
    rc = hm_download(ctx, p.data(), out, p.size() * 2);
    if (rc == HM_OK && !fused) rc = hm_download(ctx, rows.data(), t.row_unscale, rows.size() * 4);
    if (rc == HM_OK) rc = hm_sync(ctx);
    if (rc != HM_OK) return rc;
    for (int r = 0; r < m; r++)
        for (int j = 0; j < inter; j++) {
            uint16_t *at = p.data() + (size_t)r * 2 * inter + j;
            const double v = ((double)__builtin_bit_cast(_Float16, at[0]) + (double)__builtin_bit_cast(_Float16, at[inter]) / HALF_LOW) * rows[r];
            const _Float16 hi = (_Float16)v, lo = (_Float16)(v - (double)hi);
            at[0] = __builtin_bit_cast(uint16_t, hi);
            at[inter] = __builtin_bit_cast(uint16_t, lo);
        }
    rc = hm_upload(ctx, out, p.data(), p.size() * 2);
    return rc == HM_OK ? hm_sync(ctx) : rc;
}

extern "C" int hm_test_gated_down(hm_ctx *ctx, const void *x, const float *norm_w, int dtype, const void *w, const void *down, int fused, int m,
                                  int k, int inter, float *out) {
    HM_CHECK_CTX(ctx);
    HM_REQUIRE(ctx, x && norm_w && w && down && out && inter % 64 == 0, "hm_test_gated_down: bad arguments");
    GatedTest t;
    int rc = t.run(ctx, x, norm_w, dtype, w, fused, m, k, inter, nullptr);
    if (rc != HM_OK) return rc;
    const bool bf16 = dtype == HM_DTYPE_BF16;
    const int npad = half_scale_cols(k);
    uint16_t *wd = t.mem.get<uint16_t>((size_t)k * inter);
    float *factors = t.mem.get<float>(std::max<size_t>((size_t)(inter / 32) * npad, k));
    HM_REQUIRE(ctx, wd && factors, "hm_test_gated_down: out of memory");
    rc = bf16 ? half_rows(ctx, static_cast<const uint16_t *>(down), t.gate_exps, k, inter, wd, factors, t.flag)
              : half_ints(ctx, dtype, static_cast<const uint8_t *>(down), t.gate_exps, k, inter, wd, factors, npad, 1, 0, t.flag);
    if (rc == HM_OK) rc = t.exact(ctx);
    HalfProduct half{bf16 ? factors : nullptr};
    half.low = true;
    if (rc == HM_OK) rc = gemm_half_nk(ctx, t.gated, wd, half, bf16 ? nullptr : factors, npad, out, m, inter, k);
    std::vector<float> rows((size_t)m), sums((size_t)m * k);
    if (rc == HM_OK && !fused) rc = hm_download(ctx, rows.data(), t.row_unscale, rows.size() * 4);
    if (rc == HM_OK && !fused) rc = hm_download(ctx, sums.data(), out, sums.size() * 4);
    if (rc == HM_OK) rc = hm_sync(ctx);
    if (rc != HM_OK || fused) return rc;
    for (size_t i = 0; i < sums.size(); i++) sums[i] *= rows[i / k];
    rc = hm_upload(ctx, out, sums.data(), sums.size() * 4);
    return rc == HM_OK ? hm_sync(ctx) : rc;
}

extern "C" int hm_test_qkv_product(hm_ctx *ctx, const void *x, const float *norm_w, int dtype, const void *w, int fused, int S, int k, int H,
                                   int kvh, int hd, const float *bias, const float *qw, const float *kw, const float *cos, const float *sin,
                                   float *q, uint16_t *kcache, uint16_t *vcache, int max_len, int past, float eps, int *pays) {
    HM_CHECK_CTX(ctx);
    HM_REQUIRE(ctx, x && norm_w && w && cos && sin && q && kcache && vcache && pays, "hm_test_qkv_product: NULL pointer");
    const bool bf16 = dtype == HM_DTYPE_BF16;
    HM_REQUIRE(ctx, (bf16 || dtype == HM_DTYPE_Q8_0 || dtype == HM_DTYPE_Q4_0) && S > 0 && k > 0 && k % 64 == 0 && H > 0 && kvh > 0 && (hd == 64 || hd == 128) &&
                        past >= 0 && past + S <= max_len, "hm_test_qkv_product: bad arguments");
    Scratch mem;
    const int n = (H + 2 * kvh) * hd, npad = half_scale_cols(n);
    uint16_t *rows = mem.get<uint16_t>((size_t)S * k * 2), *wh = mem.get<uint16_t>((size_t)n * k);
    float *scaled = mem.get<float>(k), *factors = mem.get<float>(std::max<size_t>((size_t)(k / 32) * npad, n)), *c = mem.get<float>(8 * (size_t)S * n);
    int *exps = mem.get<int>(k), *flag = mem.get<int>(1);
    HM_REQUIRE(ctx, rows && wh && scaled && factors && c && exps && flag, "hm_test_qkv_product: out of memory");
    HM_HIP(ctx, hipMemsetAsync(flag, 0, 4, ctx->stream));
    *pays = gemm_half_tail_pays(!bf16, hd, S, k, n, ctx->num_cus, 8);
    int rc = half_norm_scales(ctx, norm_w, k, scaled, exps, flag);
    if (rc == HM_OK)
        rc = bf16 ? half_rows(ctx, static_cast<const uint16_t *>(w), exps, n, k, wh, factors, flag)
                  : half_ints(ctx, dtype, static_cast<const uint8_t *>(w), exps, n, k, wh, factors, npad, 1, 0, flag);
    if (rc == HM_OK)
        rc = rmsnorm_split_launch(ctx, static_cast<const float *>(x), nullptr, 1, scaled, rows, 2, nullptr, S, k, eps, false, nullptr, nullptr,
                                  nullptr, true);
    int bad = 0, parts = 1;
    if (rc == HM_OK) rc = hm_download(ctx, &bad, flag, 4);
    if (rc == HM_OK) rc = hm_sync(ctx);
    if (rc != HM_OK) return rc;
    if (bad) return hm_set_error(ctx, HM_ERR_STATE, "hm_test_qkv_product: the weights are not f16 without loss");
    QkvPostArgs t;
    t.qkv = fused ? q : c;
    t.bias = bias;
    t.qw = qw;
    t.kw = kw;
    t.cos_tab = cos;
    t.sin_tab = sin;
    t.kcache = kcache;
    t.vcache = vcache;
    t.S = S;
    t.H = H;
    t.kvh = kvh;
    t.hd = hd;
    t.max_len = max_len;
    t.past = past;
    t.eps = eps;
    HalfProduct half{bf16 ? factors : nullptr};
    if (fused) half.tail = &t;
    rc = gemm_half_nk(ctx, rows, wh, half, bf16 ? nullptr : factors, npad, fused ? nullptr : c, S, k, n, 8, &parts);
    if (rc == HM_OK && !fused) {
        t.parts = parts;
        t.part_stride = (size_t)S * n;
        rc = qkv_post_launch(ctx, t);
        if (rc == HM_OK) rc = hm_copy(ctx, q, c, (size_t)S * n * 4);
    }
    return rc == HM_OK ? hm_sync(ctx) : rc;
}

extern "C" int hm_test_qkv_tail(hm_ctx *ctx, float *d_qkv, const float *d_qw, const float *d_kw, const float *d_cos, const float *d_sin,
                                uint16_t *d_kcache, uint16_t *d_vcache, int S, int H, int kvh, int hd, int max_len, int past, float eps) {
    HM_CHECK_CTX(ctx);
    QkvPostArgs a;
    a.qkv = d_qkv;
    a.qw = d_qw;
    a.kw = d_kw;
    a.cos_tab = d_cos;
    a.sin_tab = d_sin;
    a.kcache = d_kcache;
    a.vcache = d_vcache;
    a.S = S;
    a.H = H;
    a.kvh = kvh;
    a.hd = hd;
    a.max_len = max_len;
    a.past = past;
    a.eps = eps;
    return qkv_post_launch(ctx, a);
}

extern "C" int hm_test_gated_product(hm_ctx *ctx, const uint16_t *a, const uint16_t *b, uint16_t *out, int m, int k, int n, int kind, float limit,
                                     float slope, int *pays) {
    HM_CHECK_CTX(ctx);
    HM_REQUIRE(ctx, pays && (kind == GatedAct::Silu || kind == GatedAct::ClampedSigmoid), "hm_test_gated_product: bad arguments");
    GatedAct act;
    act.kind = kind;
    act.limit = limit;
    act.slope = slope;
    *pays = gemm_gated_pays(m, k, n, ctx->num_cus, 8);
    return gemm_gated_nk(ctx, a, b, out, m, k, n, act);
}

extern "C" int hm_test_latent_rows(hm_ctx *ctx, const float *down, int ld, int parts, const float *q_norm, const float *kv_norm, const float *cos_tab,
                                   const float *sin_tab, int q_rank, int rank, int rot, int pieces, int n, int past, float eps, uint16_t *q_split,
                                   uint16_t *ring) {
    HM_CHECK_CTX(ctx);
    LatentRowsArgs a;
    a.s.heads = a.s.dim = a.s.vdim = 1;
    a.s.rank = rank;
    a.s.rot_dim = a.s.rot_dims = rot;
    a.s.rank_pad = (rank + 31) / 32 * 32;
    a.s.rot_pad = (rot + 31) / 32 * 32;
    a.s.pieces = a.q_pieces = pieces;
    a.s.ring_rows = past + n;
    a.down = RowSource{down, ld, parts, (size_t)n * ld, nullptr};
    a.q_norm = q_norm;
    a.kv_norm = kv_norm;
    a.cos_tab = cos_tab;
    a.sin_tab = sin_tab;
    a.q_rank = q_rank;
    a.q_rank_pad = (q_rank + 31) / 32 * 32;
    a.n = n;
    a.past = past;
    a.eps = eps;
    a.q_split = q_split;
    a.ring = ring;
    const int rc = latent_rows_launch(ctx, a);
    return rc == HM_OK ? hm_sync(ctx) : rc;
}

extern "C" int hm_test_routes(hm_ctx *ctx, long long *counts) {
    HM_CHECK_CTX(ctx);
    HM_REQUIRE(ctx, counts != nullptr, "hm_test_routes: NULL pointer");
    counts[0] = ctx->routes.die_folds;
    counts[1] = ctx->routes.gates_whole;
    counts[2] = ctx->routes.gates_sliced;
    return HM_OK;
}

extern "C" int hm_test_die_arrivals(hm_ctx *ctx, int group) {
    HM_CHECK_CTX(ctx);
    HM_REQUIRE(ctx, group >= 0 && (size_t)(group + 1) * DIE_COUNTER_STRIDE <= ctx->num_counters, "hm_test_die_arrivals: group %d", group);
    const unsigned long long came = 0x0101;
    return hm_upload(ctx, ctx->counters + (size_t)group * DIE_COUNTER_STRIDE, &came, sizeof(came));
}
