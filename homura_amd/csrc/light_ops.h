// Internal launch interfaces of the light ops, shared with the decode plan.
#pragma once
#include "hm_common.h"

struct QkRopeArgs {
    float *q = nullptr;              // [S][H][hd], in place
    float *k = nullptr;              // [S][kvh][hd], in place
    const float *qw = nullptr;       // [hd] or NULL
    const float *kw = nullptr;       // [hd] or NULL
    const float *cos = nullptr;      // [S][hd]
    const float *sin = nullptr;      // [S][hd]
    int S = 0, H = 0, kvh = 0, hd = 0;
    float eps = 0.f;
    // optional fused cache append (batch 1): v [S][kvh][hd] f32, caches [kvh][max_len][hd] bf16
    const float *v = nullptr;
    uint16_t *kcache = nullptr;
    uint16_t *vcache = nullptr;
    int max_len = 0, pos = 0;
    // Decode-plan mode: the row position comes from state->pos and cos/sin point at the FULL
    // tables [max_pos][hd] (row pos + s is used), instead of pre-sliced rows.
    const DecodeState *state = nullptr;
};

int qknorm_rope_launch(hm_ctx *ctx, const QkRopeArgs &a);
// out = rmsnorm(x [+ res]) * w per row; resid_out (optional) receives x + res
int rmsnorm_launch(hm_ctx *ctx, const float *d_x, const float *d_res, const float *d_w, float *d_out,
                   float *d_resid_out, int rows, int dim, float eps);
int embed_launch(hm_ctx *ctx, const int64_t *d_ids64, const int32_t *d_ids32, const float *d_table,
                 float *d_out, int n_ids, int vocab, int hidden);
int argmax_candidates_launch(hm_ctx *ctx, const float *d_vals, const int *d_idxs, int n,
                             int32_t *d_out);
// Decode-plan variants driven by the device-resident cursor:
// embedding of this step's input id (forced id while step < n_forced, else the last pick)
int embed_step_launch(hm_ctx *ctx, const DecodeState *state, const int32_t *d_forced,
                      const float *d_table, float *d_out, int vocab, int hidden);
// What a call leaves for the device and takes from it, by kernels instead of copies: a copy waits some 25 us on either side of itself
// (a prompt's ids, cursor, forced id, logits row and status words were five of them).
// The cursor, up to ARM_IDS forced ids and, if stop is not NULL, -1 to it, all as launch arguments.
constexpr int ARM_IDS = 16;
int arm_launch(hm_ctx *ctx, DecodeState *d_state, const DecodeState &st, int32_t *d_forced, const int32_t *h_ids, int *d_stop);
// words 4-byte words between device memory and pinned host memory (either way), and 16 more from d_status to h_status if that is not
// NULL. The host's side is free, or filled, once the stream has been synchronised with.
int move_words_launch(hm_ctx *ctx, void *dst, const void *src, size_t words, void *h_status = nullptr, const void *d_status = nullptr);
// fold the LM-head argmax candidates, record the pick, advance the cursor
int finish_step_launch(hm_ctx *ctx, DecodeState *state, const float *d_vals, const int *d_idxs,
                       int n, int32_t *d_out_tokens, int out_cap);
