// The generation loop of the framework's decoders (see decoder.h; reference src/hf/model.rs, src/generate.rs).
#include "decoder.h"

#include <algorithm>
#include <cstring>

#include "../light_ops.h"

namespace homura {

DecoderModel::~DecoderModel() {
    if (ctx_) hm_sync(ctx_);
    for (Pinned *b : {&stage_, &prompt_ids_, &draws_, &tokens_})
        if (b->p) (void)hipHostFree(b->p);
}

// At least `bytes` of pinned memory. A larger block takes the place of one that the stream may still be reading.
int DecoderModel::pinned_for(Pinned &b, size_t bytes) {
    if (b.bytes >= bytes) return HM_OK;
    if (b.p) {
        const int rc = hm_sync(ctx_);
        (void)hipHostFree(b.p);
        b = Pinned{};
        if (rc != HM_OK) return rc;
    }
    size_t size = 4096;
    while (size < bytes) size *= 2;
    HM_HIP(ctx_, hipHostMalloc(&b.p, size, hipHostMallocDefault));
    b.bytes = size;
    return HM_OK;
}

int DecoderModel::finish_sync(void *h_dst, const void *d_src, size_t words) {
    const int rc = words ? move_words_launch(ctx_, h_dst, d_src, words) : HM_OK;
    const int synced = hm_sync(ctx_);
    return rc == HM_OK ? synced : rc;
}

int DecoderModel::check_ids(const int64_t *ids, int n, std::vector<int32_t> &out) {
    out.resize(n);
    for (int i = 0; i < n; i++) {
        if (ids[i] < 0 || ids[i] >= vocab_size())
            return hm_set_error(ctx_, HM_ERR_INVALID, "token id %lld outside the vocabulary (%d)",
                                (long long)ids[i], vocab_size());
        out[i] = (int32_t)ids[i];
    }
    return HM_OK;
}

int DecoderModel::run_kv(const int64_t *h_ids, int n_ids, float *h_logits) {
    if (!finalized_) return hm_set_error(ctx_, HM_ERR_STATE, "model not finalized");
    return guarded([&] { return run_kv_once(h_ids, n_ids, h_logits); });
}

int DecoderModel::run_kv_once(const int64_t *h_ids, int n_ids, float *h_logits) {
    if (!finalized_) return hm_set_error(ctx_, HM_ERR_STATE, "model not finalized");
    if (n_ids <= 0 || !h_ids) return hm_set_error(ctx_, HM_ERR_INVALID, "run_kv: no input ids");
    if (kv_cache_len() + n_ids > max_seq_len_)
        return hm_set_error(ctx_, HM_ERR_STATE, "KV cache full (%d + %d > %d)", kv_cache_len(), n_ids, max_seq_len_);
    std::vector<int32_t> ids;
    int rc = check_ids(h_ids, n_ids, ids);
    if (rc != HM_OK) return rc;
    if (prefill_min_ > 0 && n_ids >= prefill_min_ && prefill_available()) return prefill(h_ids, n_ids, h_logits);
    if (n_ids > plan_->out_capacity())
        return hm_set_error(ctx_, HM_ERR_INVALID, "run_kv: %d ids exceed the step capacity %d", n_ids, plan_->out_capacity());
    if ((rc = plan_->arm(ids.data(), n_ids)) != HM_OK) return rc;
    std::vector<Buffer *> inputs;
    step_inputs(inputs);
    const size_t logits_slot = plan_->output_slots()[0];
    // The reference's decode loop reads a logits row per token (HfGenerationContext::decode_step,
    // src/hf/model.rs:340-371). The row and the whole-step status words are copied into pinned host memory
    // behind the step, so a token costs one stream synchronisation.
    const size_t row_bytes = (size_t)vocab_size() * 4;
    if (h_logits && (rc = pinned_for(stage_, row_bytes + 64)) != HM_OK) return rc;
    for (int i = 0; i < n_ids; i++) {
        if ((rc = plan_->run_kv(inputs, weight_bufs_, max_seq_len_)) != HM_OK) return rc;
        if (!h_logits) continue;
        char *stage = stage_.as<char>();
        const void *status = pending_status_words();
        rc = move_words_launch(ctx_, stage, plan_->slot(logits_slot)->ptr(), row_bytes / 4, status ? stage + row_bytes : nullptr, status);
        if (rc != HM_OK) return rc;
        if ((rc = hm_sync(ctx_)) != HM_OK) return rc;
        std::memcpy(h_logits + (size_t)i * vocab_size(), stage, row_bytes);
        if (status && (rc = check_status_words(reinterpret_cast<const uint32_t *>(stage + row_bytes))) != HM_OK) return rc;
    }
    return finish_sync();
}

int DecoderModel::prefill(const int64_t *h_ids, int n_ids, float *h_logits) {
    const int rc = prefill_enqueue(h_ids, n_ids, h_logits);
    return rc == HM_OK ? hm_sync(ctx_) : rc;
}

int DecoderModel::prefill_enqueue(const int64_t *h_ids, int n_ids, float *h_logits) {
    if (!finalized_) return hm_set_error(ctx_, HM_ERR_STATE, "model not finalized");
    if (!prefill_available())
        return hm_set_error(ctx_, HM_ERR_INVALID, "prefill: needs %s", prefill_needs());
    if (n_ids <= 0 || !h_ids) return hm_set_error(ctx_, HM_ERR_INVALID, "prefill: no input ids");
    if (kv_cache_len() + n_ids > max_seq_len_)
        return hm_set_error(ctx_, HM_ERR_STATE, "KV cache full (%d + %d > %d)", kv_cache_len(), n_ids, max_seq_len_);
    std::vector<int32_t> ids;
    int rc = check_ids(h_ids, n_ids, ids);
    if (rc != HM_OK) return rc;
    if ((rc = hm_sync(ctx_)) != HM_OK) return rc;  // (nothing to wait for, unless a call failed behind its prompt)
    if ((rc = pinned_for(prompt_ids_, (size_t)n_ids * 4)) != HM_OK) return rc;
    std::memcpy(prompt_ids_.p, ids.data(), (size_t)n_ids * 4);
    for (int at = 0; at < n_ids; at += chunk_rows_) {
        const int n = std::min(chunk_rows_, n_ids - at);
        rc = prefill_chunk(prompt_ids_.as<int32_t>() + at, n, h_logits ? h_logits + (size_t)at * vocab_size() : nullptr);
        if (rc != HM_OK) return rc;
    }
    return HM_OK;
}

int DecoderModel::kv_cache_len() const { return plan_ ? plan_->kv_cache_len() : 0; }

int DecoderModel::reset_kv_cache() {
    if (!finalized_) return hm_set_error(ctx_, HM_ERR_STATE, "model not finalized");
    plan_->reset_kv_cache();
    return HM_OK;
}

int DecoderModel::set_prefill_chunk(int) { return hm_set_error(ctx_, HM_ERR_INVALID, "this kind of model has a fixed chunk size"); }

int DecoderModel::rewind_to_mark(int mark_len, const std::vector<int32_t> &kept) {
    plan_->cache()->reset(mark_len + (int)kept.size());
    return HM_OK;
}

int DecoderModel::generate_greedy(const int64_t *h_prompt, int n_prompt, int n_new, int32_t *h_tokens) {
    if (!finalized_) return hm_set_error(ctx_, HM_ERR_STATE, "model not finalized");
    return guarded([&] { return generate_greedy_once(h_prompt, n_prompt, n_new, h_tokens); });
}

int DecoderModel::generate_greedy_once(const int64_t *h_prompt, int n_prompt, int n_new, int32_t *h_tokens) {
    if (!finalized_) return hm_set_error(ctx_, HM_ERR_STATE, "model not finalized");
    if (n_prompt <= 0 || n_new <= 0 || !h_prompt || !h_tokens)
        return hm_set_error(ctx_, HM_ERR_INVALID, "generate_greedy: bad arguments");
    int steps = n_prompt + n_new - 1;
    if (kv_cache_len() + steps > max_seq_len_)  // the reference's loop stops at max_seq_len
                                                // (src/generate.rs:188-194); here it is an error
        return hm_set_error(ctx_, HM_ERR_STATE, "KV cache full (%d + %d > %d)", kv_cache_len(), steps, max_seq_len_);
    if (prefill_min_ > 0 && n_prompt - 1 >= prefill_min_ && prefill_available()) {
        // reference HfGenerationContext::prefill (src/hf/model.rs:321-336): the prompt in one pass; its
        // last token goes through the decode step, whose pick is generated token 0
        int rc = prefill_enqueue(h_prompt, n_prompt - 1, nullptr);
        if (rc != HM_OK) return rc;
        h_prompt += n_prompt - 1;
        n_prompt = 1;
        steps = n_new;
    }
    if (steps > plan_->out_capacity())
        return hm_set_error(ctx_, HM_ERR_INVALID, "generate_greedy: %d steps exceed capacity %d", steps, plan_->out_capacity());
    std::vector<int32_t> ids;
    int rc = check_ids(h_prompt, n_prompt, ids);
    if (rc != HM_OK) return rc;
    if ((rc = plan_->arm(ids.data(), n_prompt)) != HM_OK) return rc;
    std::vector<Buffer *> inputs;
    step_inputs(inputs);
    for (int i = 0; i < steps; i++)
        if ((rc = plan_->run_kv(inputs, weight_bufs_, max_seq_len_)) != HM_OK) return rc;
    // the pick after prompt token n_prompt-1 is generated token 0
    if ((rc = pinned_for(tokens_, (size_t)n_new * 4)) != HM_OK) return rc;
    rc = finish_sync(tokens_.p, plan_->out_tokens() + (n_prompt - 1), n_new);
    if (rc == HM_OK) std::memcpy(h_tokens, tokens_.p, (size_t)n_new * 4);
    return rc;
}

// sampling.hip
int sample_check_config(hm_ctx *ctx, const hm_sampling_config *cfg, bool device);
int sample_token_launch(hm_ctx *ctx, const float *d_logits, float *d_work, const int *d_counts, int vocab,
                        const hm_sampling_config &cfg, float draw, int32_t *d_out, int *d_counts_update, int32_t *d_list,
                        int list_pos);
int sample_step_launch(hm_ctx *ctx, const float *d_logits, float *d_work, int *d_counts, int vocab,
                       const hm_sampling_config &cfg, DecodeState *d_cursor, const float *d_draws, int32_t *d_list,
                       int eos, int *d_stop, int32_t *d_out);
int zero_ints_launch(hm_ctx *ctx, int *d, size_t n);

int DecoderModel::generate(const int64_t *h_prompt, int n_prompt, int max_new, const hm_sampling_config &cfg, uint64_t seed,
                      int eos_token, int32_t *h_tokens, int *n_out) {
    if (!finalized_) return hm_set_error(ctx_, HM_ERR_STATE, "model not finalized");
    return guarded([&] { return generate_once(h_prompt, n_prompt, max_new, cfg, seed, eos_token, h_tokens, n_out); });
}

int DecoderModel::generate_once(const int64_t *h_prompt, int n_prompt, int max_new, const hm_sampling_config &cfg, uint64_t seed,
                           int eos_token, int32_t *h_tokens, int *n_out) {
    if (!finalized_) return hm_set_error(ctx_, HM_ERR_STATE, "model not finalized");
    if (n_prompt <= 0 || max_new <= 0 || !h_prompt || !h_tokens || !n_out)
        return hm_set_error(ctx_, HM_ERR_INVALID, "generate: bad arguments");
    *n_out = 0;
    const bool greedy = cfg.temperature <= 0.0f;
    const bool on_device = greedy || (cfg.top_k >= 1 && cfg.top_k <= 1024);
    int rc = sample_check_config(ctx_, &cfg, on_device);
    if (rc != HM_OK) return rc;
    if (kv_cache_len() + n_prompt > max_seq_len_)
        return hm_set_error(ctx_, HM_ERR_STATE, "KV cache full (%d + %d > %d)", kv_cache_len(), n_prompt, max_seq_len_);
    std::vector<int32_t> ids;
    if ((rc = check_ids(h_prompt, n_prompt, ids)) != HM_OK) return rc;
    const int vocab = vocab_size();
    SamplerScratch &s = sampler_;
    if (!s.work) {
        s.work = Buffer::alloc(ctx_, {vocab}, DType::F32);
        s.counts = Buffer::alloc(ctx_, {vocab}, DType::F32);  // int32 counts
        s.token = Buffer::alloc(ctx_, {64}, DType::F32);
        if (!s.work || !s.counts || !s.token) return HM_ERR_OOM;
    }
    if (s.list_cap < max_new) {
        s.list = Buffer::alloc(ctx_, {max_new}, DType::F32);  // int32 token list
        if (!s.list) return HM_ERR_OOM;
        s.list_cap = max_new;
    }
    const bool penalties = cfg.repetition_penalty != 1.0f || cfg.frequency_penalty != 0.0f || cfg.presence_penalty != 0.0f;
    // prompt: everything but its last token only has to reach the cache
    // (reference HfGenerationContext::prefill, src/hf/model.rs:321-336)
    if (n_prompt > 1) {
        const bool at_once = prefill_min_ > 0 && n_prompt - 1 >= prefill_min_ && prefill_available();
        rc = at_once ? prefill_enqueue(h_prompt, n_prompt - 1, nullptr) : run_kv_once(h_prompt, n_prompt - 1, nullptr);
        if (rc != HM_OK) return rc;
    }
    if ((rc = zero_ints_launch(ctx_, s.counts.as<int>(), (size_t)vocab)) != HM_OK) return rc;
    uint64_t rng = hm_rng_seed(seed);
    std::vector<Buffer *> inputs;
    step_inputs(inputs);
    const size_t logits_slot = plan_->output_slots()[0];
    std::vector<float> host_logits;
    std::vector<uint32_t> generated;
    int32_t current = ids[n_prompt - 1];
    if (on_device) {
        // Device-resident loop: steps are enqueued in chunks with nothing read back in between. The step's
        // own pick (greedy, no penalties) or the sampler launched behind it (its draw taken from a list made
        // up front, its pick written over the cursor's next input) feeds the next step on the GPU; the host
        // reads a chunk's tokens once, and on an end-of-sequence token takes the cache back to the row of the
        // step that produced it (the reference stops there: src/generate.rs:231-246).
        const bool own_pick = greedy && !penalties;
        if (!greedy) {
            if ((rc = pinned_for(draws_, (size_t)max_new * 4)) != HM_OK) return rc;
            if (n_prompt == 1 && (rc = hm_sync(ctx_)) != HM_OK) return rc;  // (a call that failed may have left a kernel that reads them)
            for (int i = 0; i < max_new; i++) draws_.as<float>()[i] = hm_rng_next_f32(&rng);
            if (s.draws_cap < max_new) {
                s.draws = Buffer::alloc(ctx_, {max_new}, DType::F32);
                if (!s.draws) return HM_ERR_OOM;
                s.draws_cap = max_new;
            }
            if ((rc = move_words_launch(ctx_, s.draws.ptr(), draws_.p, max_new)) != HM_OK) return rc;
        }
        // (no end-of-sequence token: nothing to be looked at in between)
        const int chunk_cap = std::min(plan_->out_capacity(), eos_token >= 0 ? 16 : 256);
        if ((rc = pinned_for(tokens_, (size_t)chunk_cap * 4)) != HM_OK) return rc;
        const int32_t *got = tokens_.as<int32_t>();
        int done = 0;
        while (done < max_new) {
            const int len0 = kv_cache_len();
            const int n = std::min({chunk_cap, max_new - done, max_seq_len_ - len0});
            if (n <= 0) break;  // context limit (src/generate.rs:188-194)
            if (eos_token >= 0 && (rc = mark_position()) != HM_OK) return rc;
            int32_t *d_stop = s.token.as<int32_t>() + 1;
            if ((rc = plan_->arm(&current, 1, own_pick ? nullptr : d_stop)) != HM_OK) return rc;
            for (int i = 0; i < n; i++) {
                if ((rc = plan_->run_kv(inputs, weight_bufs_, max_seq_len_)) != HM_OK) return rc;
                if (own_pick) continue;
                rc = sample_step_launch(ctx_, plan_->slot(logits_slot)->as<float>(), s.work.as<float>(),
                                        penalties ? s.counts.as<int>() : nullptr, vocab, cfg, plan_->state(),
                                        greedy ? nullptr : s.draws.as<float>() + done, s.list.as<int32_t>() + done, eos_token,
                                        d_stop, s.token.as<int32_t>());
                if (rc != HM_OK) return rc;
            }
            const int32_t *d_got = own_pick ? plan_->out_tokens() : s.list.as<int32_t>() + done;
            if (done + n == max_new) rc = finish_sync(tokens_.p, d_got, n);
            else if ((rc = move_words_launch(ctx_, tokens_.p, d_got, n)) == HM_OK) rc = hm_sync(ctx_);
            if (rc != HM_OK) return rc;
            int taken = n;
            for (int i = 0; i < n; i++)
                if (got[i] == eos_token) {
                    taken = i;
                    break;
                }
            for (int i = 0; i < taken; i++) h_tokens[(*n_out)++] = got[i];
            if (taken < n) {
                // what the steps behind the stop left in the cache is dropped
                std::vector<int32_t> kept{current};
                kept.insert(kept.end(), got, got + taken);
                if ((rc = rewind_to_mark(len0, kept)) != HM_OK) return rc;
                break;
            }
            current = got[n - 1];
            done += n;
        }
        return finish_sync();
    }
    for (int step = 0; step < max_new; step++) {
        if (kv_cache_len() >= max_seq_len_) break;  // context limit (src/generate.rs:188-194)
        if ((rc = plan_->arm(&current, 1)) != HM_OK) return rc;
        if ((rc = plan_->run_kv(inputs, weight_bufs_, max_seq_len_)) != HM_OK) return rc;
        const float *d_logits = plan_->slot(logits_slot)->as<float>();
        int32_t tok = 0;
        host_logits.resize(vocab);
        rc = hm_download(ctx_, host_logits.data(), d_logits, (size_t)vocab * 4);
        if (rc == HM_OK)
            rc = hm_sample_token_host(host_logits.data(), vocab, &cfg, generated.data(), (int)generated.size(), &rng, &tok);
        if (rc != HM_OK) return rc;
        if (tok == eos_token) break;  // the reference leaves the loop without storing the token
        generated.push_back((uint32_t)tok);
        h_tokens[(*n_out)++] = tok;
        current = tok;
    }
    return finish_sync();
}

int DecoderModel::bench_decode(int64_t first_id, int n_steps, float *ms_out, int32_t *h_tokens) {
    if (!finalized_) return hm_set_error(ctx_, HM_ERR_STATE, "model not finalized");
    return guarded([&] { return bench_decode_once(first_id, n_steps, ms_out, h_tokens); });
}

int DecoderModel::bench_decode_once(int64_t first_id, int n_steps, float *ms_out, int32_t *h_tokens) {
    if (!finalized_) return hm_set_error(ctx_, HM_ERR_STATE, "model not finalized");
    if (n_steps <= 0 || n_steps > plan_->out_capacity())
        return hm_set_error(ctx_, HM_ERR_INVALID, "bench_decode: bad step count %d", n_steps);
    if (kv_cache_len() + n_steps > max_seq_len_)
        return hm_set_error(ctx_, HM_ERR_STATE, "KV cache full (%d + %d > %d)", kv_cache_len(), n_steps, max_seq_len_);
    std::vector<int32_t> ids;
    int rc = check_ids(&first_id, 1, ids);
    if (rc != HM_OK) return rc;
    if ((rc = plan_->arm(ids.data(), 1)) != HM_OK) return rc;
    std::vector<Buffer *> inputs;
    step_inputs(inputs);
    hipEvent_t e0, e1;
    HM_HIP(ctx_, hipEventCreate(&e0));
    HM_HIP(ctx_, hipEventCreate(&e1));
    HM_HIP(ctx_, hipEventRecord(e0, ctx_->stream));
    for (int i = 0; i < n_steps; i++)
        if ((rc = plan_->run_kv(inputs, weight_bufs_, max_seq_len_)) != HM_OK) break;
    if (rc == HM_OK) {
        HM_HIP(ctx_, hipEventRecord(e1, ctx_->stream));
        HM_HIP(ctx_, hipEventSynchronize(e1));
        HM_HIP(ctx_, hipEventElapsedTime(ms_out, e0, e1));
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (rc != HM_OK) return rc;
    if (h_tokens) rc = hm_download(ctx_, h_tokens, plan_->out_tokens(), (size_t)n_steps * 4);
    return rc == HM_OK ? finish_sync() : rc;
}

int DecoderModel::time_kernels(int rounds, std::vector<StepProfile> &out) {
    if (!finalized_) return hm_set_error(ctx_, HM_ERR_STATE, "model not finalized");
    int32_t tok = 0;
    int rc = plan_->arm(&tok, 1);
    if (rc != HM_OK) return rc;
    std::vector<Buffer *> inputs;
    step_inputs(inputs);
    return plan_->time_kernels(inputs, weight_bufs_, max_seq_len_, rounds, out);
}

int DecoderModel::profile_step(int64_t token_id, std::vector<StepProfile> &out) {
    if (!finalized_) return hm_set_error(ctx_, HM_ERR_STATE, "model not finalized");
    std::vector<int32_t> ids;
    int rc = check_ids(&token_id, 1, ids);
    if (rc != HM_OK) return rc;
    if ((rc = plan_->arm(ids.data(), 1)) != HM_OK) return rc;
    std::vector<Buffer *> inputs;
    step_inputs(inputs);
    return plan_->profile_step(inputs, weight_bufs_, max_seq_len_, out);
}

}  // namespace homura
