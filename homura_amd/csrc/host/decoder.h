// What every decoder of the framework has in common: weight slots, the recorded decode step and the cache behind
// it (ExecutionPlan), the prompt pass in chunks, and the generation loops over them (reference HfModel /
// HfGenerationContext, src/hf/model.rs, and generate_streaming_core, src/generate.rs:100-315). A model supplies
// its weights, its decode plan and one chunk of its prompt pass.
#pragma once

#include <functional>
#include <map>
#include <memory>
#include <string>
#include <vector>

#include "runtime.h"

namespace homura {

// One entry of TransformerWeights::to_slot_buffers (src/hf/weights.rs:63-116 / :136-183):
// what the host hands over for this slot.
struct WeightSlotInfo {
    std::string name;
    DType dtype;
    int64_t dim0 = 0, dim1 = 0;  // bf16/f32 matrices: [K][N] as the reference keeps them;
                                 // quantised: dim0 = N rows, dim1 = K (raw blocks [N][K/32])
    size_t bytes = 0;
};

// Rotation tables [max_seq_len][dims] of f32 cosines and sines, both halves of a row alike (pairs i, i + dims / 2).
void precompute_rope_cos_sin(int dims, int max_seq_len, double theta, std::vector<float> &cosv, std::vector<float> &sinv);

class DecoderModel {
  public:
    virtual ~DecoderModel();
    // Rows of the prompt pass that go through the layers together. A model whose cache is laid out for it takes
    // another size before finalize (HM_ERR_INVALID otherwise).
    int prefill_chunk_rows() const { return chunk_rows_; }
    virtual int set_prefill_chunk(int rows);

    virtual int vocab_size() const = 0;
    virtual int hidden_size() const = 0;
    virtual int num_layers() const = 0;
    const std::vector<WeightSlotInfo> &weight_slot_infos() const { return infos_; }
    // Upload one slot (host pointer, exact byte size). bf16 matrices arrive [K][N] and are
    // re-packed once into the K-contiguous stream layout; quantised blocks stay as they are.
    virtual int set_weight(int slot, const void *h_data, size_t bytes) = 0;
    // Same, but a matrix slot (bf16 projection, LM head) arrives [N][K] - one output row after the
    // other, K contiguous: the layout of HF safetensors ([out, in]) and of GGUF tensors, and the
    // stream layout kept in HBM, so nothing is transposed on the way in.
    virtual int set_weight_nk(int slot, const void *h_data, size_t bytes) = 0;
    // reference HfModel::ensure_compiled (src/hf/model.rs:148-160) + RoPE tables (:62-66)
    virtual int finalize(int max_seq_len) = 0;

    // reference HfModel::run_kv (src/hf/model.rs:198-218); multi-token input is consumed one
    // token per plan step. h_logits: [n_ids][vocab] or NULL.
    int run_kv(const int64_t *h_ids, int n_ids, float *h_logits);
    // The multi-token pass behind run_kv for longer inputs (reference run_kv with seq > 1,
    // src/hf/model.rs:321-336): the chunk goes through the layers as a matrix, projections on the
    // matrix cores; n_ids rows are appended to the cache. h_logits: [n_ids][vocab] or NULL (then the LM
    // head is skipped).
    int prefill(const int64_t *h_ids, int n_ids, float *h_logits);
    virtual bool prefill_available() const = 0;
    // Inputs of at least this many tokens take the prefill pass (0 = never). Default 8.
    virtual int set_prefill_min(int n) {
        prefill_min_ = n;
        return HM_OK;
    }
    int prefill_min() const { return prefill_min_; }
    // bf16 pieces per f32 activation in the prefill pass; HM_ERR_INVALID when the model does not take that many
    virtual int set_prefill_pieces(int n) = 0;
    int prefill_pieces() const { return prefill_pieces_; }
    virtual int reset_kv_cache();
    int kv_cache_len() const;
    int generate_greedy(const int64_t *h_prompt, int n_prompt, int n_new, int32_t *h_tokens);
    // reference generate_streaming_core (src/generate.rs:100-315) with sample_token (:698-801)
    int generate(const int64_t *h_prompt, int n_prompt, int max_new, const hm_sampling_config &cfg, uint64_t seed,
                 int eos_token, int32_t *h_tokens, int *n_out);
    int bench_decode(int64_t first_id, int n_steps, float *ms_out, int32_t *h_tokens);
    int profile_step(int64_t token_id, std::vector<StepProfile> &out);
    int time_kernels(int rounds, std::vector<StepProfile> &out);
    ExecutionPlan *plan() { return plan_.get(); }

  protected:
    DecoderModel() = default;
    // One chunk of the prompt pass (n <= prefill_chunk_rows() ids, in memory that the device reads): appends n rows to the cache.
    virtual int prefill_chunk(const int32_t *d_ids, int n, float *h_logits) = 0;
    virtual const char *prefill_needs() const = 0;  // for the error message when the pass is not available
    virtual int step_inputs(std::vector<Buffer *> &inputs) = 0;
    // End of a call: stream synchronisation and whatever the steps left to be looked at. With words, first that many 4-byte words from d_src
    // to pinned h_dst.
    virtual int finish_sync(void *h_dst = nullptr, const void *d_src = nullptr, size_t words = 0);
    // Runs the body of a call; a model whose steps can fail recoverably runs it again.
    virtual int guarded(const std::function<int()> &body) { return body(); }
    // 64 bytes of device status words to fetch with the logits row of a step (NULL: nothing to look at), and
    // what their host copy says.
    virtual const void *pending_status_words() { return nullptr; }
    virtual int check_status_words(const uint32_t *) { return HM_OK; }
    // Ahead of steps that may have to be taken back: remember the cache as it is. rewind_to_mark returns to it
    // (length mark_len) plus the steps of `kept`, the input ids of the steps that stay. A cache of rows only
    // needs its length changed.
    virtual int mark_position() { return HM_OK; }
    virtual int rewind_to_mark(int mark_len, const std::vector<int32_t> &kept);
    int check_ids(const int64_t *ids, int n, std::vector<int32_t> &out);

    // Pinned host memory that kernels read and write: of run_kv, a logits row and the status words, which arrive with one
    // synchronisation; a prompt's ids; a generation's draws and tokens. A call that succeeds synchronises before it returns. One that fails may
    // leave kernels behind that read a prompt's ids or the draws, so these are written behind a synchronisation; the other blocks are written by kernels
    // only, in stream order, and read behind a synchronisation of their own.
    struct Pinned {
        void *p = nullptr;
        size_t bytes = 0;
        template <class T>
        T *as() const { return static_cast<T *>(p); }
    };
    int pinned_for(Pinned &b, size_t bytes);
    Pinned stage_, prompt_ids_, draws_, tokens_;

    hm_ctx *ctx_ = nullptr;
    bool finalized_ = false;
    int max_seq_len_ = 0;
    std::vector<WeightSlotInfo> infos_;
    std::vector<Buffer> weight_bufs_;   // in weight_slots order, device resident
    std::vector<bool> weight_set_;
    std::map<std::string, int> slot_by_name_;
    std::unique_ptr<ExecutionPlan> plan_;
    int prefill_min_ = 8;
    int prefill_pieces_ = 3;
    // Rows of the prompt pass that go through the layers together at most: a product of 2048 rows and more fills the CUs
    // with 128 x 256 tiles and few K slices (6000 tokens of the Qwen3-0.6B shape and 16 steps in chunks of 512 rows 60.9 ms, of
    // 3072 46.5; 1000 tokens in Q8_0 7.8 and 6.4). A longer prompt takes full chunks and a rest, which is few products' worth:
    // cut into equal chunks 4200, 5000 and 6001 tokens take 22.6, 27.8 and 33.8 ms, so 21.1, 25.2 and 31.8
    int chunk_rows_ = 4096;

  private:
    // the bodies of the calls of the same name (see guarded)
    int run_kv_once(const int64_t *h_ids, int n_ids, float *h_logits);
    int generate_greedy_once(const int64_t *h_prompt, int n_prompt, int n_new, int32_t *h_tokens);
    int generate_once(const int64_t *h_prompt, int n_prompt, int max_new, const hm_sampling_config &cfg, uint64_t seed,
                      int eos_token, int32_t *h_tokens, int *n_out);
    int bench_decode_once(int64_t first_id, int n_steps, float *ms_out, int32_t *h_tokens);
    // The prompt pass without the synchronisation at its end, for calls that go on
    int prefill_enqueue(const int64_t *h_ids, int n_ids, float *h_logits);
    struct SamplerScratch { Buffer work, counts, token, list, draws; int list_cap = 0, draws_cap = 0; } sampler_;
};

}  // namespace homura
