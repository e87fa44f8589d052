// Token sampling (reference sample_token, src/generate.rs:698-801, and its xorshift64 Rng, :609-642).
//
// Two implementations behind one configuration struct:
//  * hm_sample_token_host: the reference's procedure statement by statement on a host logits row
//    (libm expf, sequential f32 sums, full sort). Any top_k.
//  * hm_sample_token: the same procedure on a logits row that stays in HBM, for 1 <= top_k <= 1024.
//    One workgroup of 1024 threads: penalties + temperature + max, exponentials + sum, a radix select
//    (12 + 10 + 10 bits) of the top_k-th largest exponential, the candidates gathered and sorted in LDS (probability
//    descending, index ascending among equals), then one thread runs the reference's sequential top_p
//    and draw loops over at most 1024 candidates. The vocabulary-wide sum is a tree sum here, so a
//    probability may differ from the host's in the last bit; the picked token differs only when the
//    draw sits on a cumulative boundary to within that bit.
// The draw itself (Rng::next_f32) is taken on the host and passed in, so both consume the same stream.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "hm_common.h"

namespace {

constexpr int SAMPLE_THREADS = 1024;
constexpr int SAMPLE_MAX_K = 1024;

struct SampleArgs {
    const float *logits;
    float *work;          // [vocab] scratch: adjusted logits, then exponentials
    const int *counts;    // [vocab] occurrences among the generated tokens, or nullptr
    int vocab;
    hm_sampling_config cfg;
    float draw;           // Rng::next_f32 of this step
    int32_t *out;         // the picked token
    int *counts_update;   // if set: counts_update[token]++ after the pick (the token joins generated_ids)
    int32_t *list;        // if set: list[list_pos] = token
    int list_pos;
    // Device-resident loop: the step that was just taken is cursor->step - 1; its draw is draws[that], the pick
    // goes to list[that] and replaces the step's own greedy pick as the next input (cursor->token), and the
    // first step whose pick is `eos` is noted in stop[0] (-1 until then).
    DecodeState *cursor;
    const float *draws;
    int eos;
    int *stop;
};

// What a sampler kernel needs to know about its step, read once at its start: the loads are two dependent trips
// to memory (the cursor, then the draw it points at) that would otherwise sit at the very end of a kernel that
// runs as a single workgroup.
struct StepInfo {
    int idx;     // the step that was just taken (cursor->step - 1), or -1 without a cursor
    float draw;  // Rng::next_f32 of this step
    int stop;    // *stop (-1: no end-of-sequence pick so far), 0 without a stop cell
};
__device__ __forceinline__ StepInfo load_step(const SampleArgs &a) {
    StepInfo s;
    s.idx = a.cursor ? a.cursor->step - 1 : -1;
    s.draw = (a.cursor && a.draws) ? a.draws[s.idx] : a.draw;  // (a greedy pick with penalties has no draws)
    s.stop = a.stop ? *a.stop : 0;
    return s;
}

// Where the pick goes when the cursor says which step this is.
__device__ __forceinline__ void deliver_pick(const SampleArgs &a, const StepInfo &st, int pick) {
    *a.out = pick;
    if (a.counts_update) a.counts_update[pick] += 1;
    if (a.cursor) {
        if (a.list) a.list[st.idx] = pick;
        a.cursor->token = pick;
        if (a.stop && pick == a.eos && st.stop < 0) *a.stop = st.idx;
    } else if (a.list) {
        a.list[a.list_pos] = pick;
    }
}

__device__ __forceinline__ float penalised(float l, int c, const hm_sampling_config &cfg) {
    if (c > 0) {
        if (cfg.repetition_penalty != 1.0f)
            for (int k = 0; k < c; k++) l = l > 0.0f ? l / cfg.repetition_penalty : l * cfg.repetition_penalty;
        if (cfg.frequency_penalty != 0.0f || cfg.presence_penalty != 0.0f) {
            l -= cfg.frequency_penalty * (float)c;
            l -= cfg.presence_penalty;
        }
    }
    return l;
}

// a > b in the candidate order: larger probability first, smaller index first among equals
__device__ __forceinline__ bool cand_before(float pa, int ia, float pb, int ib) {
    return pa > pb || (pa == pb && ia < ib);
}

// One pass of the workgroup over [0, n): thread t visits t, t + 1024, ... in ascending order, eight elements'
// loads in flight before the first is used (a plain strided loop waits for every load in turn, and with one
// workgroup on the whole chip the passes are pure latency).
template <class Load, class Use>
__device__ __forceinline__ void sweep(int n, int tid, Load load, Use use) {
    constexpr int UN = 8;
    for (int base = tid; base < n; base += UN * SAMPLE_THREADS) {
        decltype(load(0)) v[UN];
#pragma unroll
        for (int u = 0; u < UN; u++) {
            const int i = base + u * SAMPLE_THREADS;
            if (i < n) v[u] = load(i);
        }
#pragma unroll
        for (int u = 0; u < UN; u++) {
            const int i = base + u * SAMPLE_THREADS;
            if (i < n) use(i, v[u]);
        }
    }
}

struct LogitAndCount {
    float l;
    int c;
};

// Shared memory of the selection below.
struct SelectShared {
    float red_f[SAMPLE_THREADS / WAVE];
    int red_i[SAMPLE_THREADS / WAVE];
    unsigned hist[4096];
    unsigned sel_prefix, sel_need;
    float cand_p[SAMPLE_MAX_K];
    int cand_i[SAMPLE_MAX_K];
    unsigned n_cand, eq_taken, n_eq;
    int eq_idx[SAMPLE_MAX_K];
};

// The second half of the procedure over n items: key_at(j) is item j's 32-bit key (larger key = larger
// exponential; items with equal keys must appear in ascending token order), idx_at(j) its token,
// weight_of(key) its exponential; `sum` is the sum of all n_all exponentials of the vocabulary. Selects the
// top_k items, normalises, applies min_p, sorts and runs the reference's sequential top_p and draw loops.
template <class KeyAt, class IdxAt, class WeightOf>
__device__ __forceinline__ void select_sort_draw(SelectShared &sh, const SampleArgs &a, const StepInfo &st, int n, int n_all,
                                                 float sum, KeyAt key_at, IdxAt idx_at, WeightOf weight_of) {
    float (&red_f)[SAMPLE_THREADS / WAVE] = sh.red_f;
    int (&red_i)[SAMPLE_THREADS / WAVE] = sh.red_i;
    unsigned (&hist)[4096] = sh.hist;
    unsigned &sel_prefix = sh.sel_prefix, &sel_need = sh.sel_need;
    float (&cand_p)[SAMPLE_MAX_K] = sh.cand_p;
    int (&cand_i)[SAMPLE_MAX_K] = sh.cand_i;
    unsigned &n_cand = sh.n_cand, &eq_taken = sh.eq_taken, &n_eq = sh.n_eq;
    int (&eq_idx)[SAMPLE_MAX_K] = sh.eq_idx;
    (void)red_f;
    const int tid = threadIdx.x, lane = tid & (WAVE - 1), wave = tid / WAVE;
    const hm_sampling_config cfg = a.cfg;
    // ── radix select: key of the K-th largest item (keys order like the exponentials). 12 + 10 + 10 bits: the first pass sees every element, and 4096 bins keep neighbouring
    //    lanes off each other's LDS word; later passes only count the elements inside the chosen bin. ──
    const unsigned K = (unsigned)min(cfg.top_k, n_all);
    if (tid == 0) {
        sel_prefix = 0;
        sel_need = K;
    }
    for (int pass = 0; pass < 3; pass++) {
        const int shift = pass == 0 ? 20 : pass == 1 ? 10 : 0;
        const int bits = pass == 0 ? 12 : 10;
        const int bpt = (1 << bits) / SAMPLE_THREADS;  // bins per thread: 4, 1, 1
        for (int b = tid; b < (1 << bits); b += SAMPLE_THREADS) hist[b] = 0;
        __syncthreads();
        const unsigned prefix = sel_prefix, need = sel_need;
        const unsigned mask = pass == 0 ? 0u : 0xFFFFFFFFu << (shift + bits);
        sweep(n, tid, key_at, [&](int, unsigned u) {
            if ((u & mask) == prefix) atomicAdd(&hist[(u >> shift) & ((1u << bits) - 1u)], 1u);
        });
        __syncthreads();
        // the bin that holds the need-th largest of the counted elements: thread t owns bins [t*bpt, (t+1)*bpt)
        unsigned mine = 0;
        for (int j = 0; j < bpt; j++) mine += hist[tid * bpt + j];
        unsigned incl = mine;  // inclusive prefix sum over threads, low bins first
        for (int off = 1; off < WAVE; off <<= 1) {
            const unsigned up = __shfl_up(incl, off, WAVE);
            if (lane >= off) incl += up;
        }
        if (lane == WAVE - 1) red_i[wave] = (int)incl;
        __syncthreads();
        unsigned before = 0, total = 0;
        for (int w = 0; w < SAMPLE_THREADS / WAVE; w++) {
            if (w < wave) before += (unsigned)red_i[w];
            total += (unsigned)red_i[w];
        }
        const unsigned below_or_mine = before + incl;      // elements in bins up to and including mine
        const unsigned above = total - below_or_mine;      // elements in higher bins
        if (above < need && need <= above + mine) {        // exactly one thread
            unsigned acc = above;
            for (int j = bpt - 1; j >= 0; j--) {
                const unsigned h = hist[tid * bpt + j];
                if (acc + h >= need) {
                    sel_prefix = prefix | ((unsigned)(tid * bpt + j) << shift);
                    sel_need = need - acc;  // how many elements of this bin are still wanted
                    break;
                }
                acc += h;
            }
        }
        __syncthreads();
    }
    const unsigned T = sel_prefix;
    const unsigned need_eq = sel_need;
    if (tid == 0) {
        n_cand = 0;
        eq_taken = 0;
        n_eq = 0;
    }
    __syncthreads();
    // everything above the K-th value; then the wanted number of elements equal to it, lowest indices first
    sweep(n, tid, key_at, [&](int i, unsigned u) {
        if (u > T) {
            const unsigned at = atomicAdd(&n_cand, 1u);
            cand_p[at] = weight_of(u);
            cand_i[at] = idx_at(i);
        } else if (u == T) {
            const unsigned at = atomicAdd(&n_eq, 1u);
            if (at < (unsigned)SAMPLE_MAX_K) eq_idx[at] = idx_at(i);
        }
    });
    __syncthreads();
    // Few elements equal the K-th value (nearly always exactly one): they were noted on the way, and each takes
    // its rank among them by index. Otherwise (a flat tail, underflowed exponentials) one ordered walk.
    const bool eq_listed = n_eq <= (unsigned)SAMPLE_MAX_K;
    if (eq_listed && tid < (int)n_eq) {
        const int mine = eq_idx[tid];
        unsigned rank = 0;
        for (unsigned j = 0; j < n_eq; j++) rank += eq_idx[j] < mine ? 1u : 0u;
        if (rank < need_eq) {
            const unsigned at = atomicAdd(&n_cand, 1u);
            cand_p[at] = weight_of(T);
            cand_i[at] = mine;
        }
    }
    for (int base = 0; base < n; base += SAMPLE_THREADS) {  // index order: one block-wide ordered take per 1024
        if (eq_listed || eq_taken >= need_eq) break;
        const int i = base + tid;
        const bool eq = i < n && key_at(i) == T;
        const unsigned long long m = __ballot(eq);
        if (lane == 0) red_i[wave] = __popcll(m);
        __syncthreads();
        unsigned before = eq_taken;
        for (int w = 0; w < wave; w++) before += red_i[w];
        const unsigned rank = before + __popcll(m & ((1ull << lane) - 1ull));
        if (eq && rank < need_eq) {
            const unsigned at = atomicAdd(&n_cand, 1u);
            cand_p[at] = weight_of(T);
            cand_i[at] = idx_at(i);
        }
        __syncthreads();
        if (tid == 0) {
            unsigned tot = 0;
            for (int w = 0; w < SAMPLE_THREADS / WAVE; w++) tot += red_i[w];
            eq_taken += tot;
        }
        __syncthreads();
    }
    __syncthreads();
    const int nc = (int)n_cand;  // == K
    // normalise, min_p (the maximum probability is exp(0) / sum), pad to the sort size
    const float max_prob = 1.0f / sum;
    const float threshold = cfg.min_p * max_prob;
    int sort_n = 2;  // the power of two that holds the candidates: 64 for the default top_k of 50, not 1024
    while (sort_n < nc) sort_n <<= 1;
    if (tid < sort_n) {
        if (tid < nc) {
            float p = cand_p[tid] / sum;
            if (cfg.min_p > 0.0f && p < threshold) p = 0.0f;
            cand_p[tid] = p;
        } else {
            cand_p[tid] = -1.0f;  // sorts behind every real candidate
            cand_i[tid] = 0x7FFFFFFF;
        }
    }
    __syncthreads();
    // bitonic sort of sort_n (probability descending, index ascending among equals)
    for (int k = 2; k <= sort_n; k <<= 1)
        for (int j = k >> 1; j > 0; j >>= 1) {
            const int partner = tid ^ j;
            if (partner > tid && tid < sort_n) {
                const float pa = cand_p[tid], pb = cand_p[partner];
                const int ia = cand_i[tid], ib = cand_i[partner];
                const bool up = (tid & k) == 0;  // this pair ends in candidate order
                if (cand_before(pb, ib, pa, ia) == up) {
                    cand_p[tid] = pb;
                    cand_i[tid] = ib;
                    cand_p[partner] = pa;
                    cand_i[partner] = ia;
                }
            }
            __syncthreads();
        }
    // the reference's sequential loops (src/generate.rs:771-800). Up to a wavefront's worth of candidates (the
    // default top_k of 50) sit in the registers of wavefront 0 and the loops read them lane by lane: the same
    // additions in the same order, without an LDS round trip per step.
    if (nc <= WAVE) {
        if (wave != 0) return;
        const float p = lane < nc ? cand_p[lane] : 0.0f;
        const int ci = lane < nc ? cand_i[lane] : 0;
        auto p_at = [&](int i) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(p), i)); };
        float cumulative = 0.0f;
        int cutoff = nc;
        for (int i = 0; i < nc; i++) {
            cumulative += p_at(i);
            if (cumulative >= cfg.top_p) {
                cutoff = i + 1;
                break;
            }
        }
        float total = 0.0f;
        for (int i = 0; i < cutoff; i++) total += p_at(i);
        const float r = st.draw * total;
        float accum = 0.0f;
        int at = cutoff > 0 ? cutoff - 1 : -1;
        for (int i = 0; i < cutoff; i++) {
            accum += p_at(i);
            if (accum >= r) {
                at = i;
                break;
            }
        }
        const int pick = at >= 0 ? __builtin_amdgcn_readlane(ci, at) : 0;
        if (lane == 0) deliver_pick(a, st, pick);
        return;
    }
    if (tid == 0) {
        float cumulative = 0.0f;
        int cutoff = nc;
        for (int i = 0; i < nc; i++) {
            cumulative += cand_p[i];
            if (cumulative >= cfg.top_p) {
                cutoff = i + 1;
                break;
            }
        }
        float total = 0.0f;
        for (int i = 0; i < cutoff; i++) total += cand_p[i];
        const float r = st.draw * total;
        float accum = 0.0f;
        int pick = cutoff > 0 ? cand_i[cutoff - 1] : 0;
        for (int i = 0; i < cutoff; i++) {
            accum += cand_p[i];
            if (accum >= r) {
                pick = cand_i[i];
                break;
            }
        }
        deliver_pick(a, st, pick);
    }
}

__global__ __launch_bounds__(SAMPLE_THREADS) void sample_token_kernel(SampleArgs a) {
    __shared__ SelectShared sh;
    float (&red_f)[SAMPLE_THREADS / WAVE] = sh.red_f;
    int (&red_i)[SAMPLE_THREADS / WAVE] = sh.red_i;
    const int tid = threadIdx.x, lane = tid & (WAVE - 1), wave = tid / WAVE;
    const int n = a.vocab;
    const hm_sampling_config cfg = a.cfg;
    const StepInfo st = load_step(a);

    // ── pass 1: penalties, then either the greedy pick or temperature + maximum ──
    const bool greedy = cfg.temperature <= 0.0f;
    const float inv_temp = greedy ? 1.0f : 1.0f / cfg.temperature;
    float mx = -INFINITY;
    int best = -1;  // greedy: last index of the maximum (Rust max_by keeps the last of equal maxima)
    sweep(n, tid, [&](int i) { return LogitAndCount{a.logits[i], a.counts ? a.counts[i] : 0}; },
          [&](int i, const LogitAndCount &lc) {
              float l = penalised(lc.l, lc.c, cfg);
              if (greedy) {
                  if (best < 0 || l >= mx) {
                      mx = l;
                      best = i;
                  }
              } else {
                  l *= inv_temp;
                  a.work[i] = l;
                  mx = fmaxf(mx, l);
              }
          });
    if (greedy) {
        for (int off = 32; off >= 1; off >>= 1) {
            const float om = __shfl_xor(mx, off, WAVE);
            const int ob = __shfl_xor(best, off, WAVE);
            if (ob >= 0 && (best < 0 || om > mx || (om == mx && ob > best))) {
                mx = om;
                best = ob;
            }
        }
        if (lane == 0) {
            red_f[wave] = mx;
            red_i[wave] = best;
        }
        __syncthreads();
        if (tid == 0) {
            for (int w = 1; w < SAMPLE_THREADS / WAVE; w++)
                if (red_i[w] >= 0 && (best < 0 || red_f[w] > mx || (red_f[w] == mx && red_i[w] > best))) {
                    mx = red_f[w];
                    best = red_i[w];
                }
            deliver_pick(a, st, best < 0 ? 0 : best);
        }
        return;
    }
    mx = wave_max(mx);
    if (lane == 0) red_f[wave] = mx;
    __syncthreads();
    mx = red_f[0];
    for (int w = 1; w < SAMPLE_THREADS / WAVE; w++) mx = fmaxf(mx, red_f[w]);
    __syncthreads();

    // ── pass 2: exponentials and their sum ──
    float sum = 0.f;
    sweep(n, tid, [&](int i) { return a.work[i]; }, [&](int i, float l) {
        const float e = expf(l - mx);
        a.work[i] = e;
        sum += e;
    });
    sum = wave_sum(sum);
    if (lane == 0) red_f[wave] = sum;
    __syncthreads();
    sum = 0.f;
    for (int w = 0; w < SAMPLE_THREADS / WAVE; w++) sum += red_f[w];
    __syncthreads();
    // exponentials are >= 0, so their bit patterns order like their values
    select_sort_draw(sh, a, st, n, n, sum, [&](int i) { return __float_as_uint(a.work[i]); }, [&](int i) { return i; },
                     [&](unsigned key) { return __uint_as_float(key); });
}

// ── Small top_k (<= 64) over a large vocabulary: two launches instead of one workgroup's eight passes ──
// Front: a wavefront per group of 64 tokens or more (the least power of two with at most 1024 groups) applies penalties
// and temperature and writes the group's maximum, the sum of its exponentials relative to it and its first four tokens by
// (logit descending, token ascending): one trip to memory and ten reductions, no LDS. (Groups of more than 256 tokens, which
// vocabularies beyond 262144 have, do not stay in registers and are read again for each of these.) Back: one workgroup combines maxima and sums (sum over the vocabulary =
// sum_g sum_g * exp(max_g - max), equal to the single pass's up to rounding). The K-th largest of the groups' first
// keys is a floor for the K-th largest of the vocabulary (K tokens reach it), so the top K are among the kept tokens
// that reach it, a hundred or so, unless all four of a group do: then such groups are read again.
// It selects by logit, which orders tokens like their exponentials except where two different logits round to one
// exponential.
// What bounds the pair is latency: a launch, one trip to memory and the barriers between the steps of a single
// workgroup, whose instructions come from memory too (the step before it has swept the instruction cache): loops
// here are rolled, and what is rare lies behind a branch. 151936 tokens, top_k 50, behind a whole-step decode kernel:
// front 4.7 us, back 5.6 (the 64 first of every 1024 tokens by a radix select in a workgroup each, and all of those
// looked through by the back: 6.6 and 11.7; the listed groups always read again, instead of kept tokens: 4.6 and 10.4).
// Rows that are no model's, 151936 tokens, top_k 50, a call from the host, us (a peaked row takes 29.5): all but ten tokens masked 29, equal
// logits 37, the first 30 % well above the rest 43. With every group that reaches the floor, or the first 50 of them, read again and
// no floor above zero probabilities: 107, 111 and 85; with the 64 first of every 1024 tokens: 73, 78 and 55.
constexpr int FRONT_THREADS = 256;
constexpr int FRONT_MAX_K = WAVE;                 // largest top_k
constexpr int FRONT_GROUP_BITS = 6;               // tokens of a group: the least power of two from 64 with at most 1024 groups
constexpr int FRONT_UNITS = SAMPLE_THREADS / 4;   // the floor is taken over at most so many maxima

// larger float <-> larger key (-inf the smallest key of all finite and infinite values)
__device__ __forceinline__ unsigned order_key(float x) {
    const unsigned u = __float_as_uint(x);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float key_value(unsigned k) {
    return __uint_as_float((k & 0x80000000u) ? (k & 0x7FFFFFFFu) : ~k);
}
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ unsigned dpp_keys(unsigned k) {
    return (unsigned)__builtin_amdgcn_update_dpp(0, (int)k, CTRL, ROW_MASK, 0xF, false);
}
__device__ __forceinline__ unsigned wave_max_key(unsigned k) {  // (the steps of wave_max)
    k = max(k, dpp_keys<0xB1, 0xF>(k));
    k = max(k, dpp_keys<0x4E, 0xF>(k));
    k = max(k, dpp_keys<0x141, 0xF>(k));
    k = max(k, dpp_keys<0x140, 0xF>(k));
    k = max(k, dpp_keys<0x142, 0xA>(k));
    k = max(k, dpp_keys<0x143, 0xC>(k));
    return (unsigned)__builtin_amdgcn_readlane((int)k, 63);
}

constexpr int FRONT_KEEP = 4;
struct FrontOut {
    unsigned *key;  // [groups][FRONT_KEEP]
    int *token;     // [groups][FRONT_KEEP]
    float *most, *sum;
};
__host__ __device__ inline FrontOut front_out(float *work, int groups) {
    const size_t n = (size_t)groups * FRONT_KEEP;
    return FrontOut{reinterpret_cast<unsigned *>(work), reinterpret_cast<int *>(work) + n, work + 2 * n, work + 2 * n + groups};
}

__global__ __launch_bounds__(FRONT_THREADS) void sample_front_kernel(SampleArgs a, int groups, int group_bits) {
    const int lane = threadIdx.x & (WAVE - 1), g = (int)((blockIdx.x * FRONT_THREADS + threadIdx.x) / WAVE);
    if (g >= groups) return;
    const float inv_temp = 1.0f / a.cfg.temperature;
    const int first = g << group_bits, end = min(a.vocab, first + (1 << group_bits)), chunks = group_bits <= 8 ? 1 : 1 << (group_bits - 8);
    auto load = [&](int j, float (&x)[4]) {
        const int base = first + j * 256 + lane;
        float l[4];
        int c[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int i = min(base + u * WAVE, end - 1);
            l[u] = a.logits[i];
            c[u] = a.counts ? a.counts[i] : 0;
        }
#pragma unroll
        for (int u = 0; u < 4; u++) x[u] = base + u * WAVE < end ? penalised(l[u], c[u], a.cfg) * inv_temp : -INFINITY;
    };
    float x[4], m = -INFINITY;
    for (int j = 0; j < chunks; j++) {
        load(j, x);
#pragma unroll
        for (int u = 0; u < 4; u++) m = fmaxf(m, x[u]);
    }
    m = wave_max(m);
    float e = 0.f;
    for (int j = 0; j < chunks; j++) {
        if (chunks > 1) load(j, x);
#pragma unroll
        for (int u = 0; u < 4; u++) e += x[u] > -INFINITY ? expf(x[u] - m) : 0.f;
    }
    e = wave_sum(e);
    // The group's tokens in order, each the first of those behind the one before it. (Lanes past the group's end hold
    // the key of -inf and higher token numbers.)
    unsigned last = 0xFFFFFFFFu, my_key = 0;
    int last_token = -1, my_token = 0;
#pragma unroll 1
    for (int r = 0; r < FRONT_KEEP; r++) {
        unsigned best = 0;
        int token = 0x7FFFFFFF;
        for (int j = 0; j < chunks; j++) {
            if (chunks > 1) load(j, x);
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const unsigned k = order_key(x[u]);
                const int t = first + j * 256 + u * WAVE + lane;
                if (((k < last) | ((k == last) & (t > last_token))) & (k > best)) {
                    best = k;
                    token = t;
                }
            }
        }
        last = wave_max_key(best);
        last_token = (int)~wave_max_key(best == last ? ~(unsigned)token : 0u);
        if (lane == r) {
            my_key = last;
            my_token = last_token;
        }
    }
    const FrontOut f = front_out(a.work, groups);
    if (lane < FRONT_KEEP) {
        f.key[g * FRONT_KEEP + lane] = my_key;
        f.token[g * FRONT_KEEP + lane] = my_token;
    }
    if (lane == 0) {
        f.most[g] = m;
        f.sum[g] = e;
    }
}

__global__ __launch_bounds__(SAMPLE_THREADS) void sample_back_kernel(SampleArgs a, int groups, int group_bits) {
    __shared__ SelectShared sh;
    __shared__ unsigned floor_key, listed, survived[2], more;
    __shared__ alignas(16) unsigned unit_key[FRONT_UNITS];
    __shared__ float red_sum[SAMPLE_THREADS / WAVE];
    __shared__ int list[SAMPLE_THREADS];
    // a survivor as one 64-bit number that orders like (logit descending, token ascending): key, then the
    // token counted down from the largest
    __shared__ unsigned long long fcomp[SAMPLE_MAX_K];
    const int tid = threadIdx.x, lane = tid & (WAVE - 1), wave = tid / WAVE;
    const FrontOut f = front_out(a.work, groups);
    const float gm = tid < groups ? f.most[tid] : -INFINITY, gs = tid < groups ? f.sum[tid] : 0.f;
    u32x4 kept_key{0u, 0u, 0u, 0u}, kept_token{0u, 0u, 0u, 0u};
    if (tid < groups) {
        kept_key = *reinterpret_cast<const u32x4 *>(f.key + tid * FRONT_KEEP);
        kept_token = *reinterpret_cast<const u32x4 *>(f.token + tid * FRONT_KEEP);
    }
    const unsigned key = kept_key[0];
    const StepInfo st = load_step(a);
    const float inv_temp = 1.0f / a.cfg.temperature;
    const unsigned K = (unsigned)min(a.cfg.top_k, a.vocab);
    // Up to 256 units, four threads each: the groups, or fours of them (64 at least: the vocabulary has 4096 tokens or more)
    const bool fours = groups > FRONT_UNITS;
    const int units = fours ? (groups + 3) / 4 : groups;
    unsigned four = max(key, dpp_keys<0xB1, 0xF>(key));
    four = max(four, dpp_keys<0x4E, 0xF>(four));
    if (fours ? (tid & 3) == 0 : tid < FRONT_UNITS) unit_key[fours ? tid / 4 : tid] = fours ? four : key;
    if (tid == 0) {
        floor_key = 0xFFFFFFFFu;
        listed = survived[0] = survived[1] = more = 0;
    }
    float m = wave_max(gm);
    if (lane == 0) sh.red_f[wave] = m;
    __syncthreads();
    m = sh.red_f[0];
#pragma unroll
    for (int w = 1; w < SAMPLE_THREADS / WAVE; w++) m = fmaxf(m, sh.red_f[w]);
    float sum = wave_sum(gm > -INFINITY ? gs * expf(gm - m) : 0.f);
    if (lane == 0) red_sum[wave] = sum;
    // the K-th largest of the units' keys: the least of those with fewer than K above them; four threads count for one unit
    if (tid / WAVE * (WAVE / 4) < units) {
        const int unit = tid / 4, part = (units + 15) / 16 * 4, from = (tid & 3) * part;
        const unsigned mine = unit_key[unit];
        unsigned above = 0;
#pragma unroll 2
        for (int c = from; c < from + part; c += 4) {  // (units <= 256: the last part ends within unit_key, and keys past the units are 0)
            const u32x4 o = *reinterpret_cast<const u32x4 *>(&unit_key[c]);
#pragma unroll
            for (int u = 0; u < 4; u++) above += o[u] > mine ? 1u : 0u;
        }
        above += dpp_keys<0xB1, 0xF>(above);
        above += dpp_keys<0x4E, 0xF>(above);
        if ((tid & 3) == 0 && unit < units && above < K) atomicMin(&floor_key, mine);
    }
    __syncthreads();
    sum = 0.f;
#pragma unroll
    for (int w = 0; w < SAMPLE_THREADS / WAVE; w++) sum += red_sum[w];
    // What lies 104 below the maximum has the probability 0, of which nothing below depends: a vocabulary masked down to fewer than K
    // tokens keeps those. (fmaxf leaves no NaN in m; behind an infinite m, or a min_p that leaves no token a probability, the floor stays.)
    unsigned floor = m < INFINITY && a.cfg.min_p <= 1.0f ? max(floor_key, order_key(m - 104.0f)) : floor_key;
    auto weight = [&](unsigned k) {
        const float x = key_value(k);
        return x > -INFINITY ? expf(x - m) : 0.f;
    };
    int round = 0;  // 1: with groups read again
    auto survive = [&](unsigned k, int token) {
        const unsigned at = atomicAdd(&survived[round], 1u);
        if (at < (unsigned)SAMPLE_MAX_K) fcomp[at] = ((unsigned long long)k << 32) | (unsigned)(0x7FFFFFFF - token);
    };
    bool in = tid < groups && key >= floor;
    auto keep = [&](unsigned k0, unsigned k1, unsigned k2, unsigned k3, unsigned i0, unsigned i1, unsigned i2, unsigned i3) {
#pragma unroll 1
        for (int u = 0; u < FRONT_KEEP && k0 >= floor; u++) {
            survive(k0, (int)i0);
            k0 = k1, k1 = k2, k2 = k3, k3 = 0u;
            i0 = i1, i1 = i2, i2 = i3, i3 = 0u;
        }
    };
    if (in) {
        keep(kept_key[0], kept_key[1], kept_key[2], kept_key[3], kept_token[0], kept_token[1], kept_token[2], kept_token[3]);
        if (kept_key[3] >= floor) more = 1;
    }
    // survivors ahead of `mine`, one of n, for which 1 << bits threads count
    auto survivors_ahead = [&](unsigned long long mine, int n, int bits) {
        unsigned rank = 0;
#pragma unroll 4
        for (int c = tid & ((1 << bits) - 1); c < n; c += 1 << bits) rank += fcomp[c] > mine ? 1u : 0u;
        if (bits > 0) rank += dpp_keys<0xB1, 0xF>(rank);
        if (bits > 1) rank += dpp_keys<0x4E, 0xF>(rank);
        if (bits > 2) rank += dpp_keys<0x141, 0xF>(rank);
        return rank;
    };
    auto threads_for = [](int n) { return n <= SAMPLE_THREADS / 8 ? 3 : n <= SAMPLE_THREADS / 4 ? 2 : n <= SAMPLE_THREADS / 2 ? 1 : 0; };
    __syncthreads();
    if (more || survived[0] > (unsigned)SAMPLE_MAX_K) {
        // A group may have more than it kept, or the list takes no more: only groups all of whose kept tokens reach the floor are read again.
        // Of more than SAMPLE_THREADS / 8 survivors the K-th is a better floor to begin with (fewer have 32 such groups at most, which is one
        // trip to memory). Of the groups that end at the floor itself (equal keys all over the vocabulary) the first in token order are
        // taken that, with one token of each group above the floor, surely hold K tokens ahead of all others': as many of a group as it kept,
        // then, of these groups, as many as it has.
        const int had = (int)survived[0];
        round = 1;
        if (had > SAMPLE_THREADS / 8 && had <= SAMPLE_THREADS / 2) {
            const int bits = threads_for(had);
            const unsigned long long mine = fcomp[min(tid >> bits, had - 1)];
            if (survivors_ahead(mine, had, bits) == K - 1) floor_key = (unsigned)(mine >> 32);
            __syncthreads();
            floor = max(floor, floor_key);
        } else if (had > SAMPLE_THREADS / 2 && had <= SAMPLE_MAX_K) {  // (counting as above is had compares a thread: 1000 of them 25 us, this 11)
            const unsigned mine = tid < had ? (unsigned)(fcomp[tid] >> 32) : 0u;
            const int bits = 32 - __clz((int)(floor ^ order_key(m)));  // below the ones that all keys from the floor to the maximum share
            unsigned kth = bits < 32 ? floor >> bits << bits : 0u;
            for (int bit = bits - 1; bit >= 0; bit--)
                if (__syncthreads_count(mine >= (kth | 1u << bit)) >= (int)K) kth |= 1u << bit;
            floor = max(floor, kth);
        }
        in = in && key >= floor;
        bool full = in && kept_key[3] >= floor, at_floor = in && key == floor;
        if (full) list[atomicAdd(&listed, 1u)] = tid;
        auto first_groups = [&](unsigned has) {  // drops groups at the floor
            const unsigned mine = at_floor ? has : in ? 1u << 20 : 0u;
            unsigned before = mine;
            for (int off = 1; off < WAVE; off <<= 1) {
                const unsigned up = __shfl_up(before, off, WAVE);
                if (lane >= off) before += up;
            }
            if (lane == WAVE - 1) sh.red_i[wave] = (int)before;
            __syncthreads();
            before -= mine;
            unsigned above = 0;
            for (int w = 0; w < SAMPLE_THREADS / WAVE; w++) {
                if (w < wave) before += (unsigned)sh.red_i[w];
                above += (unsigned)sh.red_i[w] >> 20;
            }
            at_floor = at_floor && above + (before & 0xFFFFFu) < K;
            in = in && (at_floor || key > floor);
            full = full && in;
            __syncthreads();
        };
        auto enlist = [&](bool mine) {  // lists groups in order; how many
            const unsigned long long mask = __ballot(mine);
            if (lane == 0) sh.red_i[wave] = __popcll(mask);
            __syncthreads();
            int at = __popcll(mask & ((1ull << lane) - 1ull)), all = 0;
            for (int w = 0; w < SAMPLE_THREADS / WAVE; w++) {
                if (w < wave) at += sh.red_i[w];
                all += sh.red_i[w];
            }
            if (mine) list[at] = tid;
            fcomp[tid] = 0;
            __syncthreads();
            return all;
        };
        auto token_at = [&](int j) { return (list[j >> group_bits] << group_bits) + (j & ((1 << group_bits) - 1)); };
        auto logit_at = [&](int j) {
            const int i = min(token_at(j), a.vocab - 1);
            return LogitAndCount{a.logits[i], a.counts ? a.counts[i] : 0};
        };
        // (tokens past the vocabulary come last: the smallest key, the largest number)
        auto key_of = [&](int j, LogitAndCount v) { return token_at(j) < a.vocab ? order_key(penalised(v.l, v.c, a.cfg) * inv_temp) : 0u; };
        auto idx_at = [&](int j) { return token_at(j) < a.vocab ? token_at(j) : 0x7FFFFFFF; };
        const int n_floor = __syncthreads_count(at_floor);
        int n_list = (int)listed;
        if (n_floor > 1) {
            const unsigned reach = 1u + (kept_key[1] >= floor) + (kept_key[2] >= floor) + (kept_key[3] >= floor);
            first_groups(reach);
            n_list = enlist(full);
            sweep(n_list << group_bits, tid, logit_at, [&](int j, LogitAndCount v) {  // (a wavefront's tokens are of one group)
                const unsigned long long has = __ballot(key_of(j, v) >= floor);
                if (lane == 0) atomicAdd(&fcomp[list[j >> group_bits]], (unsigned long long)__popcll(has));
            });
            __syncthreads();
            first_groups(full ? (unsigned)min(fcomp[tid], (unsigned long long)K) : reach);
            n_list = enlist(full);
        }
        if (in && !full) keep(kept_key[0], kept_key[1], kept_key[2], kept_key[3], kept_token[0], kept_token[1], kept_token[2], kept_token[3]);
        sweep(n_list << group_bits, tid, logit_at, [&](int j, LogitAndCount v) {
            const unsigned k = key_of(j, v);
            if (k >= floor) survive(k, idx_at(j));
        });
        __syncthreads();
        if (survived[1] > (unsigned)SAMPLE_MAX_K) {  // a flat distribution: the general selection, which wants its items in token order
            const int n = enlist(in) << group_bits;
            select_sort_draw(sh, a, st, n, a.vocab, sum, [&](int j) { return key_of(j, logit_at(j)); }, idx_at, weight);
            return;
        }
    }
    // Selection by rank: every survivor counts the survivors ahead of it, and the first K take their rank as their
    // place.
    const int nf = (int)survived[round];
    float (&cand_p)[SAMPLE_MAX_K] = sh.cand_p;
    int (&cand_i)[SAMPLE_MAX_K] = sh.cand_i;
    {
        const int bits = threads_for(nf), s = tid >> bits;
        const unsigned long long mine = fcomp[min(s, nf - 1)];
        const unsigned rank = survivors_ahead(mine, nf, bits);
        if (s < nf && rank < K) {  // normalise, min_p (the maximum probability is exp(0) / sum)
            float p = weight((unsigned)(mine >> 32)) / sum;
            if (a.cfg.min_p > 0.0f && p < a.cfg.min_p * (1.0f / sum)) p = 0.0f;
            cand_p[rank] = p;
            cand_i[rank] = 0x7FFFFFFF - (int)(unsigned)(mine & 0xFFFFFFFFull);
        }
    }
    __syncthreads();
    if (wave != 0) return;
    // K <= 64 candidates, one per lane, in the order the reference's sequential loops walk (src/generate.rs:771-800):
    // probability descending, token ascending. That is their order already, except where two logits have one
    // probability (rounding, min_p).
    const int nc = min((int)K, nf);
    float p = lane < nc ? cand_p[lane] : 0.0f;
    int ci = lane < nc ? cand_i[lane] : 0;
    const float p_next = __shfl_down(p, 1, WAVE);
    const int i_next = __shfl_down(ci, 1, WAVE);
    if (__ballot(lane + 1 < nc && !cand_before(p, ci, p_next, i_next))) {
        int place = 0;
        for (int c = 0; c < nc; c++) {
            const float pc = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(p), c));
            const int ic = __builtin_amdgcn_readlane(ci, c);
            place += cand_before(pc, ic, p, ci) ? 1 : 0;
        }
        // lane l wants the candidate whose place is l: scatter through LDS, where every place holds a candidate before
        // (wavefront 0 only; no other wavefront touches cand_p / cand_i any more, and a wavefront's LDS operations
        // execute in order)
        if (lane < nc) {
            cand_p[place] = p;
            cand_i[place] = ci;
        }
        __builtin_amdgcn_wave_barrier();
        p = lane < nc ? cand_p[lane] : 0.0f;
        ci = lane < nc ? cand_i[lane] : 0;
    }
    // The reference's three loops add the same probabilities in the same order from zero: cumulative until top_p is
    // reached, the total of the kept candidates (= that cumulative sum), and the running sum the draw is compared
    // with. One chain of additions gives all three, lane i ends with the sum after candidate i: every step adds to each
    // lane's p the lane before's sum (0 ahead of lane 0), and the i-th step leaves lane i - 1's at its last value.
    float upto = 0.0f;
    for (int i = 0; i < nc; i += 8)
#pragma unroll
        for (int u = 0; u < 8; u++) upto = dpp_move<0x138, 0xF>(upto, 0.0f) + p;  // wave_shr:1
    const unsigned long long live = nc >= WAVE ? ~0ull : ((1ull << nc) - 1ull);
    const unsigned long long reached = __ballot(upto >= a.cfg.top_p) & live;
    const int cutoff = reached ? __ffsll((long long)reached) : nc;  // index of the first + 1
    const float total = cutoff > 0 ? __int_as_float(__builtin_amdgcn_readlane(__float_as_int(upto), cutoff - 1)) : 0.0f;
    const float r = st.draw * total;
    const unsigned long long kept = cutoff >= WAVE ? ~0ull : ((1ull << cutoff) - 1ull);
    const unsigned long long hit = __ballot(upto >= r) & kept;
    const int at = hit ? __ffsll((long long)hit) - 1 : cutoff - 1;
    const int pick = at >= 0 ? __builtin_amdgcn_readlane(ci, at) : 0;
    if (lane == 0) deliver_pick(a, st, pick);
}

__global__ void count_tokens_kernel(const uint32_t *__restrict__ ids, int n_ids, int *__restrict__ counts, int vocab) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n_ids && ids[i] < (uint32_t)vocab) atomicAdd(&counts[ids[i]], 1);
}

__global__ void zero_ints_kernel(int *__restrict__ p, size_t n) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

}  // namespace

namespace homura {

int sample_check_config(hm_ctx *ctx, const hm_sampling_config *cfg, bool device) {
    HM_REQUIRE(ctx, cfg != nullptr, "sampling: NULL configuration");
    HM_REQUIRE(ctx, cfg->top_k >= 0 && cfg->top_p > 0.0f && cfg->min_p >= 0.0f && cfg->repetition_penalty > 0.0f,
               "sampling: need top_k >= 0, top_p > 0, min_p >= 0, repetition_penalty > 0");
    if (device && cfg->temperature > 0.0f)
        HM_REQUIRE(ctx, cfg->top_k >= 1 && cfg->top_k <= SAMPLE_MAX_K,
                   "sampling on the device needs 1 <= top_k <= %d (got %d); use the host sampler", SAMPLE_MAX_K, cfg->top_k);
    return HM_OK;
}

// One workgroup for everything, or the front / back pair when top_k is small and the vocabulary large (the pair
// keeps ten words per group in `work`, which has a word per token: a group has 64 tokens or more, but for the last one).
static_assert((2 * FRONT_KEEP + 2) * 2 <= 1 << FRONT_GROUP_BITS, "front_out fits a word per token, the last group's too");
static int sample_enqueue(hm_ctx *ctx, const SampleArgs &a) {
    const bool pair = a.cfg.temperature > 0.0f && a.cfg.top_k >= 1 && a.cfg.top_k <= FRONT_MAX_K && a.vocab >= 4096;
    if (pair) {
        int bits = FRONT_GROUP_BITS;
        while (((a.vocab - 1) >> bits) + 1 > SAMPLE_THREADS) bits++;
        const int groups = ((a.vocab - 1) >> bits) + 1, per_block = FRONT_THREADS / WAVE;
        hipLaunchKernelGGL(sample_front_kernel, dim3((groups + per_block - 1) / per_block), dim3(FRONT_THREADS), 0, ctx->stream, a, groups, bits);
        HM_LAUNCH_CHECK(ctx);
        hipLaunchKernelGGL(sample_back_kernel, dim3(1), dim3(SAMPLE_THREADS), 0, ctx->stream, a, groups, bits);
    } else {
        hipLaunchKernelGGL(sample_token_kernel, dim3(1), dim3(SAMPLE_THREADS), 0, ctx->stream, a);
    }
    HM_LAUNCH_CHECK(ctx);
    return HM_OK;
}

// counts: device [vocab] occurrences (or nullptr); work: device [vocab] floats
int sample_token_launch(hm_ctx *ctx, const float *d_logits, float *d_work, const int *d_counts, int vocab,
                        const hm_sampling_config &cfg, float draw, int32_t *d_out, int *d_counts_update, int32_t *d_list,
                        int list_pos) {
    SampleArgs a;
    a.logits = d_logits;
    a.work = d_work;
    a.counts = d_counts;
    a.vocab = vocab;
    a.cfg = cfg;
    a.draw = draw;
    a.out = d_out;
    a.counts_update = d_counts_update;
    a.list = d_list;
    a.list_pos = list_pos;
    a.cursor = nullptr;
    a.draws = nullptr;
    a.eos = -1;
    a.stop = nullptr;
    return sample_enqueue(ctx, a);
}

// The sampler behind a decode step whose cursor has already moved on: no argument depends on the step, so the
// host can enqueue step after step without reading anything back.
int sample_step_launch(hm_ctx *ctx, const float *d_logits, float *d_work, int *d_counts, int vocab,
                       const hm_sampling_config &cfg, DecodeState *d_cursor, const float *d_draws, int32_t *d_list,
                       int eos, int *d_stop, int32_t *d_out) {
    SampleArgs a;
    a.logits = d_logits;
    a.work = d_work;
    a.counts = d_counts;
    a.vocab = vocab;
    a.cfg = cfg;
    a.draw = 0.0f;
    a.out = d_out;
    a.counts_update = d_counts;
    a.list = d_list;
    a.list_pos = 0;
    a.cursor = d_cursor;
    a.draws = d_draws;
    a.eos = eos;
    a.stop = d_stop;
    return sample_enqueue(ctx, a);
}

int zero_ints_launch(hm_ctx *ctx, int *d, size_t n) {
    if (n == 0) return HM_OK;
    hipLaunchKernelGGL(zero_ints_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, ctx->stream, d, n);
    HM_LAUNCH_CHECK(ctx);
    return HM_OK;
}

}  // namespace homura

extern "C" {

uint64_t hm_rng_seed(uint64_t seed) { return seed | 1u; }

float hm_rng_next_f32(uint64_t *state) {
    uint64_t s = *state;
    s ^= s << 13;
    s ^= s >> 7;
    s ^= s << 17;
    *state = s;
    return (float)(s >> 40) / (float)(1ull << 24);
}

int hm_sample_token_host(const float *h_logits, int vocab, const hm_sampling_config *cfg, const uint32_t *h_generated,
                         int n_generated, uint64_t *rng_state, int32_t *token_out) {
    if (!h_logits || vocab <= 0 || !cfg || !rng_state || !token_out || n_generated < 0 || (n_generated && !h_generated))
        return HM_ERR_INVALID;
    std::vector<float> logits(h_logits, h_logits + vocab);
    if (cfg->repetition_penalty != 1.0f)
        for (int g = 0; g < n_generated; g++) {
            const uint32_t idx = h_generated[g];
            if (idx < (uint32_t)vocab) {
                if (logits[idx] > 0.0f)
                    logits[idx] /= cfg->repetition_penalty;
                else
                    logits[idx] *= cfg->repetition_penalty;
            }
        }
    if (cfg->frequency_penalty != 0.0f || cfg->presence_penalty != 0.0f) {
        std::vector<int> counts(vocab, 0);
        for (int g = 0; g < n_generated; g++)
            if (h_generated[g] < (uint32_t)vocab) counts[h_generated[g]]++;
        for (int i = 0; i < vocab; i++)
            if (counts[i]) {
                logits[i] -= cfg->frequency_penalty * (float)counts[i];
                logits[i] -= cfg->presence_penalty;
            }
    }
    if (cfg->temperature <= 0.0f) {  // greedy: the last of equal maxima (Rust max_by)
        int best = 0;
        for (int i = 1; i < vocab; i++)
            if (!(logits[best] > logits[i])) best = i;
        *token_out = best;
        return HM_OK;
    }
    const float inv_temp = 1.0f / cfg->temperature;
    float max_logit = -INFINITY;
    for (float &l : logits) {
        l *= inv_temp;
        max_logit = std::fmax(max_logit, l);
    }
    struct Cand {
        int idx;
        float p;
    };
    std::vector<Cand> c(vocab);
    float sum = 0.0f;
    for (int i = 0; i < vocab; i++) {
        c[i] = Cand{i, std::exp(logits[i] - max_logit)};
        sum += c[i].p;
    }
    for (Cand &x : c) x.p /= sum;
    if (cfg->min_p > 0.0f) {
        float max_prob = 0.0f;
        for (const Cand &x : c) max_prob = std::fmax(max_prob, x.p);
        const float threshold = cfg->min_p * max_prob;
        for (Cand &x : c)
            if (x.p < threshold) x.p = 0.0f;
    }
    // probability descending; the reference's sort_unstable_by leaves equal probabilities in an
    // unspecified order, here they keep index order
    std::sort(c.begin(), c.end(), [](const Cand &x, const Cand &y) { return x.p > y.p || (x.p == y.p && x.idx < y.idx); });
    size_t len = c.size();
    if (cfg->top_k > 0 && (size_t)cfg->top_k < len) len = (size_t)cfg->top_k;
    float cumulative = 0.0f;
    size_t cutoff = len;
    for (size_t i = 0; i < len; i++) {
        cumulative += c[i].p;
        if (cumulative >= cfg->top_p) {
            cutoff = i + 1;
            break;
        }
    }
    float total = 0.0f;
    for (size_t i = 0; i < cutoff; i++) total += c[i].p;
    const float r = hm_rng_next_f32(rng_state) * total;
    float accum = 0.0f;
    int pick = cutoff > 0 ? c[cutoff - 1].idx : 0;
    for (size_t i = 0; i < cutoff; i++) {
        accum += c[i].p;
        if (accum >= r) {
            pick = c[i].idx;
            break;
        }
    }
    *token_out = pick;
    return HM_OK;
}

int hm_sample_token(hm_ctx *ctx, const float *d_logits, int vocab, const hm_sampling_config *cfg,
                    const uint32_t *h_generated, int n_generated, uint64_t *rng_state, int32_t *token_out) {
    HM_CHECK_CTX(ctx);
    HM_REQUIRE(ctx, d_logits && vocab > 0 && rng_state && token_out && n_generated >= 0 && (!n_generated || h_generated),
               "hm_sample_token: bad arguments");
    int rc = homura::sample_check_config(ctx, cfg, true);
    if (rc != HM_OK) return rc;
    // workspace: work [vocab] f32 | counts [vocab] i32 | token i32 | generated ids
    const size_t need = (size_t)vocab * 8 + 256 + (size_t)n_generated * 4;
    HM_REQUIRE(ctx, need <= ctx->workspace_bytes, "hm_sample_token: vocabulary / history too large for the workspace");
    float *work = (float *)ctx->workspace;
    int *counts = (int *)(work + vocab);
    int32_t *d_tok = (int32_t *)(counts + vocab);
    uint32_t *d_gen = (uint32_t *)((char *)d_tok + 256);
    const bool need_counts = n_generated > 0 && (cfg->repetition_penalty != 1.0f || cfg->frequency_penalty != 0.0f ||
                                                 cfg->presence_penalty != 0.0f);
    if (need_counts) {
        if ((rc = homura::zero_ints_launch(ctx, counts, (size_t)vocab)) != HM_OK) return rc;
        if ((rc = hm_upload(ctx, d_gen, h_generated, (size_t)n_generated * 4)) != HM_OK) return rc;
        hipLaunchKernelGGL(count_tokens_kernel, dim3((unsigned)((n_generated + 255) / 256)), dim3(256), 0, ctx->stream,
                           d_gen, n_generated, counts, vocab);
        HM_LAUNCH_CHECK(ctx);
    }
    const float draw = cfg->temperature > 0.0f ? hm_rng_next_f32(rng_state) : 0.0f;  // greedy leaves the stream alone
    rc = homura::sample_token_launch(ctx, d_logits, work, need_counts ? counts : nullptr, vocab, *cfg, draw, d_tok, nullptr,
                                     nullptr, 0);
    if (rc != HM_OK) return rc;
    return hm_download(ctx, token_out, d_tok, 4);
}

}  // extern "C"
