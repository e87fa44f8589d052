// Partial results of a launch's workgroups joined by the last of them, inside one accelerator die.
//
// Workgroups are dealt to the eight dies round-robin, so those with the same blockIdx.x % 8 share an L2 (hm_init looks whether they do:
// hm_ctx::dies_round_robin). A group of splits that sits on one die can hand its results over through that L2 without a fence: every
// workgroup stores its results, waits until the L2 has them, and counts itself in; the one that finds all others counted reads them back
// past its L1 and folds. Nobody waits for anybody. The counting says by die who came: a launch whose groups were dealt
// otherwise after all tells the host, which fails the next synchronisation instead of handing out what was folded from another die's memory. A launch of its own for the fold costs a kernel boundary and two trips to memory;
// between dies the hand-over itself takes them (a counter and stores through memory made the attention launch 4.9 us longer to
// save 4.1 of fold).
#pragma once
#include "hm_common.h"

namespace homura {

constexpr int DIES = 8, DIE_SPLITS_MAX = 32;
// A counter has a cache line of its own: two dies counting in one line pass it to and fro (256 workgroups' arrivals 3.7 us instead of 0.6).
// Its bytes are the arrivals from the eight dies.
constexpr int DIE_COUNTER_STRIDE = 32;

// Group p's split s is workgroup (p / 8 * splits + s) * 8 + p % 8 of a one-dimensional grid.
__host__ __device__ inline int die_grid(int groups, int splits) { return (groups + DIES - 1) / DIES * splits * DIES; }
__device__ __forceinline__ void die_place(int block, int splits, int &group, int &split) {
    const int r = block / DIES;
    split = r % splits;
    group = r / splits * DIES + block % DIES;
}

// Whether a launch of `groups` groups of up to `splits` splits that reads `bytes` in all goes this way: the groups on at least half of the dies,
// not two workgroups on some CUs and one on others, and no more than 1 us of reading lost to dies with fewer groups. us with the fold in
// a launch of its own / here, replayed: 1 sequence x 16 heads on 8 x 128, 300 / 1000 / 4000 rows 6.97 / 6.2, 7.31 / 6.35, 9.42 / 7.95; 32 on 4 x 64,
// 1000 rows 7.75 / 6.7; 32 on 32 x 64, 500 rows 6.39 / 6.0; 2 x 12 on 2 x 128, 1000 rows 8.02 / 7.0; 8 x 12 on 2, 4096 rows 11.7 / 11.4; 8 x 14
// on 2 x 64, 5000 rows 11.0 / 10.3; and 3 x 32 on 4 x 64, 8000 rows (12 groups of 22 splits) 11.05 / 13.4, which this rule leaves alone.
inline bool die_fold_pays(const hm_ctx *ctx, long long groups, int splits, double bytes) {
    if (!ctx->dies_round_robin || splits < 2 || splits > DIE_SPLITS_MAX || groups < 1 || groups > (long long)ctx->num_counters / DIE_COUNTER_STRIDE)
        return false;
    const long long most = (groups + DIES - 1) / DIES;  // groups of a die
    return groups >= DIES / 2 && (most * splits <= ctx->num_cus / DIES || most * DIES == groups) && bytes / 6.2e6 * ((double)(most * DIES) / groups - 1) <= 1;
}

__device__ __forceinline__ int die_id() { return __builtin_amdgcn_s_getreg((3 << 11) | (0 << 6) | 20) & 0xF; }  // XCC_ID

// Called by all threads behind their last store of results; true in every thread of the workgroup that is the last of n to come here.
// The counter is left at zero. If they came from several dies nobody is, and `apart` (memory of the host's) is set.
__device__ __forceinline__ bool last_on_die(unsigned long long *counters, int group, int n, int *apart) {
    __shared__ int last;
    unsigned long long *counter = counters + (size_t)group * DIE_COUNTER_STRIDE;
    const int shift = die_id() % DIES * 8;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the L2 has this wavefront's stores
    __syncthreads();
    if (threadIdx.x == 0) {
        const unsigned long long came = __hip_atomic_fetch_add(counter, 1ull << shift, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const bool all = (int)((came * 0x0101010101010101ull) >> 56) == n - 1;  // (the sum of its bytes, at most 31)
        last = all && came >> shift == (unsigned)(n - 1);
        if (all) __hip_atomic_store(counter, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (all && !last) __hip_atomic_store(apart, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    __syncthreads();
    return last != 0;
}

// A result that another workgroup of the die stored: from the L2, whatever this CU's L1 holds
__device__ __forceinline__ float from_die(const float *p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
// Four at once, for results in cache lines of their own that no workgroup of this launch has read before (a kernel begins with an empty L1, and
// its own stores go through it). Past the L1 as above, eight bytes at a time: 8 sequences x 12 heads on 2 x 128, 4096 rows 11.83 -> 12.09 us.
constexpr int DIE_LINE = 128;  // bytes
__device__ __forceinline__ f32x4 from_die4(const float *p) { return __builtin_nontemporal_load(reinterpret_cast<const f32x4 *>(p)); }

}  // namespace homura
