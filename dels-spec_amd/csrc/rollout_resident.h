// Pieces shared by the rollouts that hold the low-rank head's B on chip
// (rollout_resident.hip, markov_resident.hip): the tagged-word exchanges
// between the workgroups of one launch.
#pragma once

#include <algorithm>
#include <climits>

#include "dels_device.h"
#include "dels_internal.h"

namespace dels {

constexpr int kRrWaves = 8;
constexpr int kRrThreads = kRrWaves * 64;
constexpr int kRrRegTiles = 4;                        // vocabulary tiles per wave in registers

// control area: one 128-byte line (32 words) per counter
constexpr int kRrDoneCounter = 250 * 32;
constexpr int kRrErrorWord = 251 * 32;
constexpr int kRrNotDoneWord = 252 * 32;              // a resident launch left its rollout to the ordered one
constexpr int kRrTicketWord = 253 * 32;               // the ordered rollout's next task
constexpr int kRrExitCounter = 254 * 32;              // ... and its workgroups that have run out of tasks
static_assert(kRrExitCounter < kMaxCounters, "the control words lie below the line that persists");

// Polls for the other workgroups' arrival (about 1 us each) before a launch
// that has a stand-in gives up.
constexpr int kRrArrivalLimit = 2048;

constexpr int kRrSlotSet = 16 * kResidentMaxWGs;      // slot words of 16 rows per parity set

__device__ __forceinline__ uint32_t rr_tag(uint32_t gen, int step) {
    const uint32_t x = gen * 256u + (uint32_t)step + 1u;
    const uint32_t t = x * 0x2C1B3C6Du;
    return t == 0u ? 0x5bd1e995u : t;
}

template <typename Args>
__device__ __forceinline__ bool rr_failed(const Args& a) {
    return __hip_atomic_load(a.counters + kRrErrorWord, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u;
}
template <typename Args>
__device__ __forceinline__ void rr_fail(const Args& a) {
    __hip_atomic_store(a.counters + kRrErrorWord, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Where a reader finds the words of one exchange.  Every producer writes its
// words as one block (rows x words per row, the rows rounded up to a power of
// two) starting on its own 128-byte line or lines: when one line gathers words
// of many producers, their writes and the readers' polls of it queue behind one
// another (an all-to-all of 256 x 8 words takes ~1.9 us with a line per
// producer, ~3.4 us with sixteen producers per line).  The reader numbers the
// words j < n = producers << blk and takes them in that order.
struct RrWords {
    int n;        // words the reader takes
    int blk;      // log2 of one producer's block (rows rounded up x words per row)
    int stride;   // log2 of the words from one producer's block to the next (>= blk)
    int row;      // log2 of the words per row
    int mp;       // log2 of the rows rounded up
    int M;        // rows present
    int split = INT_MAX, M2 = 0;   // from word `split` on: a second group, of M2 rows
    __device__ __forceinline__ uint32_t addr(int j) const {
        j = j < n ? j : n - 1;   // past the end: the last word again (loaded, never examined)
        return ((uint32_t)(j >> blk) << stride) + (uint32_t)(j & ((1 << blk) - 1));
    }
    __device__ __forceinline__ int row_of(int j) const { return (j >> row) & ((1 << mp) - 1); }
    __device__ __forceinline__ bool live(int j) const { return j < n && row_of(j) < (j < split ? M : M2); }
};

// Load the words j = tid + kRrThreads * i, i < NPT -- every load issued before
// any value is examined -- then re-read the live ones that `arrived` rejects,
// at most spin_limit rounds.  False when they did not all arrive or another
// workgroup reported a failure (this thread's view).
template <int NPT, typename Args, typename Arrived>
__device__ __forceinline__ bool rr_gather(const Args& a, const unsigned long long* src, const RrWords& pl, int tid,
                                          unsigned long long (&w)[NPT], Arrived arrived) {
    static_assert(NPT <= 32, "one bit per word in a 32-bit mask");
#pragma unroll
    for (int i = 0; i < NPT; ++i)
        w[i] = __hip_atomic_load(src + pl.addr(tid + kRrThreads * i), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    uint32_t missing = 0;
#pragma unroll
    for (int i = 0; i < NPT; ++i)
        if (pl.live(tid + kRrThreads * i)) missing |= (uint32_t)!arrived(w[i]) << i;
    int it = 0;
    while (missing != 0) {
        // poll the first missing word alone (one load per thread and round, not
        // one per missing word: the polls of every workgroup share the memory
        // system with the words being written), then re-read the rest once
        const int f = __builtin_ctz(missing);
        const unsigned long long* pf = src + pl.addr(tid + kRrThreads * f);
        for (;;) {
            if (it >= a.spin_limit) return false;
            if ((it & 63) == 63 && rr_failed(a)) return false;
            ++it;
            __builtin_amdgcn_s_sleep(2);
            if (arrived(__hip_atomic_load(pf, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))) break;
        }
#pragma unroll
        for (int i = 0; i < NPT; ++i)
            if ((missing >> i) & 1u)
                w[i] = __hip_atomic_load(src + pl.addr(tid + kRrThreads * i), __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT);
        uint32_t still = 0;
#pragma unroll
        for (int i = 0; i < NPT; ++i)
            if ((missing >> i) & 1u) still |= (uint32_t)!arrived(w[i]) << i;
        missing = still;
    }
    return true;
}

// Read the tagged words of `pl` until every live one carries `tag` (word j to
// the LDS pair slot map(j)); all threads.  Returns false (for every thread)
// when they did not all arrive.  Ends with a barrier.
template <int NPT, typename Args, typename Map>
__device__ __forceinline__ bool rr_read_words(const Args& a, const unsigned long long* src, const RrWords& pl,
                                              uint32_t tag, Map map) {
    // the thread index passes through an empty asm statement so that the word
    // addresses are formed here, not held in registers across the caller's loop
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    unsigned long long w[NPT];
    const bool got = rr_gather<NPT>(a, src, pl, tid, w,
                                    [&](unsigned long long x) { return (uint32_t)(x >> 32) == tag; });
    if (got) {
#pragma unroll
        for (int i = 0; i < NPT; ++i) {
            const int j = tid + kRrThreads * i;
            if (pl.live(j)) *map(j) = (uint32_t)w[i];
        }
    }
    return !__syncthreads_or(!got);
}

// The step's slot words (one per row and workgroup, `pl` with one word per row)
// once every live one carries the step's flag bits `low2`; each row's maximum
// into s_rowmax[row] (an LDS maximum, s_rowmax zero before).  All threads;
// false for every thread when they did not all arrive.  Ends with a barrier.
template <int NPT, typename Args>
__device__ __forceinline__ bool rr_slot_maxima(const Args& a, const unsigned long long* src, const RrWords& pl,
                                               uint32_t low2, unsigned long long* s_rowmax) {
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    unsigned long long w[NPT];
    const bool got = rr_gather<NPT>(a, src, pl, tid, w,
                                    [&](unsigned long long x) { return ((uint32_t)x & 3u) == low2; });
    // word j holds row j mod 2^mp, so lanes with equal low mp bits share a row
    const int lane = tid & 63;
    unsigned long long k = 0;
#pragma unroll
    for (int i = 0; i < NPT; ++i) {
        const unsigned long long v = got && pl.live(tid + kRrThreads * i) ? w[i] : 0ull;
        k = v > k ? v : k;
    }
    for (int off = 1 << pl.mp; off < 64; off <<= 1) {
        const unsigned long long o = __shfl_xor(k, off, 64);
        k = o > k ? o : k;
    }
    if (lane < pl.M && lane < (1 << pl.mp)) atomicMax(&s_rowmax[lane], k);
    return !__syncthreads_or(!got);
}

// One step of a maximum over the 16 lanes of each DPP row of 64-bit argmax keys
// (pack_argmax): every lane takes the larger of its key and that of the lane K
// below it in its row (lanes with none read key 0, the lowest).  After K = 1,
// 2, 4, 8 lane 15 of a row holds the row's best.
template <int K>
__device__ __forceinline__ void rr_row_max(unsigned long long& k) {
    constexpr int kRowShr = 0x110 + K;
    const uint32_t lo = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)k, kRowShr, 0xf, 0xf, true);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)(k >> 32), kRowShr, 0xf, 0xf, true);
    const unsigned long long o = ((unsigned long long)hi << 32) | lo;
    k = o > k ? o : k;
}

}  // namespace dels
