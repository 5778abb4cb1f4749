// Pieces shared by the rollouts that hold the low-rank head's B on chip
// (rollout_resident.hip, markov_resident.hip): the tagged-word exchanges
// between the workgroups of one launch.
#pragma once

#include <algorithm>
#include <climits>

#include "dels_device.h"
#include "dels_internal.h"
#include "fused_argmax_rows.h"

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
// that has a stand-in gives up.  Workgroups of other streams' kernels usually end
// in well under that and the rollout then has their CUs: beside a stream of 4096 x
// 4096 x 4096 products it takes 319 us (Markov, 4 rows) and 444 (DeLS, 24), of
// 256 MB copies 161 and 458.  Giving up at 512 polls leaves the last of these to
// the stand-in, at 2472 us.
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

// The prior in LDS: a float per column of the workgroup's tiles, then a tile of zeros.
constexpr int kRrPriorZeros = (kRrWaves * kRrRegTiles + kResidentLdsTiles) * 16;
constexpr int kRrPriorWords = kRrPriorZeros + 16;

// Base logits of the wave's tiles for one group of 16 rows: lane (col, kg) takes
// row `col` of the group, columns 4 kg .. 4 kg + 3 of each tile, as one 8- or
// 16-byte load per tile.  VEC: V and the row stride multiples of four, the base
// aligned to four elements.  (Element loads take a line per row each: twenty of
// them per lane and group made a vocabulary of 50257 slower than one of 151936.)
template <typename BaseT>
using RrBase = rows::Quad<BaseT>[kRrRegTiles + 1];

// `row`: the lane's row of the step.  Tiles past the workgroup's repeat its last one.
template <typename BaseT, bool VEC>
__device__ __forceinline__ void rr_load_base(const BaseT* row, int T0, int ntl, int ntiles, int wave, int kg, int V,
                                             RrBase<BaseT>& w) {
#pragma unroll
    for (int j = 0; j <= kRrRegTiles; ++j) {
        const int tc = min(T0 + min(wave + 8 * j, max(ntl - 1, 0)), ntiles - 1);
        const int v = tc * 16 + 4 * kg;
        if constexpr (VEC) {
            const BaseT* p = row + min(v, V - 4);
            if constexpr (sizeof(BaseT) == 2) {
                const u32x2 x = *reinterpret_cast<const u32x2*>(p);
                w[j][0] = x[0]; w[j][1] = x[1];
            } else {
                const u32x4 x = *reinterpret_cast<const u32x4*>(p);
#pragma unroll
                for (int q = 0; q < 4; ++q) w[j][q] = x[q];
            }
        } else if (V >= 4) {
            rows::load_quad_any<BaseT>(row, v, V, w[j]);
        } else {
            uint32_t e[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) e[q] = load_raw(row + min(v + q, V - 1));
            if constexpr (sizeof(BaseT) == 2) {
                w[j][0] = (e[0] & 0xffffu) | e[1] << 16;
                w[j][1] = (e[2] & 0xffffu) | e[3] << 16;
            } else {
#pragma unroll
                for (int q = 0; q < 4; ++q) w[j][q] = e[q];
            }
        }
    }
}

// The wave's best of one group of 16 rows over its resident tiles (register
// tile j: vocabulary tile T0 + wave + 8 j; the LDS tile at `ltile`, vocabulary
// tile T0 + 32 + wave, when lds_tile) as an argmax key, valid in lanes 0 .. 15
// for row `lane` of the group.  The tile is the MFMA's A operand and the rank
// (`rank`: the lane's first octet of row `col`) its B operand, so that lane
// (col, kg) ends with row col and the four consecutive columns 4 kg ..: one quad
// load of base logits per tile, one (score, candidate) pair per lane and two
// exchanges across lanes.  (The other way round a lane holds four rows of one
// column: twenty 2-byte loads, four pairs and sixteen exchanges.)  K step
// outermost: each rank operand is read from LDS once and feeds every tile; no
// branches between the MFMAs: a tile that is not the wave's is not combined.
// A row whose best score is -inf names its first column at that score.
template <int KS, typename BaseT, typename PriorT, bool VEC>
__device__ __forceinline__ unsigned long long rr_tiles_best(const bf16x8 (&bt)[kRrRegTiles][KS], const char* ltile,
                                                            bool lds_tile, const uint16_t* rank,
                                                            RrBase<BaseT>& braw, const float* s_prior,
                                                            int T0, int ntl, int wave, int kg, int V, float al,
                                                            float be) {
#pragma clang fp contract(off)
    const int lane = threadIdx.x & 63;
    f32x4 acc[kRrRegTiles + 1];
#pragma unroll
    for (int j = 0; j <= kRrRegTiles; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < KS; ++k) {
        const bf16x8 rk = *reinterpret_cast<const bf16x8*>(rank + k * 32);
        const bf16x8 bv = *reinterpret_cast<const bf16x8*>(ltile + k * 1024 + lane * 16);
#pragma unroll
        for (int j = 0; j < kRrRegTiles; ++j)
            acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bt[j][k], rk, acc[j], 0, 0, 0);
        acc[kRrRegTiles] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bv, rk, acc[kRrRegTiles], 0, 0, 0);
    }
    asm volatile("" ::: "memory");   // the prior is read now: held from before the contraction it costs spills
    // Scores in place of the sums.  A column that is not there scores NaN (through
    // its alpha), which neither the maximum nor the comparison takes; beta 0 reads
    // the zeros behind the prior, and fma(-0, 0, s) is s.
    const float nan = __builtin_nanf("");
    float best = -__builtin_inff();
#pragma unroll
    for (int j = 0; j <= kRrRegTiles; ++j) {
        const int ti = wave + 8 * j;
        const bool live = j < kRrRegTiles ? ti < ntl : lds_tile;   // wave-uniform
        const int tc = min(ti, max(ntl - 1, 0));
        const int left = live ? V - (T0 + tc) * 16 - 4 * kg : 0;   // columns from the lane's first one on
        if constexpr (!VEC)
            if ((T0 + tc) * 16 + 16 > V) rows::shift_quad<BaseT>(braw[j], (T0 + tc) * 16 + 4 * kg, V);   // wave-uniform
        f32x4 pv = {0.f, 0.f, 0.f, 0.f};
        if constexpr (!is_no_prior<PriorT>::value)
            pv = *reinterpret_cast<const f32x4*>(s_prior + (be != 0.f ? tc * 16 : kRrPriorZeros) + 4 * kg);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float al_q = (VEC ? 0 : q) < left ? al : nan;
            float sc = __builtin_fmaf(acc[j][q], al_q, rows::quad_at<BaseT>(braw[j], q));
            if constexpr (!is_no_prior<PriorT>::value) sc = __builtin_fmaf(-be, pv[q], sc);
            acc[j][q] = sc;
            best = __builtin_fmaxf(best, sc);
        }
    }
    // the lowest of the lane's columns at its maximum, which grow with 4 j + q
    int cand = -1;
#pragma unroll
    for (int c = 4 * kRrRegTiles + 3; c >= 0; --c) cand = acc[c >> 2][c & 3] == best ? c : cand;
    // candidate 4 j + q is column (T0 + wave + 8 j) * 16 + 4 kg + q; none (every score NaN): INT_MAX
    const int idx = cand < 0 ? INT_MAX : (T0 + wave + 8 * (cand >> 2)) * 16 + 4 * kg + (cand & 3);
    unsigned long long key = pack_argmax(best, (uint32_t)idx);
#pragma unroll
    for (int off = 16; off < 64; off <<= 1) {
        const unsigned long long o = __shfl_xor(key, off, 64);
        key = o > key ? o : key;
    }
    return key;
}

// Whether quads of base logits can be loaded as one.
inline bool rr_vec(const void* base, int base_dtype, int64_t ld_base, int64_t V) {
    const uintptr_t align = base_dtype == 0 ? 15 : 7;
    return V % 4 == 0 && ld_base % 4 == 0 && (reinterpret_cast<uintptr_t>(base) & align) == 0;
}

}  // namespace dels
