// The Markov rollout as one launch with the low-rank head's B resident on chip.
//
// The rollout (code/kernel/markov_dels.py:261-278: token_0 = the previous ids;
// each step the rank rows are the embedding rows of the current tokens, then
// the fused combine + argmax picks the next ones) reads the same B [V, r]
// every step.  Per-step launches stream it from HBM each time (77.8 MB at
// V = 151936, r = 256: 18.6 us a step, of which 13 are the stream and the rest
// launch, hand-off and drain).  Here, as in rollout_resident.hip, one workgroup
// per CU keeps its share of B for the whole rollout -- 4 vocabulary tiles of 16
// rows per wave in VGPRs, up to 6 more per workgroup in LDS -- so a step moves
// its base logits, the rank rows and one slot word per row and workgroup.
// What bounds a step is the chain: publish the slot words, read everyone's,
// gather the embedding rows they name, contract, publish.  14 steps of 4 rows at
// V = 151936, r = 256, with the copies of a runner's call: 279.6 -> 107.9 us.
//
//   * argmax: every wave contracts its resident tiles against the rank of up
//     to two groups of 16 rows and combines s = fma(-beta, prior, fma(dot,
//     alpha, base)) as every kernel of the path does (rr_tiles_best), and the
//     workgroup publishes each row's best as one slot word (rr_slot_maxima);
//   * every workgroup reads all slots of each row, takes the maximum, and so
//     knows the step's ids, whose embedding rows it loads into LDS.
//
// Slot words carry the step's low bits only, so a launch clears its own slots
// (returning exchanges) before it publishes an arrival word with the launch's
// tag; every workgroup waits for all arrival words (while its tiles of B load)
// before it publishes a slot.  The wait for the arrivals doubles as the test
// that the grid is resident as a whole, which it needs one CU per workgroup
// for: it is short, and when it -- or any later wait, all of them bounded --
// runs out, the launch ends without a result and marks the rollout as not done;
// the launch that follows it on the stream (rollout_ordered.hip, which needs no
// co-residency and otherwise returns at once) then does the whole rollout.
#include "rollout_resident.h"

namespace dels {

namespace {

constexpr int kMrPad = 8;   // bf16 of padding per rank row in LDS (rows 16 B apart in banks)

template <int RG, int KS, typename BaseT, typename PriorT, bool VEC>
__global__ __launch_bounds__(kRrThreads) void markov_resident_kernel(MarkovRolloutArgs a) {
#pragma clang fp contract(off)
    constexpr int kRows = 16 * RG;
    constexpr int kPitch = KS * 32 + kMrPad;
    __shared__ __attribute__((aligned(16))) char s_b[kResidentLdsTiles * KS * 1024];
    __shared__ __attribute__((aligned(16))) uint16_t s_rank[kRows * kPitch];
    __shared__ __attribute__((aligned(16))) float s_prior[kRrPriorWords];
    __shared__ unsigned long long s_key[kRrWaves][kRows];   // each wave's best key of each row
    __shared__ unsigned long long s_rowmax[kRows];          // the step's maximum slot word of each row
    __shared__ float s_ab[2][kResidentMaxSteps];
    __shared__ int64_t s_ids[kRows];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane & 15, kg = lane >> 4;
    const int w = blockIdx.x, nwg = gridDim.x;
    const int M = a.M, V = a.V;
    const uint32_t gen = __hip_atomic_load(a.counters + kDecodeGenWord, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const uint32_t tag = rr_tag(gen, 0);
    const BaseT* base = static_cast<const BaseT*>(a.base);

    // this workgroup's slots of both parity sets and every row group back to
    // zero; their old values have returned before the barrier, so the clearing
    // is done before the arrival word goes out
    if (threadIdx.x < 4 * 16) {
        const int set = threadIdx.x >> 4, m = threadIdx.x & 15;
        const unsigned long long old = __hip_atomic_exchange(a.slots + set * kRrSlotSet + w * 16 + m, 0ull,
                                                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("" ::"v"(old));
    }
    if (threadIdx.x < kRows) {
        s_rowmax[threadIdx.x] = 0ull;
        s_ids[threadIdx.x] = threadIdx.x < M ? a.prev_ids[(int64_t)threadIdx.x * a.ld_prev] : 0;
    }
    for (int i = threadIdx.x; i < a.steps; i += kRrThreads) {
        s_ab[0][i] = a.alpha[i];
        s_ab[1][i] = a.beta[i];
    }
    __syncthreads();
    if (threadIdx.x == 0)
        __hip_atomic_store(a.words + w * 16, (unsigned long long)tag << 32, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);

    // ---- resident operands: tiles [T0, T0 + ntl), register tile j of this wave
    // T0 + wave + 8 j, LDS tile e (contracted by wave e) T0 + 32 + e
    const int T0 = (int)(((int64_t)w * a.ntiles) / nwg);
    const int ntl = (int)(((int64_t)(w + 1) * a.ntiles) / nwg) - T0;
    const int nlds = max(0, ntl - kRrWaves * kRrRegTiles);
    for (int i = threadIdx.x; i < nlds * KS * 64; i += kRrThreads) {
        const int e = i / (KS * 64), rem = i - e * (KS * 64), s = rem >> 6, l = rem & 63;
        const int t = T0 + kRrWaves * kRrRegTiles + e;
        *reinterpret_cast<u32x4*>(s_b + (e * KS + s) * 1024 + l * 16) =
            *reinterpret_cast<const u32x4*>(a.B + ((int64_t)t * KS + s) * 512 + l * 8);
    }
    if (threadIdx.x < 16) s_prior[kRrPriorZeros + threadIdx.x] = 0.f;
    for (int i = threadIdx.x; i < ntl * 16; i += kRrThreads) {
        const int v = min(T0 * 16 + i, V - 1);
        if constexpr (is_no_prior<PriorT>::value) s_prior[i] = 0.f;
        else s_prior[i] = widen_raw<PriorT>(load_raw(static_cast<const PriorT*>(a.prior) + v));
    }
    asm volatile("" ::: "memory");   // the register tiles after the LDS operands (whose stores wait for their loads)
    bf16x8 bt[kRrRegTiles][KS];
#pragma unroll
    for (int j = 0; j < kRrRegTiles; ++j) {
        // a tile that is not this wave's loads the last tile (in bounds) and is not combined
        const int t = min(T0 + wave + 8 * j, a.ntiles - 1);
#pragma unroll
        for (int s = 0; s < KS; ++s) bt[j][s] = load_bf16x8_nt(a.B + ((int64_t)t * KS + s) * 512 + lane * 8);
    }

    // every workgroup is here: one word each, a line per workgroup
    bool ok;
    {
        MarkovRolloutArgs first = a;
        first.spin_limit = min(a.spin_limit, a.arrival_limit);
        const RrWords pl{nwg, 0, 4, 0, 0, 1};
        int tid = threadIdx.x;
        unsigned long long word[1];
        const bool got = rr_gather<1>(first, a.words, pl, tid, word,
                                      [&](unsigned long long x) { return (uint32_t)(x >> 32) == tag; });
        ok = !__syncthreads_or(!got);
    }

    const int mp = a.mp_shift;   // log2 of the first group's rows rounded up
    const RrWords s_pl{nwg << mp, mp, 4, 0, mp, min(M, 16)};
    int s = 0;
    for (; ok && s < a.steps; ++s) {
        // lane values pass through an empty asm statement each step, so that the
        // compiler forms the step's addresses here instead of holding them in
        // registers across the loop
        int lcol = col, lkg = kg;
        asm volatile("" : "+v"(lcol), "+v"(lkg));
        // the rank rows first (the step waits for them), then the base logits
        constexpr int kPieces = KS * 4;                           // 16-byte pieces per rank row
        constexpr int kPer = (kRows * kPieces + kRrThreads - 1) / kRrThreads;
        u32x4 rp[kPer];
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            const int p = min((int)threadIdx.x + kRrThreads * i, M * kPieces - 1);
            const int m = p / kPieces;
            int64_t t = s_ids[m];
            t = t < 0 ? 0 : (t >= a.table_rows ? a.table_rows - 1 : t);
            rp[i] = *reinterpret_cast<const u32x4*>(a.embedding + t * a.ld_embedding + (p - m * kPieces) * 8);
        }
        RrBase<BaseT> braw[RG];
#pragma unroll
        for (int g = 0; g < RG; ++g) {
            const int m = 16 * g + lcol;
            rr_load_base<BaseT, VEC>(base + (int64_t)s * V + (int64_t)(m < M ? m : 0) * a.ld_base, T0, ntl, a.ntiles,
                                     wave, lkg, V, braw[g]);
        }
        asm volatile("" ::: "memory");   // the base loads are issued before the rank rows are waited for
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            const int p = threadIdx.x + kRrThreads * i;
            const int m = p / kPieces;
            if (p < M * kPieces) *reinterpret_cast<u32x4*>(&s_rank[m * kPitch + (p - m * kPieces) * 8]) = rp[i];
        }
        __syncthreads();

        const bool lds_tile = wave < nlds;
        const char* ltile = s_b + (lds_tile ? wave : 0) * KS * 1024;
#pragma unroll
        for (int g = 0; g < RG; ++g) {
            const unsigned long long key = rr_tiles_best<KS, BaseT, PriorT, VEC>(
                bt, ltile, lds_tile, &s_rank[(16 * g + lcol) * kPitch + lkg * 8], braw[g], s_prior, T0, ntl, wave, lkg,
                V, s_ab[0][s], s_ab[1][s]);
            // Sixteen idle cycles.  Without them rollouts of 2 to 4 rows take 1.5 % longer (14
            // steps, V = 151936, r = 256: 94.0 / 94.7 / 96.1 us for 2 / 3 / 4 rows, 93.4 / 93.7 /
            // 95.1 with them; 1, 5, 8 and 16 rows the same): where the code or the polls fall,
            // not what they do, makes the difference.
            asm volatile("s_nop 7\n\ts_nop 7");
            if (kg == 0) s_key[wave][16 * g + col] = key;
        }
        __syncthreads();
        // the workgroup's best of each row into its slot word for the step
        const uint32_t low2 = 1u | ((((uint32_t)s >> 1) & 1u) << 1);
        unsigned long long* slot_set = a.slots + (s & 1) * 2 * kRrSlotSet;
        if ((int)threadIdx.x < M) {
            const int m = threadIdx.x;
            unsigned long long k = s_key[0][m];
#pragma unroll
            for (int ww = 1; ww < kRrWaves; ++ww) k = max(k, s_key[ww][m]);
            // no candidate (index INT_MAX): index 2^30 - 1, past every vocabulary
            const unsigned long long word =
                low2 | (k & 0xffffffff00000000ull) | ((unsigned long long)((uint32_t)k & 0x3fffffffu) << 2);
            __hip_atomic_store(slot_set + (m >> 4) * kRrSlotSet + w * 16 + (m & 15), word, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        }
        if (s + 1 == a.steps && w != 0) break;   // the last ids: workgroup 0 alone writes them
        // ---- the step's ids ------------------------------------------------------------
        // as few loads per thread as cover the words
        if (s_pl.n <= 2 * kRrThreads) ok = rr_slot_maxima<2>(a, slot_set, s_pl, low2, s_rowmax);
        else if (s_pl.n <= 4 * kRrThreads) ok = rr_slot_maxima<4>(a, slot_set, s_pl, low2, s_rowmax);
        else ok = rr_slot_maxima<8>(a, slot_set, s_pl, low2, s_rowmax);
        if constexpr (RG == 2) {
            if (ok) {
                const RrWords pl{nwg << 4, 4, 4, 0, 4, M - 16};
                ok = rr_slot_maxima<8>(a, slot_set + kRrSlotSet, pl, low2, s_rowmax + 16);
            }
        }
        if (!ok) break;
        if ((int)threadIdx.x < M) {
            const int m = threadIdx.x;
            int64_t id = 0;
            float val = -__builtin_inff();
            const unsigned long long key = s_rowmax[m];
            s_rowmax[m] = 0ull;   // for the next step (barriers come between)
            const uint32_t idx = ~(uint32_t)(key >> 2) & 0x3fffffffu;
            if (idx < (uint32_t)V) {
                id = idx;
                val = f32_from_order_key((uint32_t)(key >> 32));
            }
            s_ids[m] = id;
            if (w == 0) {
                a.out_ids[(int64_t)m * a.ld_out + s] = id;
                if (a.out_scores) a.out_scores[(int64_t)m * a.ld_out + s] = val;
            }
        }
        __syncthreads();
    }
    if (!ok && threadIdx.x == 0) rr_fail(a);

    // ---- the last workgroup clears the control area, advances the generation and,
    // after a failure, leaves the word that lets the ordered rollout run
    __syncthreads();
    if (threadIdx.x != 0) return;
    __builtin_amdgcn_s_waitcnt(0);   // a failure is stored before this workgroup counts as done
    const unsigned prev = __hip_atomic_fetch_add(a.counters + kRrDoneCounter, 1u, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT);
    if (prev != (unsigned)nwg - 1) return;
    const unsigned failed = __hip_atomic_exchange(a.counters + kRrErrorWord, 0u, __ATOMIC_RELAXED,
                                                  __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(a.counters + kRrDoneCounter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(a.counters + kRrNotDoneWord, failed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_fetch_add(a.counters + kDecodeGenWord, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <int RG, int KS, typename BaseT, bool VEC>
hipError_t launch_mr(const MarkovRolloutArgs& a, int prior_kind, int nwg, hipStream_t s) {
    const dim3 grid(nwg), block(kRrThreads);
    switch (prior_kind) {
        case 0: hipLaunchKernelGGL((markov_resident_kernel<RG, KS, BaseT, no_prior_t, VEC>), grid, block, 0, s, a); break;
        case 1: hipLaunchKernelGGL((markov_resident_kernel<RG, KS, BaseT, float, VEC>), grid, block, 0, s, a); break;
        case 2: hipLaunchKernelGGL((markov_resident_kernel<RG, KS, BaseT, bf16_t, VEC>), grid, block, 0, s, a); break;
        default: hipLaunchKernelGGL((markov_resident_kernel<RG, KS, BaseT, f16_t, VEC>), grid, block, 0, s, a); break;
    }
    return hipGetLastError();
}

template <typename BaseT>
hipError_t launch_mr_base(const MarkovRolloutArgs& a, int prior_kind, int nwg, hipStream_t s) {
    auto by_shape = [&](auto vec) -> hipError_t {
        constexpr bool VEC = decltype(vec)::value;
        if (a.r == 256)
            return a.M <= 16 ? launch_mr<1, 8, BaseT, VEC>(a, prior_kind, nwg, s)
                             : launch_mr<2, 8, BaseT, VEC>(a, prior_kind, nwg, s);
        return a.M <= 16 ? launch_mr<1, 4, BaseT, VEC>(a, prior_kind, nwg, s)
                         : launch_mr<2, 4, BaseT, VEC>(a, prior_kind, nwg, s);
    };
    return rr_vec(a.base, a.base_dtype, a.ld_base, a.V) ? by_shape(std::true_type{}) : by_shape(std::false_type{});
}

}  // namespace

bool markov_resident_eligible(int64_t batch, int64_t r, int64_t V, int64_t steps, bool packed,
                              size_t ws_bytes) {
    const int nwg = device_cu_count();
    if (!packed || ws_bytes < kDataOff + kMarkovSlotBytes || batch < 1 || batch > 32) return false;
    if (!(r == 128 || r == 256)) return false;
    if (steps < 2 || steps > kResidentMaxSteps) return false;
    if (nwg < 64 || nwg > kResidentMaxWGs || nwg % 64 != 0) return false;
    const int64_t ntiles = (V + 15) / 16;
    return (ntiles + nwg - 1) / nwg <= kRrWaves * kRrRegTiles + kResidentLdsTiles;
}

// One launch takes 13 to 21 us before its first step (B on chip, everyone's
// arrival, the stand-in behind it) and about 5 a step (two groups of rows 8), the
// per-step launches 6 and as much a step as the vocabulary asks: at V = 2000 /
// 8192 / 16384 / 32000 / 65536 / 151936, r = 256, 16 rows 6.4 / 7.7 / 10.2 / 10.6
// / 13.1 / 18.5, 32 rows 7.0 / 7.3 / 8.5 / 10.8 / 13.6 / 18.5.  The steps from
// which one launch is ahead (r = 128 differs little); below the last line it never
// was in 24 steps of two groups.
bool markov_resident_pays(int64_t batch, int64_t V, int64_t steps) {
    if (batch <= 16) return steps >= (V >= 65536 ? 2 : V >= 32768 ? 3 : V >= 16384 ? 4 : V >= 8192 ? 8 : 16);
    return V >= 30720 && steps >= (V >= 98304 ? 3 : V >= 65536 ? 4 : 8);
}

hipError_t launch_markov_resident(MarkovRolloutArgs a, void* ws, hipStream_t s) {
    char* w = static_cast<char*>(ws);
    a.ntiles = (a.V + 15) / 16;
    a.mp_shift = 0;
    while ((1 << a.mp_shift) < std::min(a.M, 16)) ++a.mp_shift;
    a.counters = reinterpret_cast<unsigned int*>(w + kCountersOff);
    a.keys = reinterpret_cast<unsigned long long*>(w + kKeysOff);
    a.words = reinterpret_cast<unsigned long long*>(w + kResidentOff);
    a.slots = reinterpret_cast<unsigned long long*>(w + kDataOff);
    a.spin_limit = resident_spin_limit();
    a.arrival_limit = kRrArrivalLimit;
    const int nwg = device_cu_count();
    const int pk = a.prior == nullptr ? 0 : (a.prior_dtype == 1 ? 2 : (a.prior_dtype == 2 ? 3 : 1));
    hipError_t e;
    if (a.base_dtype == 1) e = launch_mr_base<bf16_t>(a, pk, nwg, s);
    else if (a.base_dtype == 2) e = launch_mr_base<f16_t>(a, pk, nwg, s);
    else e = launch_mr_base<float>(a, pk, nwg, s);
    if (e != hipSuccess) return e;
    return launch_markov_ordered(a, s);
}

}  // namespace dels
