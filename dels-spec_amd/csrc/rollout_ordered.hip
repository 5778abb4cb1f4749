// The stand-in of a rollout that needs its whole grid resident at once.
//
// Enqueued right after such a launch (markov_resident_kernel, or
// rollout_resident_kernel with two groups of rows) on the same stream.  When
// that launch finished its rollout (the word it leaves is zero) every workgroup
// here returns at once: a launch of about 3.9 us.  When it could not get all the
// CUs it needs -- other streams or processes hold some of them for longer than
// the arrivals are waited for -- this launch does the whole rollout with no such
// need: the work is cut into tasks, taken by ticket in order.  A step is, for a GRU local head, a phase of tasks of 16
// GRU units and one of 16 rank columns (each for 16 rows), and then
// kOrdChunks argmax tasks over chunks of the vocabulary; a task waits for every
// task of the phase before its own.  Those have lower tickets, so they are held
// by workgroups that are already running and themselves only wait for lower
// tickets: every wait ends, however few workgroups run at a time.  All the same
// each is bounded (a control area that was not clean could leave a count short
// for ever): one that runs out reports it in the error word, the workgroups stop
// taking tasks, and the last one writes ids of -1 and leaves the control area
// clean.  Correctness is the point, not speed: B streams through the caches every
// step (as in the per-step launches), and what another workgroup wrote is read
// with device-scope loads.  14 steps at V = 151936, r = 256 take 514 us for 4 rows
// of a Markov rollout and 1012 for 24, 1237 for 24 of a DeLS rollout (the one
// launch: 102, 151 and 251).  Sums run in the resident kernels' order, so the
// results are theirs bit for bit.
#include "rollout_resident.h"

namespace dels {

namespace {

constexpr int kOrdChunks = 128;   // argmax tasks per step, and workgroups

struct OrderedArgs {
    const uint16_t* embedding; int64_t ld_embedding;          // Markov: the rank is a row of this table
    const uint16_t* w_hh; const uint16_t* b_hh;               // GRU: [3G, G] MFMA-16 blocks, [3G] or null
    const uint16_t* A; const uint16_t* rank_b; int act;       // [r, G] MFMA-16 blocks, [r] or null
    const uint16_t* gi_table; int64_t ld_gi; int G;
    uint16_t* h[2]; uint16_t* rank;                           // [M, G] twice (by step parity), [M, r]
    int64_t table_rows;                                       // of the embedding or the input table
    const uint16_t* B;
    const void* base; int64_t ld_base;
    const void* prior;
    const float* alpha; const float* beta;
    const int64_t* first_ids; int64_t ld_first;
    int M, V, steps, ntiles;
    int64_t* out_ids; float* out_scores; int64_t ld_out;
    unsigned int* counters;
    unsigned long long* keys;                                 // [steps][32]
    int wait_limit;                                           // looks at a phase's count before giving up
};

// Table row of row m's token at step s: given for step 0, else the index in its key of step s - 1.
__device__ __forceinline__ int64_t ordered_token(const OrderedArgs& a, int s, int m) {
    int64_t t;
    if (s == 0) {
        t = a.first_ids[(int64_t)m * a.ld_first];
    } else {
        const unsigned long long k = atomic_load_u64(a.keys + (s - 1) * 32 + m);
        const uint32_t idx = ~(uint32_t)k;
        t = k == 0ull || idx >= (uint32_t)a.V ? 0 : (int64_t)idx;
    }
    return t < 0 ? 0 : (t >= a.table_rows ? a.table_rows - 1 : t);
}

// Eight bf16 that another workgroup of this launch may have written.
__device__ __forceinline__ bf16x8 coherent_bf16x8(const uint16_t* p) {
    unsigned long long* q = reinterpret_cast<unsigned long long*>(const_cast<uint16_t*>(p));
    const unsigned long long x = atomic_load_u64(q), y = atomic_load_u64(q + 1);
    return __builtin_bit_cast(bf16x8, u32x4{(uint32_t)x, (uint32_t)(x >> 32), (uint32_t)y, (uint32_t)(y >> 32)});
}

// Sum of element e of the eight waves' 256-element accumulators in s_red, in wave order.
__device__ __forceinline__ float ordered_sum(const float* s_red, int e) {
    float v = s_red[e];
#pragma unroll
    for (int ww = 1; ww < kRrWaves; ++ww) v = v + s_red[ww * 256 + e];
    return v;
}

// 16 GRU units from u0 for rows m0 .. m0 + 15: h(s) = GRU(gi_table[token], h(s - 1)).
__device__ __forceinline__ void ordered_gru(const OrderedArgs& a, int s, int m0, int u0, float* s_red) {
#pragma clang fp contract(off)
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int KB = a.G / 32;
    const uint16_t* hp = a.h[(s + 1) & 1];
    f32x4 acc[3];
#pragma unroll
    for (int g = 0; g < 3; ++g) acc[g] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (s > 0) {
        const int m = min(m0 + (lane & 15), a.M - 1);
        for (int kb = wave; kb < KB; kb += kRrWaves) {
            const bf16x8 hv = coherent_bf16x8(hp + (int64_t)m * a.G + kb * 32 + (lane >> 4) * 8);
#pragma unroll
            for (int g = 0; g < 3; ++g)
                acc[g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                    hv, load_bf16x8(a.w_hh + ((int64_t)((g * a.G + u0) >> 4) * KB + kb) * 512 + lane * 8), acc[g], 0, 0, 0);
        }
    }
    float gh[3] = {0.f, 0.f, 0.f};
    const int mi = threadIdx.x >> 4, j = threadIdx.x & 15;       // this thread's row and unit (first 256 threads)
    const int e = (((mi >> 2) * 16 + j) << 2) + (mi & 3);
#pragma unroll
    for (int g = 0; g < 3; ++g) {
        __syncthreads();
        *reinterpret_cast<f32x4*>(&s_red[wave * 256 + lane * 4]) = acc[g];
        __syncthreads();
        if (threadIdx.x < 256) {
            float v = ordered_sum(s_red, e);
            if (a.b_hh) v = v + bf16_bits_to_f32(a.b_hh[g * a.G + u0 + j]);
            gh[g] = round_bf16(v);
        }
    }
    const int m = m0 + mi, u = u0 + j;
    uint32_t bits = 0;
    const bool live = threadIdx.x < 256 && m < a.M;
    if (live) {
        const uint16_t* gi = a.gi_table + ordered_token(a, s, m) * a.ld_gi + u;
        float hv = 0.f;
        if (s > 0) {   // the pair of units that holds this one
            const uint32_t pair = __hip_atomic_load(
                reinterpret_cast<uint32_t*>(const_cast<uint16_t*>(hp) + (int64_t)m * a.G + (u & ~1)), __ATOMIC_RELAXED,
                __HIP_MEMORY_SCOPE_AGENT);
            hv = bf16_bits_to_f32((u & 1) ? pair >> 16 : pair & 0xffffu);
        }
        bits = f32_to_bf16_bits(gru_unit(bf16_bits_to_f32(gi[0]), bf16_bits_to_f32(gi[a.G]),
                                         bf16_bits_to_f32(gi[2 * a.G]), gh[0], gh[1], gh[2], hv));
    }
    const uint32_t other = (uint32_t)__shfl_down((int)bits, 1, 64);
    if (live && (j & 1) == 0)
        atomic_store_u32(reinterpret_cast<unsigned int*>(a.h[s & 1] + (int64_t)m * a.G + u), bits | (other << 16));
}

// 16 rank columns from n0 for rows m0 .. m0 + 15.
__device__ __forceinline__ void ordered_rank(const OrderedArgs& a, int s, int m0, int n0, float* s_red) {
#pragma clang fp contract(off)
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int KB = a.G / 32;
    const uint16_t* h = a.h[s & 1];
    const int mr = min(m0 + (lane & 15), a.M - 1);
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int kb = wave; kb < KB; kb += kRrWaves)
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            coherent_bf16x8(h + (int64_t)mr * a.G + kb * 32 + (lane >> 4) * 8),
            load_bf16x8(a.A + ((int64_t)(n0 >> 4) * KB + kb) * 512 + lane * 8), acc, 0, 0, 0);
    *reinterpret_cast<f32x4*>(&s_red[wave * 256 + lane * 4]) = acc;
    __syncthreads();
    const int mi = threadIdx.x >> 4, j = threadIdx.x & 15;
    uint32_t bits = 0;
    const bool live = threadIdx.x < 256 && m0 + mi < a.M;
    if (live) {
        float v = ordered_sum(s_red, (((mi >> 2) * 16 + j) << 2) + (mi & 3));
        if (a.rank_b) v = v + bf16_bits_to_f32(a.rank_b[n0 + j]);
        v = round_bf16(v);
        if (a.act == 1) v = round_bf16(silu_f32(v));
        bits = f32_to_bf16_bits(v);
    }
    const uint32_t other = (uint32_t)__shfl_down((int)bits, 1, 64);
    if (live && (j & 1) == 0)
        atomic_store_u32(reinterpret_cast<unsigned int*>(a.rank + (int64_t)(m0 + mi) * kResidentRank + n0 + j),
                         bits | (other << 16));
}

// The argmax of every row over vocabulary chunk c, into the step's keys.
template <bool GRU, int KS, typename BaseT, typename PriorT>
__device__ __forceinline__ void ordered_argmax(const OrderedArgs& a, int s, int c,
                                               unsigned long long (&s_key)[kRrWaves][32]) {
#pragma clang fp contract(off)
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane & 15, kg = lane >> 4;
    const int t0 = (int)(((int64_t)c * a.ntiles) / kOrdChunks), t1 = (int)(((int64_t)(c + 1) * a.ntiles) / kOrdChunks);
    const float al = a.alpha[s], be = a.beta[s];
    const bool use_prior = !is_no_prior<PriorT>::value && be != 0.f;
    for (int m0 = 0; m0 < a.M; m0 += 16) {
        bf16x8 ra[KS];
        const int mr = min(m0 + col, a.M - 1);
        if constexpr (GRU) {
#pragma unroll
            for (int k = 0; k < KS; ++k) ra[k] = coherent_bf16x8(a.rank + (int64_t)mr * (KS * 32) + k * 32 + kg * 8);
        } else {
            const uint16_t* rp = a.embedding + ordered_token(a, s, mr) * a.ld_embedding + kg * 8;
#pragma unroll
            for (int k = 0; k < KS; ++k) ra[k] = load_bf16x8(rp + k * 32);
        }
        float best[4];
        int bidx[4];
        const BaseT* brow[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            best[q] = -__builtin_inff();
            bidx[q] = INT_MAX;
            brow[q] = static_cast<const BaseT*>(a.base) + (int64_t)min(m0 + 4 * kg + q, a.M - 1) * a.ld_base +
                      (int64_t)s * a.V;
        }
        for (int t = t0 + wave; t < t1; t += kRrWaves) {
            f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int k = 0; k < KS; ++k)
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                    ra[k], load_bf16x8_nt(a.B + ((int64_t)t * KS + k) * 512 + lane * 8), acc, 0, 0, 0);
            const int v = t * 16 + col, vc = min(v, a.V - 1);
            float pv = 0.f;
            if constexpr (!is_no_prior<PriorT>::value) pv = load_f32(static_cast<const PriorT*>(a.prior) + vc);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                float sc = __builtin_fmaf(acc[q], al, load_f32(brow[q] + vc));
                if (use_prior) sc = __builtin_fmaf(-be, pv, sc);
                const bool take = (v < a.V) & argmax_better(sc, v, best[q], bidx[q]);
                best[q] = take ? sc : best[q];
                bidx[q] = take ? v : bidx[q];
            }
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            // a lane without a candidate: key 0, below every real one
            unsigned long long key = bidx[q] == INT_MAX ? 0ull : pack_argmax(best[q], (uint32_t)bidx[q]);
            rr_row_max<1>(key);
            rr_row_max<2>(key);
            rr_row_max<4>(key);
            rr_row_max<8>(key);
            if (col == 15) s_key[wave][m0 + 4 * kg + q] = key;
        }
    }
    __syncthreads();
    unsigned long long seen = 0;
    if ((int)threadIdx.x < a.M) {
        unsigned long long k = s_key[0][threadIdx.x];
#pragma unroll
        for (int ww = 1; ww < kRrWaves; ++ww) k = max(k, s_key[ww][threadIdx.x]);
        if (k != 0ull)
            seen = __hip_atomic_fetch_max(a.keys + s * 32 + threadIdx.x, k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    asm volatile("" ::"v"(seen));   // the maxima have returned
}

// Wait until a phase's count of finished tasks reaches `want`.  False when it did
// not within wait_limit looks, or another workgroup gave up.
__device__ __forceinline__ bool ordered_wait(const OrderedArgs& a, const unsigned int* count, unsigned want) {
    for (int it = 0; it < a.wait_limit; ++it) {
        if (__hip_atomic_load(count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= want) return true;
        if ((it & 63) == 63 && rr_failed(a)) return false;
        __builtin_amdgcn_s_sleep(8);
    }
    return false;
}

template <bool GRU, int KS, typename BaseT, typename PriorT>
__global__ __launch_bounds__(kRrThreads) void rollout_ordered_kernel(OrderedArgs a) {
    __shared__ unsigned long long s_key[kRrWaves][32];
    __shared__ __attribute__((aligned(16))) float s_red[GRU ? kRrWaves * 256 : 4];
    __shared__ unsigned int s_task;
    if (__hip_atomic_load(a.counters + kRrNotDoneWord, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0u) return;

    // tasks of each phase of a step, and of the step
    const unsigned groups = (a.M + 15) / 16;
    const unsigned n0 = GRU ? groups * (a.G / 16) : 0, n1 = GRU ? groups * (KS * 2) : 0, per = n0 + n1 + kOrdChunks;
    const unsigned total = (unsigned)a.steps * per;
    unsigned int* done = a.counters;   // [steps][3]: finished tasks of each phase
    for (;;) {
        __syncthreads();   // the LDS of the task before has been read
        if (threadIdx.x == 0) {
            unsigned t = __hip_atomic_fetch_add(a.counters + kRrTicketWord, 1u, __ATOMIC_RELAXED,
                                                __HIP_MEMORY_SCOPE_AGENT);
            if (t < total) {
                // the phase before this task's: its counter and how many tasks it has
                const unsigned s = t / per, i = t % per;
                const unsigned ph = i < n0 ? 0 : i < n0 + n1 ? 1 : 2;
                unsigned int* before = nullptr;
                unsigned want = 0;
                if (GRU && ph > 0) { before = done + s * 3 + ph - 1; want = ph == 1 ? n0 : n1; }
                else if (s > 0) { before = done + (s - 1) * 3 + 2; want = kOrdChunks; }
                if (before && !ordered_wait(a, before, want)) {
                    rr_fail(a);
                    t = total;
                }
            }
            s_task = t;
        }
        __syncthreads();
        const unsigned task = s_task;
        if (task >= total) break;
        const int s = (int)(task / per);
        const unsigned i = task % per;
        int ph = 2;
        if (GRU && i < n0) {
            ph = 0;
            ordered_gru(a, s, 16 * (int)(i % groups), 16 * (int)(i / groups), s_red);
        } else if (GRU && i < n0 + n1) {
            ph = 1;
            ordered_rank(a, s, 16 * (int)((i - n0) % groups), 16 * (int)((i - n0) / groups), s_red);
        } else {
            ordered_argmax<GRU, KS, BaseT, PriorT>(a, s, (int)(i - n0 - n1), s_key);
        }
        __builtin_amdgcn_s_waitcnt(0);     // every wave's stores have reached device coherence ...
        __syncthreads();
        if (threadIdx.x == 0)              // ... before the task counts as done
            __hip_atomic_fetch_add(done + s * 3 + ph, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    // the last workgroup to run out of tasks decodes the keys and leaves the control area clean
    if (threadIdx.x == 0) {
        __builtin_amdgcn_s_waitcnt(0);   // a failure is stored before this workgroup counts as out of tasks
        s_task = __hip_atomic_fetch_add(a.counters + kRrExitCounter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (s_task != gridDim.x - 1) return;
    const bool failed = rr_failed(a);
    __syncthreads();   // every thread has read the error word before it is cleared
    for (int i = threadIdx.x; i < a.steps * 32; i += kRrThreads) {
        const int s = i >> 5, m = i & 31;
        const unsigned long long k = __hip_atomic_exchange(a.keys + i, 0ull, __ATOMIC_RELAXED,
                                                           __HIP_MEMORY_SCOPE_AGENT);
        if (m >= a.M) continue;
        int64_t id = (int64_t)(uint32_t)~(uint32_t)k;
        float val = f32_from_order_key((uint32_t)(k >> 32));
        if (failed || k == 0ull || id >= a.V) {    // not produced, or no candidate at all
            id = failed ? -1 : 0;
            val = -__builtin_inff();
        }
        a.out_ids[(int64_t)m * a.ld_out + s] = id;
        if (a.out_scores) a.out_scores[(int64_t)m * a.ld_out + s] = val;
    }
    for (int i = threadIdx.x; i < a.steps * 3; i += kRrThreads)
        __hip_atomic_store(done + i, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (threadIdx.x < 4) {
        const int word = threadIdx.x == 0   ? kRrNotDoneWord
                         : threadIdx.x == 1 ? kRrTicketWord
                         : threadIdx.x == 2 ? kRrExitCounter
                                            : kRrErrorWord;
        __hip_atomic_store(a.counters + word, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

template <bool GRU, int KS, typename BaseT>
hipError_t launch_ordered(const OrderedArgs& a, int prior_kind, hipStream_t s) {
    const dim3 grid(kOrdChunks), block(kRrThreads);
    switch (prior_kind) {
        case 0: hipLaunchKernelGGL((rollout_ordered_kernel<GRU, KS, BaseT, no_prior_t>), grid, block, 0, s, a); break;
        case 1: hipLaunchKernelGGL((rollout_ordered_kernel<GRU, KS, BaseT, float>), grid, block, 0, s, a); break;
        case 2: hipLaunchKernelGGL((rollout_ordered_kernel<GRU, KS, BaseT, bf16_t>), grid, block, 0, s, a); break;
        default: hipLaunchKernelGGL((rollout_ordered_kernel<GRU, KS, BaseT, f16_t>), grid, block, 0, s, a); break;
    }
    return hipGetLastError();
}

template <bool GRU, int KS>
hipError_t launch_ordered_base(const OrderedArgs& a, const void* prior, int prior_dtype, int base_dtype, hipStream_t s) {
    const int pk = prior == nullptr ? 0 : (prior_dtype == 1 ? 2 : (prior_dtype == 2 ? 3 : 1));
    if (base_dtype == 1) return launch_ordered<GRU, KS, bf16_t>(a, pk, s);
    if (base_dtype == 2) return launch_ordered<GRU, KS, f16_t>(a, pk, s);
    return launch_ordered<GRU, KS, float>(a, pk, s);
}

constexpr int kOrdWaitLimit = 1 << 22;   // looks (about 1 us each) before a wait gives up
int g_ordered_wait_limit = kOrdWaitLimit;

}  // namespace

void set_ordered_wait_limit(int limit) { g_ordered_wait_limit = limit < 0 ? kOrdWaitLimit : limit; }

hipError_t launch_markov_ordered(const MarkovRolloutArgs& r, hipStream_t s) {
    OrderedArgs a{};
    a.embedding = r.embedding; a.ld_embedding = r.ld_embedding; a.table_rows = r.table_rows;
    a.B = r.B;
    a.base = r.base; a.ld_base = r.ld_base;
    a.prior = r.prior;
    a.alpha = r.alpha; a.beta = r.beta;
    a.first_ids = r.prev_ids; a.ld_first = r.ld_prev;
    a.M = r.M; a.V = r.V; a.steps = r.steps; a.ntiles = r.ntiles;
    a.out_ids = r.out_ids; a.out_scores = r.out_scores; a.ld_out = r.ld_out;
    a.counters = r.counters;
    a.keys = r.keys;
    a.wait_limit = g_ordered_wait_limit;
    if (r.r == 256) return launch_ordered_base<false, 8>(a, r.prior, r.prior_dtype, r.base_dtype, s);
    return launch_ordered_base<false, 4>(a, r.prior, r.prior_dtype, r.base_dtype, s);
}

hipError_t launch_rollout_ordered(const ResidentRolloutArgs& r, void* ws, hipStream_t s) {
    char* w = static_cast<char*>(ws);
    OrderedArgs a{};
    a.w_hh = r.w_hh; a.b_hh = r.b_hh;
    a.A = r.A; a.rank_b = r.rank_b; a.act = r.act;
    a.gi_table = r.gi_table; a.ld_gi = r.ld_gi; a.table_rows = r.table_rows; a.G = (int)r.G;
    a.h[0] = r.h_a; a.h[1] = r.h_b; a.rank = r.rank;
    a.B = r.B;
    a.base = r.base; a.ld_base = r.ld_base;
    a.prior = r.prior;
    a.alpha = r.alpha; a.beta = r.beta;
    a.first_ids = r.prefix; a.ld_first = r.ld_prefix;
    a.M = (int)r.batch; a.V = (int)r.V; a.steps = (int)r.steps; a.ntiles = (int)((r.V + 15) / 16);
    a.out_ids = r.out_ids; a.out_scores = r.out_scores; a.ld_out = r.ld_out;
    a.counters = reinterpret_cast<unsigned int*>(w + kCountersOff);
    a.keys = reinterpret_cast<unsigned long long*>(w + kKeysOff);
    a.wait_limit = g_ordered_wait_limit;
    return launch_ordered_base<true, kResidentRank / 32>(a, r.prior, r.prior_dtype, r.base_dtype, s);
}

}  // namespace dels
