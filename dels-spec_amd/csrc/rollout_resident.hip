// The DeLS rollout as one launch with the low-rank head's B resident on chip.
//
// The rollout (code/kernel/dels.py:425-467: prefix GRU, then per step rank
// projection -> fused combine + argmax -> GRU on the chosen id, none after the
// last step) reads the same B [V, r] every step; per-step launches stream it
// from HBM each time (77.8 MB at V = 151936, r = 256: ~11 us of every ~24 us
// step).  Here one workgroup per CU holds its share of B for the whole
// rollout -- 4 vocabulary tiles of 16 rows per wave in VGPRs (the MFMA
// operand of every K step, 128 registers), up to 6 more per workgroup in LDS
// -- so a step moves only its base rows and a few tagged words:
//   * GRU: every workgroup owns G / nwg units (4 at G = 1024 on 256 CUs) and
//     keeps their W_hh rows in LDS as one 16-row MFMA operand per K step
//     (3 gates x units <= 16 rows); gh = h . W_hh^T + b_hh is summed per wave
//     over its K steps, then over the eight waves in a fixed order, rounded to
//     bf16 after the bias (as F.linear in bf16), and the gates combine with
//     the gathered input-table row (gru_unit);
//   * the new state goes out as words {tag, two bf16} (an agent-scope store
//     per word); every workgroup reads all of them into LDS (bounded
//     re-reads of words whose tag is not this step's);
//   * rank: workgroups 0 .. r/16 - 1 each own one 16-column tile of the rank
//     and keep its 16 rows of A in LDS; rank = bf16(act(bf16(h . A^T + b)))
//     goes out as words {tag, two bf16}, read by every workgroup;
//   * argmax: every wave contracts its resident tiles against the rank and
//     combines s = fma(-beta, prior, fma(dot, alpha, base)) as every kernel of
//     the path does (rr_tiles_best: 2.2 us of an 11.1 us step with a running
//     (score, index) pair for each of a lane's four rows, 1.65 here; 8 rows); the
//     workgroup publishes each row's best as one slot word (order(score) in the
//     high half, ~index above two flag bits in the low half, so the
//     larger word is the argmax with ties to the lower index) and every
//     workgroup reads all nwg slots of each row, takes the maximum and so
//     knows the step's ids for its GRU units.  Each workgroup owns its slots
//     (no two workgroups write one address: no atomics queue on a hot word).
// Pacing the exchanges: every read issues all its loads before it examines
// any (a value consumed as soon as it is loaded would cost one memory round
// trip per word instead of one per read).
// The tag of a state or rank word is a function of the launch generation and
// the step, and the words live in a workspace region no other kernel writes,
// so a word of an earlier step or launch never passes.  Slot words alternate
// between two sets by step parity and carry bit 1 of the step; a launch first
// clears its own slots (returning exchanges, complete before the workgroup
// publishes its first state words, which every reader waits for), so a slot
// holds zero, this launch's word for the step or its word of two steps
// before.  Every wait is bounded: a wait that runs out sets a sticky error
// word, every other wait sees it and stops, the remaining ids are written as
// -1, and the launch still ends (every workgroup reaches the end, the last
// one resets the error word and advances the generation).  The workgroups
// must be resident at once (one per CU) for the waits to succeed.
//
// Up to 16 rows run as one group.  17 to 32 run as two (see the kernel); a launch
// that cannot finish them leaves the rollout to the ordered one behind it.  14
// steps of 24 rows at V = 151936, G = 1024, with the copies of a runner's call:
// 577.9 us as per-step launches (argmax 17 us, GRU 8.6, rank 7.7 a step), 295.3 here.
#include <algorithm>
#include <climits>

#include "rollout_resident.h"

namespace dels {

namespace {

constexpr int kRrKs = kResidentRank / 32;             // K steps of 32 over r
constexpr int kRrRankWGs = kResidentRank / 16;        // rank column tiles, one workgroup each
constexpr int kRrHPitch = kResidentMaxG + 8;          // bf16 per row of the state in LDS (rows 16 B apart in banks)
constexpr int kRrRPitch = kResidentRank + 8;          // bf16 per row of the rank in LDS
constexpr int kRrUnionBytes = std::max(kResidentLdsTiles * kRrKs * 1024, (kResidentMaxG / 32) * 1024);

struct RrArgs {
    const uint16_t* w_hh; const uint16_t* b_hh;     // [3G, G] MFMA-16 blocks, [3G] or null
    const uint16_t* A; const uint16_t* rank_b;      // [r, G] MFMA-16 blocks, [r] or null
    int act;
    const uint16_t* B;                              // [V, r] MFMA-16 blocks
    const uint16_t* gi_table; int64_t ld_gi; int64_t table_rows;
    const int64_t* prefix; int64_t ld_prefix;       // row m at prefix[m * ld_prefix]
    const void* base; int64_t ld_base;              // row m, step s at base + m * ld_base + s * V (elements)
    const void* prior;
    const float* alpha; const float* beta;          // [steps]
    int M, G, V, steps, ntiles, upw;                // upw: GRU units per workgroup
    int mp_shift;                                   // log2 of M rounded up to a power of two
    int np_shift;                                   // log2(upw / 2): state words per row and workgroup
    int64_t* out_ids; float* out_scores;            // row m, step s at [m * ld_out + s]
    int64_t ld_out;
    unsigned int* counters;                         // control area
    unsigned long long* h_words;                    // per workgroup: rows x upw/2 words, on lines of its own
    unsigned long long* rank_words;                 // per rank workgroup: rows x 8 words
    unsigned long long* slots;                      // [2][RG][nwg][16]: parity, group, workgroup (a line each), row
    unsigned long long* arrivals;                   // two groups: a word per workgroup, on lines of their own
    int spin_limit;
};

// RG: groups of 16 rows.  With two, the even workgroups advance the GRU (and the
// rank) of rows 0..15 and the odd ones that of rows 16..: each group's state is
// exchanged among half the workgroups, which own twice the units, so that no
// workgroup reads more state words than with 16 rows; every workgroup contracts
// its tiles of B with both groups' ranks.  A group's rows are numbered from its
// first: M rows of the group from row m0 of the batch.
template <int RG, typename BaseT, typename PriorT, bool VEC>
__global__ __launch_bounds__(kRrThreads) void rollout_resident_kernel(RrArgs a) {
#pragma clang fp contract(off)
    constexpr int kUnitTiles = RG;                  // operand tiles of W_hh rows: RG * 4 units x 3 gates
    constexpr int kGhPitch = 16 * kUnitTiles;
    __shared__ __attribute__((aligned(16))) uint16_t s_h[16 * kRrHPitch];        // the state, rows >= M zero
    __shared__ __attribute__((aligned(16))) char s_whh[(kResidentMaxG / 32) * 1024];   // W_hh rows of the units
    __shared__ __attribute__((aligned(16))) char s_union[kRrUnionBytes];       // A rows (rank WGs) or B tiles
    __shared__ __attribute__((aligned(16))) uint16_t s_rank[RG * 16 * kRrRPitch];
    __shared__ __attribute__((aligned(16))) float s_red[RG * kRrWaves * 256];
    __shared__ __attribute__((aligned(16))) float s_prior[kRrPriorWords];
    __shared__ unsigned long long s_key[kRrWaves][RG * 16];    // each wave's best key of each row
    __shared__ float s_gh[16 * kGhPitch];
    __shared__ float s_ab[2][kResidentMaxSteps];          // alpha, beta of each step
    __shared__ float s_bias[16 * kUnitTiles + 16];                        // b_hh of the operand rows, rank bias of the tile
    __shared__ unsigned long long s_rowmax[16];           // the step's maximum slot word of each row
    __shared__ int64_t s_ids[16];
    __shared__ int s_flag;

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane & 15, kg = lane >> 4;
    const int w = blockIdx.x, nwg = gridDim.x;
    const int grp = RG == 2 ? (w & 1) : 0, wg = RG == 2 ? w >> 1 : w, ng = nwg / RG;   // group, place in it, its size
    const int m0 = 16 * grp;
    const int G = a.G, KB = G / 32, V = a.V;
    const int M = RG == 2 ? (grp ? a.M - 16 : 16) : a.M;
    const uint32_t gen = __hip_atomic_load(a.counters + kDecodeGenWord, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const BaseT* base = static_cast<const BaseT*>(a.base);
    const PriorT* prior = static_cast<const PriorT*>(a.prior);
    const bool rank_wg = wg < kRrRankWGs;

    // ---- this workgroup's vocabulary tiles [T0, T1): 32 for a rank workgroup, the
    // rest shared evenly by the others (the plan checks they fit)
    int T0, T1;
    {
        const int first = min(a.ntiles, RG * kRrRankWGs * kRrWaves * kRrRegTiles);
        if (rank_wg) {
            T0 = min(a.ntiles, w * kRrWaves * kRrRegTiles);
            T1 = min(a.ntiles, T0 + kRrWaves * kRrRegTiles);
        } else {
            const int rest = a.ntiles - first, j = w - RG * kRrRankWGs, n = nwg - RG * kRrRankWGs;
            T0 = first + (int)(((int64_t)j * rest) / n);
            T1 = first + (int)(((int64_t)(j + 1) * rest) / n);
        }
    }
    const int ntl = T1 - T0;
    // register tile j of this wave: T0 + wave + 8 j; LDS tile e (e < ntl - 32): T0 + 32 + e, contracted by wave e
    const int nlds = max(0, ntl - kRrWaves * kRrRegTiles);
    const bool has_lds_tile = wave < nlds;

    const int u0 = wg * a.upw;   // this workgroup's first GRU unit
    const int upt = RG == 2 ? min(a.upw, 4) : a.upw;   // units per operand tile
    for (int i = threadIdx.x; i < 16 * kRrHPitch / 2; i += kRrThreads) reinterpret_cast<uint32_t*>(s_h)[i] = 0u;
    for (int i = threadIdx.x; i < RG * 16 * kRrRPitch / 2; i += kRrThreads) reinterpret_cast<uint32_t*>(s_rank)[i] = 0u;
    for (int i = threadIdx.x; i < a.steps; i += kRrThreads) {
        s_ab[0][i] = a.alpha[i];
        s_ab[1][i] = a.beta[i];
    }
    if (threadIdx.x < 16) {
        const int j = threadIdx.x;
        float br = 0.f;
#pragma unroll
        for (int t = 0; t < kUnitTiles; ++t) {
            float bh = 0.f;
            if (a.b_hh && j < 3 * upt && (RG == 1 || t * upt < a.upw)) {
                const int g = j / upt, u = u0 + t * upt + (j - g * upt);
                bh = bf16_bits_to_f32(a.b_hh[g * G + u]);
            }
            s_bias[16 * t + j] = bh;
        }
        if (rank_wg && a.rank_b) br = bf16_bits_to_f32(a.rank_b[wg * 16 + j]);
        s_bias[16 * kUnitTiles + j] = br;
        s_rowmax[j] = 0ull;
    } else if (RG == 1 && threadIdx.x < 48) {
        // this workgroup's slots of both parity sets back to zero; waiting for the
        // old values means the exchanges are done before the barrier below, so
        // before the prefix state words that every reader waits for
        const int p = (threadIdx.x - 16) >> 4, m = threadIdx.x & 15;
        const unsigned long long old = __hip_atomic_exchange(a.slots + p * kRrSlotSet + w * 16 + m, 0ull,
                                                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("" ::"v"(old));
    }
    __syncthreads();

    // ---- the exchanges' word blocks: the state (upw / 2 words per row and
    // workgroup, each workgroup on lines of its own), the rank (8 words per row
    // and rank workgroup), the argmax slots (one word per row and workgroup, a
    // line per workgroup)
    const int mp = a.mp_shift;
    const RrWords h_pl{ng << (mp + a.np_shift), mp + a.np_shift, max(4, mp + a.np_shift), a.np_shift, mp, M};
    const RrWords r_pl{kRrRankWGs << (mp + 3), mp + 3, mp + 3, 3, mp, M};
    const RrWords s_pl{nwg << mp, mp, 4, 0, mp, M};
    // each group's words in a region of their own (one group: the region)
    unsigned long long* const h_words = a.h_words + (RG == 2 ? grp * (int)(kResidentHWordBytes / 8) : 0);
    constexpr int kRankGroup = (int)(kResidentRankWordBytes / 8);
    unsigned long long* const rank_words = a.rank_words + (RG == 2 ? grp * kRankGroup : 0);
    const uint32_t atag = rr_tag(gen, 255);
    bool ok = true;
    if constexpr (RG == 2) {
        // The words lie in the data region, where anything may have been left: each
        // workgroup clears the words it will write and only then publishes an
        // arrival word (in the region of tagged words); everyone waits for all
        // arrivals (below) before it reads any other word.  The wait is short and
        // also tells whether the whole grid is resident.
        const int nh = 1 << h_pl.stride;                  // state words of this workgroup
        const int nr = rank_wg ? 1 << r_pl.stride : 0;
        for (int i = threadIdx.x; i < nh + nr + 64; i += kRrThreads) {
            unsigned long long* p = i < nh ? h_words + ((int64_t)wg << h_pl.stride) + i
                                    : i < nh + nr ? rank_words + ((int64_t)wg << r_pl.stride) + (i - nh)
                                    : a.slots + ((i - nh - nr) >> 4) * kRrSlotSet + w * 16 + ((i - nh - nr) & 15);
            const unsigned long long old = __hip_atomic_exchange(p, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            asm volatile("" ::"v"(old));
        }
        __syncthreads();
        if (threadIdx.x == 0)
            __hip_atomic_store(a.arrivals + w * 16, (unsigned long long)atag << 32, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
    }

    // ---- pieces of a step ----------------------------------------------------------
    // gh of the workgroup's units from the state in s_h (zero previous state:
    // no product) into s_gh[m * 16 + j], bf16-rounded after the bias.
    auto compute_gh = [&](bool zero_state) __attribute__((always_inline)) {
        f32x4 acc[kUnitTiles];
#pragma unroll
        for (int t = 0; t < kUnitTiles; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (!zero_state) {
            for (int kb = wave; kb < KB; kb += kRrWaves) {
                const bf16x8 hv = *reinterpret_cast<const bf16x8*>(&s_h[col * kRrHPitch + kb * 32 + kg * 8]);
                const bf16x8 wv = *reinterpret_cast<const bf16x8*>(s_whh + kb * 1024 + lane * 16);
                acc[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(hv, wv, acc[0], 0, 0, 0);
                if constexpr (RG == 2) {
                    // the second tile's rows do not fit the LDS beside the rest: from the L2 every step
                    const int g = col / upt, row = g * G + u0 + upt + (col - g * upt);
                    const bool live = col < 3 * upt && upt < a.upw;
                    const u32x4 w1 = *reinterpret_cast<const u32x4*>(
                        a.w_hh + ((int64_t)((live ? row : 0) >> 4) * KB + kb) * 512 + ((live ? row & 15 : 0) + 16 * kg) * 8);
                    acc[kUnitTiles - 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        hv, masked_bf16x8(w1, live ? ~0u : 0u), acc[kUnitTiles - 1], 0, 0, 0);
                }
            }
        }
#pragma unroll
        for (int t = 0; t < kUnitTiles; ++t)
            *reinterpret_cast<f32x4*>(&s_red[t * kRrWaves * 256 + wave * 256 + lane * 4]) = acc[t];
        __syncthreads();
        if (RG == 2 || threadIdx.x < 256) {
            // element (row m, operand row j): lane (m/4)*16 + j, entry m%4
            const int t = RG == 2 ? (int)threadIdx.x >> 8 : 0;
            const int m = (threadIdx.x & 255) >> 4, j = threadIdx.x & 15;
            const int e = t * kRrWaves * 256 + ((((m >> 2) * 16 + j) << 2) + (m & 3));
            float v = s_red[e];
#pragma unroll
            for (int ww = 1; ww < kRrWaves; ++ww) v = v + s_red[ww * 256 + e];
            if (a.b_hh) v = v + s_bias[16 * t + j];
            s_gh[m * kGhPitch + 16 * t + j] = round_bf16(v);
        }
        __syncthreads();
    };
    // the workgroup's units of the next state for tokens tok[m], published as words
    auto gru_publish = [&](const int64_t* tok, int64_t tok_stride, uint32_t tag) __attribute__((always_inline)) {
        const int np = a.upw / 2;   // words per row
        if ((int)threadIdx.x < M * np) {
            const int m = threadIdx.x / np, p = threadIdx.x - m * np;
            int64_t t = tok[(int64_t)m * tok_stride];
            t = t < 0 ? 0 : (t >= a.table_rows ? a.table_rows - 1 : t);
            const uint16_t* gi = a.gi_table + t * a.ld_gi + u0 + 2 * p;
            // the six input-table values first: one memory round trip
            uint16_t gv[3][2];
#pragma unroll
            for (int g = 0; g < 3; ++g)
#pragma unroll
                for (int h = 0; h < 2; ++h) gv[g][h] = gi[g * G + h];
            uint32_t pair = 0;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int i = 2 * p + h, u = u0 + i;
                const int gi0 = RG == 2 && i >= upt ? m * kGhPitch + 16 + i - upt : m * kGhPitch + i;   // gate r of unit i
                const float hv = bf16_bits_to_f32(s_h[m * kRrHPitch + u]);
                const float v = gru_unit(bf16_bits_to_f32(gv[0][h]), bf16_bits_to_f32(gv[1][h]),
                                         bf16_bits_to_f32(gv[2][h]), s_gh[gi0], s_gh[gi0 + upt],
                                         s_gh[gi0 + 2 * upt], hv);
                pair |= (uint32_t)f32_to_bf16_bits(v) << (16 * h);
            }
            __hip_atomic_store(h_words + h_pl.addr((m << a.np_shift) + p + (wg << h_pl.blk)),
                               ((unsigned long long)tag << 32) | pair, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    };
    // every row's state from the words into s_h
    auto read_state = [&](uint32_t tag) __attribute__((always_inline)) -> bool {
        auto map = [&](int j) {
            const int m = h_pl.row_of(j), wp = j >> h_pl.blk, p = j & ((1 << a.np_shift) - 1);
            return reinterpret_cast<uint32_t*>(&s_h[m * kRrHPitch + wp * a.upw + 2 * p]);
        };
        // as few loads per thread as cover the words
        if (h_pl.n <= 4 * kRrThreads) return rr_read_words<4>(a, h_words, h_pl, tag, map);
        if (h_pl.n <= 8 * kRrThreads) return rr_read_words<8>(a, h_words, h_pl, tag, map);
        return rr_read_words<16>(a, h_words, h_pl, tag, map);
    };
    // rank workgroup: its 16 columns of the rank from s_h, published as words
    auto rank_publish = [&](uint32_t tag) __attribute__((always_inline)) {
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
        for (int kb = wave; kb < KB; kb += kRrWaves) {
            const bf16x8 hv = *reinterpret_cast<const bf16x8*>(&s_h[col * kRrHPitch + kb * 32 + kg * 8]);
            const bf16x8 av = *reinterpret_cast<const bf16x8*>(s_union + kb * 1024 + lane * 16);
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(hv, av, acc, 0, 0, 0);
        }
        *reinterpret_cast<f32x4*>(&s_red[wave * 256 + lane * 4]) = acc;
        __syncthreads();
        if (threadIdx.x < 128) {
            const int m = threadIdx.x >> 3, p = threadIdx.x & 7;
            if (m < M) {
                uint32_t pair = 0;
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int n = 2 * p + h;
                    const int e = (((m >> 2) * 16 + n) << 2) + (m & 3);
                    float v = s_red[e];
#pragma unroll
                    for (int ww = 1; ww < kRrWaves; ++ww) v = v + s_red[ww * 256 + e];
                    if (a.rank_b) v = v + s_bias[16 * kUnitTiles + n];
                    v = round_bf16(v);
                    if (a.act == 1) v = round_bf16(silu_f32(v));
                    pair |= (uint32_t)f32_to_bf16_bits(v) << (16 * h);
                }
                __hip_atomic_store(rank_words + r_pl.addr((wg << r_pl.blk) + (m << 3) + p),
                                   ((unsigned long long)tag << 32) | pair, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
        __syncthreads();   // s_red is reused
    };
    auto read_rank = [&](uint32_t tag) __attribute__((always_inline)) -> bool {
        if constexpr (RG == 2) {
            // both groups' words in one gather: producer wr of group wr / kRrRankWGs
            const RrWords pl{2 * kRrRankWGs << 7, 7, 7, 3, 4, 16, kRrRankWGs << 7, a.M - 16};
            auto map = [&](int j) {
                const int m = pl.row_of(j) + 16 * (j >> 11), wr = (j >> 7) & (kRrRankWGs - 1), p = j & 7;
                return reinterpret_cast<uint32_t*>(&s_rank[m * kRrRPitch + wr * 16 + 2 * p]);
            };
            return rr_read_words<8>(a, a.rank_words, pl, tag, map);
        }
        auto map = [&](int j) {
            const int m = r_pl.row_of(j), wr = j >> r_pl.blk, p = j & 7;
            return reinterpret_cast<uint32_t*>(&s_rank[m * kRrRPitch + wr * 16 + 2 * p]);
        };
        if (r_pl.n <= 2 * kRrThreads) return rr_read_words<2>(a, rank_words, r_pl, tag, map);
        return rr_read_words<4>(a, rank_words, r_pl, tag, map);
    };

    // ---- prefix: h_0 = GRU(gi_table[prefix], 0) --------------------------------
    compute_gh(true);
    gru_publish(a.prefix + m0 * a.ld_prefix, a.ld_prefix, rr_tag(gen, 0));

    // ---- resident operands, loaded while the prefix state travels (a read
    // waits for every load issued before it, so the state went out first):
    // the LDS operands, then this wave's register tiles of B
    if (rank_wg) {
        // A rows 16 wg .. 16 wg + 15: the MFMA-16 blocks of that row block, in order
        for (int i = threadIdx.x; i < KB * 64; i += kRrThreads) {
            const int kb = i >> 6, l = i & 63;
            *reinterpret_cast<u32x4*>(s_union + kb * 1024 + l * 16) =
                *reinterpret_cast<const u32x4*>(a.A + ((int64_t)wg * KB + kb) * 512 + l * 8);
        }
    } else {
        for (int i = threadIdx.x; i < nlds * kRrKs * 64; i += kRrThreads) {
            const int e = i / (kRrKs * 64), rem = i - e * (kRrKs * 64), s = rem >> 6, l = rem & 63;
            const int t = T0 + kRrWaves * kRrRegTiles + e;
            *reinterpret_cast<u32x4*>(s_union + (e * kRrKs + s) * 1024 + l * 16) =
                *reinterpret_cast<const u32x4*>(a.B + ((int64_t)t * kRrKs + s) * 512 + l * 8);
        }
    }
    // W_hh rows of the first operand tile, units u0 .. u0 + upt - 1: operand row
    // j = g * upt + i holds row g * G + u0 + i of W_hh (rows past 3 upt are zero)
    for (int i = threadIdx.x; i < KB * 64; i += kRrThreads) {
        const int kb = i >> 6, l = i & 63;
        const int j = l & 15, oct = l >> 4;
        u32x4 v = {0u, 0u, 0u, 0u};
        if (j < 3 * upt) {
            const int g = j / upt, row = g * G + u0 + (j - g * upt);
            v = *reinterpret_cast<const u32x4*>(a.w_hh + ((int64_t)(row >> 4) * KB + kb) * 512 + ((row & 15) + 16 * oct) * 8);
        }
        *reinterpret_cast<u32x4*>(s_whh + kb * 1024 + l * 16) = v;
    }
    // the prior of every column of the workgroup's tiles (widened)
    if (threadIdx.x < 16) s_prior[kRrPriorZeros + threadIdx.x] = 0.f;
    for (int i = threadIdx.x; i < ntl * 16; i += kRrThreads) {
        const int v = min(T0 * 16 + i, V - 1);
        if constexpr (is_no_prior<PriorT>::value) s_prior[i] = 0.f;
        else s_prior[i] = widen_raw<PriorT>(load_raw(prior + v));
    }
    // the register tiles after the LDS operands (whose stores wait for their loads)
    asm volatile("" ::: "memory");
    bf16x8 bt[kRrRegTiles][kRrKs];
#pragma unroll
    for (int j = 0; j < kRrRegTiles; ++j) {
        // a tile that is not this wave's loads the last tile (in bounds) and keeps zeros
        const int ti = wave + 8 * j;
        const int t = min(T0 + ti, a.ntiles - 1);
        const uint32_t keep = ti < ntl ? ~0u : 0u;
#pragma unroll
        for (int s = 0; s < kRrKs; ++s)
            bt[j][s] = masked_bf16x8(__builtin_nontemporal_load(reinterpret_cast<const u32x4*>(
                                         a.B + ((int64_t)t * kRrKs + s) * 512 + lane * 8)),
                                     keep);
    }

    if constexpr (RG == 2) {
        RrArgs first = a;
        first.spin_limit = min(a.spin_limit, kRrArrivalLimit);
        const RrWords pl{nwg, 0, 4, 0, 0, 1};
        unsigned long long word[1];
        const bool got = rr_gather<1>(first, a.arrivals, pl, (int)threadIdx.x, word,
                                      [&](unsigned long long x) { return (uint32_t)(x >> 32) == atag; });
        ok = !__syncthreads_or(!got);
    }
    if (ok) ok = read_state(rr_tag(gen, 0));

    int s = 0;
    for (; ok && s < a.steps; ++s) {
        const uint32_t tag = rr_tag(gen, s);
        // lane values pass through an empty asm statement each step, so that the
        // compiler forms the step's addresses here instead of holding them in
        // registers across the loop
        int lcol = col, lkg = kg;
        asm volatile("" : "+v"(lcol), "+v"(lkg));
        if (rank_wg) rank_publish(tag);
        // base values of this wave's tiles, issued before the rank wait; the second
        // group's after it where they are two words a tile, else when its turn comes
        constexpr bool kBoth = RG == 2 && sizeof(BaseT) == 2;
        RrBase<BaseT> braw[kBoth ? 2 : 1];
        auto load_base = [&](int g) __attribute__((always_inline)) {
            const int m = 16 * g + lcol;
            rr_load_base<BaseT, VEC>(base + (int64_t)s * V + (int64_t)(m < a.M ? m : 0) * a.ld_base, T0, ntl,
                                     a.ntiles, wave, lkg, V, braw[kBoth ? g : 0]);
        };
        load_base(0);
        // keep these loads ahead of the rank wait (the compiler would otherwise
        // issue them after it, where their round trip adds to the step)
        asm volatile("" ::: "memory");
        ok = read_rank(tag);
        if (!ok) break;
        if constexpr (kBoth) load_base(1);

        // ---- argmax over the resident tiles -------------------------------------
        const bool lds_tile = !rank_wg && has_lds_tile;
        const char* ltile = s_union + (lds_tile ? wave : 0) * kRrKs * 1024;
#pragma unroll
        for (int g = 0; g < RG; ++g) {
            if (g > 0 && !kBoth) load_base(g);
            const unsigned long long key = rr_tiles_best<kRrKs, BaseT, PriorT, VEC>(
                bt, ltile, lds_tile, &s_rank[(16 * g + lcol) * kRrRPitch + lkg * 8], braw[kBoth ? g : 0], s_prior, T0,
                ntl, wave, lkg, V, s_ab[0][s], s_ab[1][s]);
            if (kg == 0) s_key[wave][16 * g + col] = key;
        }
        __syncthreads();
        // the workgroup's best of each row into its slot word for the step
        const uint32_t low2 = 1u | ((((uint32_t)s >> 1) & 1u) << 1);
        unsigned long long* slot_set = a.slots + (s & 1) * RG * kRrSlotSet;
        unsigned long long* const own_set = slot_set + (RG == 2 ? grp * kRrSlotSet : 0);
        if ((int)threadIdx.x < a.M) {
            const int m = threadIdx.x;
            unsigned long long k = s_key[0][m];   // order(score) << 32 | ~index
#pragma unroll
            for (int ww = 1; ww < kRrWaves; ++ww) k = max(k, s_key[ww][m]);
            // no candidate (index INT_MAX) leaves the index field zero: index
            // 2^30 - 1, past every vocabulary, below every real candidate
            const unsigned long long word =
                low2 | (k & 0xffffffff00000000ull) | ((unsigned long long)((uint32_t)k & 0x3fffffffu) << 2);
            __hip_atomic_store(slot_set + (RG == 2 ? (m >> 4) * kRrSlotSet + w * 16 + (m & 15) : w * 16 + m), word,
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }

        // next step's gh while the slot words travel (every workgroup: placed
        // before the rank wait it would delay the rank workgroups' argmax, and
        // with it every workgroup's slot read)
        if (s + 1 < a.steps) compute_gh(false);

        // ---- the step's ids (every workgroup: its GRU units need them) ---------------
        const bool need = s + 1 < a.steps || wg == 0;
        if (need) {
            if (s_pl.n <= 2 * kRrThreads) ok = rr_slot_maxima<2>(a, own_set, s_pl, low2, s_rowmax);
            else if (s_pl.n <= 4 * kRrThreads) ok = rr_slot_maxima<4>(a, own_set, s_pl, low2, s_rowmax);
            else ok = rr_slot_maxima<8>(a, own_set, s_pl, low2, s_rowmax);
            if (!ok) break;
            if (threadIdx.x < 16) {
                const int m = threadIdx.x;
                int64_t id = 0;
                float val = -__builtin_inff();
                if (m < M) {
                    const unsigned long long key = s_rowmax[m];
                    s_rowmax[m] = 0ull;   // for the next step (barriers come between)
                    const uint32_t idx = ~(uint32_t)(key >> 2) & 0x3fffffffu;
                    if (idx < (uint32_t)V) {
                        id = idx;
                        val = f32_from_order_key((uint32_t)(key >> 32));
                    }
                    if (wg == 0) {
                        a.out_ids[(int64_t)(m0 + m) * a.ld_out + s] = id;
                        if (a.out_scores) a.out_scores[(int64_t)(m0 + m) * a.ld_out + s] = val;
                    }
                }
                s_ids[m] = id;
            }
            __syncthreads();
        }
        if (s + 1 < a.steps) {
            gru_publish(s_ids, 1, rr_tag(gen, s + 1));
            // the other workgroups read the state later than those that project the
            // rank from it: 8 MB of words (8 rows) on their way to everyone at once
            // delay the ones that the step waits for.  14 steps at V = 151936 without
            // and with the pause, G = 1024: 1 / 4 / 8 / 16 rows 160 / 153 / 165 / 203 ->
            // 149 / 148 / 161 / 197 us, 17 / 24 / 32 rows 253 / 250 / 262 -> 243 / 242 /
            // 251; G = 512: 1 / 8 / 16 rows 159 / 155 / 175 -> 145 / 152 / 173, likewise
            // at V = 2000 to 100000 (half the pause gains nothing, more loses again).  Two
            // groups at G = 512 have half the words: 206 / 206 / 213 without, 211 / 209 /
            // 218 with, so they take none.
            if (!rank_wg && (RG == 1 || a.upw > 4)) __builtin_amdgcn_s_sleep(RG == 1 ? 40 : 56);
            ok = read_state(rr_tag(gen, s + 1));
        }
    }
    if (!ok) {
        if (threadIdx.x == 0) rr_fail(a);
        // the ids this launch could not produce (two groups: the ordered rollout produces them all)
        if (RG == 1 && w == 0) {
            for (int i = threadIdx.x; i < M * a.steps; i += kRrThreads) {
                const int m = i / a.steps, st = i - m * a.steps;
                if (st >= s) {
                    a.out_ids[(int64_t)m * a.ld_out + st] = -1;
                    if (a.out_scores) a.out_scores[(int64_t)m * a.ld_out + st] = -__builtin_inff();
                }
            }
        }
    }

    // ---- the last workgroup clears the control area and advances the generation
    __syncthreads();
    if (threadIdx.x == 0) {
        __builtin_amdgcn_s_waitcnt(0);   // a failure is stored before this workgroup counts as done
        const unsigned prev = __hip_atomic_fetch_add(a.counters + kRrDoneCounter, 1u, __ATOMIC_RELAXED,
                                                     __HIP_MEMORY_SCOPE_AGENT);
        s_flag = prev == (unsigned)nwg - 1 ? 3 : 0;
    }
    __syncthreads();
    if (s_flag != 3) return;
    if (threadIdx.x == 0) {
        const unsigned failed = __hip_atomic_exchange(a.counters + kRrErrorWord, 0u, __ATOMIC_RELAXED,
                                                      __HIP_MEMORY_SCOPE_AGENT);
        if (RG == 2) __hip_atomic_store(a.counters + kRrNotDoneWord, failed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(a.counters + kRrDoneCounter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_fetch_add(a.counters + kDecodeGenWord, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

template <int RG, typename BaseT, bool VEC>
hipError_t launch_rr_base(const RrArgs& a, int prior_kind, int nwg, hipStream_t s) {
    const dim3 grid(nwg), block(kRrThreads);
    switch (prior_kind) {
        case 0: hipLaunchKernelGGL((rollout_resident_kernel<RG, BaseT, no_prior_t, VEC>), grid, block, 0, s, a); break;
        case 1: hipLaunchKernelGGL((rollout_resident_kernel<RG, BaseT, float, VEC>), grid, block, 0, s, a); break;
        case 2: hipLaunchKernelGGL((rollout_resident_kernel<RG, BaseT, bf16_t, VEC>), grid, block, 0, s, a); break;
        default: hipLaunchKernelGGL((rollout_resident_kernel<RG, BaseT, f16_t, VEC>), grid, block, 0, s, a); break;
    }
    return hipGetLastError();
}

template <int RG>
hipError_t launch_rr(const RrArgs& a, int base_dtype, int prior_kind, int nwg, hipStream_t s) {
    auto by_base = [&](auto vec) -> hipError_t {
        constexpr bool VEC = decltype(vec)::value;
        if (base_dtype == 1) return launch_rr_base<RG, bf16_t, VEC>(a, prior_kind, nwg, s);
        if (base_dtype == 2) return launch_rr_base<RG, f16_t, VEC>(a, prior_kind, nwg, s);
        return launch_rr_base<RG, float, VEC>(a, prior_kind, nwg, s);
    };
    return rr_vec(a.base, base_dtype, a.ld_base, a.V) ? by_base(std::true_type{}) : by_base(std::false_type{});
}

int g_resident_spin_limit = 1 << 16;   // re-reads before a wait gives up (each ~1-2 us)
int g_resident_enabled = 1;

}  // namespace

int resident_spin_limit() { return g_resident_spin_limit; }
int set_resident_spin_limit(int limit) {
    const int prev = g_resident_spin_limit;
    g_resident_spin_limit = std::max(0, limit);
    return prev;
}
int set_rollout_resident(int enable) {   // 0: off, 1: where it pays, 2: wherever it can run
    const int prev = g_resident_enabled;
    g_resident_enabled = std::max(0, std::min(enable, 2));
    return prev;
}
bool rollout_resident_enabled() { return g_resident_enabled != 0; }
bool rollout_resident_forced() { return g_resident_enabled > 1; }

// Two groups of rows take about 18 to 25 us before their first step (B and the
// other operands on chip) and 13 to 16 a step, the per-step launches 2 to 4 and 17
// to 35: one step is always theirs (17 rows, G = 1024, V = 32000: 27 / 38 us), two
// on a short vocabulary (V = 32000: 49 / 55; V = 65536 53 / 55; V = 151936 64 /
// 57), three are even at the shortest (V = 2000: 63 / 64).
bool rollout_resident_pays(int64_t batch, int64_t V, int64_t steps) {
    return batch <= 16 || steps >= 3 || (steps == 2 && V >= 65536);
}

bool rollout_resident_eligible(int64_t batch, int64_t G, int64_t r, int64_t V, int64_t steps, bool packed,
                               size_t ws_bytes) {
    const int nwg = device_cu_count();
    if (!packed || batch < 1 || batch > 32 || r != kResidentRank || steps < 1 || steps > kResidentMaxSteps) return false;
    const int rg = batch > 16 ? 2 : 1;
    if (rg == 2 && ws_bytes < kDataOff + kResident2Bytes) return false;
    if (G < 64 || G > kResidentMaxG || (G & (G - 1)) != 0 || G % nwg != 0) return false;
    // slot rows of whole 64-word chunks, at most the slots the workspace holds
    if (nwg < 64 || nwg > kResidentMaxWGs || nwg % 64 != 0 || V >= (int64_t)1 << 30) return false;
    const int upw = (int)(G / (nwg / rg));
    if (upw % 2 != 0 || upw > 4 * rg) return false;   // up to four units (12 gate rows) per operand tile
    const int64_t ntiles = (V + 15) / 16;
    const int64_t first = std::min<int64_t>(ntiles, (int64_t)rg * kRrRankWGs * kRrWaves * kRrRegTiles);
    const int64_t rest = ntiles - first, others = nwg - rg * kRrRankWGs;
    const int64_t per = (rest + others - 1) / others;
    return per <= kRrWaves * kRrRegTiles + kResidentLdsTiles;
}

hipError_t launch_rollout_resident(const ResidentRolloutArgs& r, void* ws, hipStream_t s) {
    char* w = static_cast<char*>(ws);
    RrArgs a{};
    a.w_hh = r.w_hh; a.b_hh = r.b_hh;
    a.A = r.A; a.rank_b = r.rank_b; a.act = r.act;
    a.B = r.B;
    a.gi_table = r.gi_table; a.ld_gi = r.ld_gi; a.table_rows = r.table_rows;
    a.prefix = r.prefix; a.ld_prefix = r.ld_prefix;
    a.base = r.base; a.ld_base = r.ld_base;
    a.prior = r.prior;
    a.alpha = r.alpha; a.beta = r.beta;
    a.M = (int)r.batch; a.G = (int)r.G; a.V = (int)r.V; a.steps = (int)r.steps;
    a.ntiles = (int)((r.V + 15) / 16);
    const int nwg = device_cu_count();
    const int rg = a.M > 16 ? 2 : 1;
    a.upw = (int)(r.G / (nwg / rg));
    a.mp_shift = 0;
    while ((1 << a.mp_shift) < std::min(a.M, 16)) ++a.mp_shift;
    a.np_shift = 0;
    while ((2 << a.np_shift) < a.upw) ++a.np_shift;   // upw / 2 = 1 << np_shift (upw a power of two)
    a.out_ids = r.out_ids; a.out_scores = r.out_scores; a.ld_out = r.ld_out;
    a.counters = reinterpret_cast<unsigned int*>(w + kCountersOff);
    // one group: the regions that only this kernel writes; two: the data region
    char* words = rg == 2 ? w + kDataOff : w + kResidentOff;
    a.h_words = reinterpret_cast<unsigned long long*>(words);
    a.rank_words = reinterpret_cast<unsigned long long*>(words + rg * kResidentHWordBytes);
    a.slots = reinterpret_cast<unsigned long long*>(words + rg * (kResidentHWordBytes + kResidentRankWordBytes));
    a.arrivals = reinterpret_cast<unsigned long long*>(w + kResidentOff);
    a.spin_limit = resident_spin_limit();
    const int pk = r.prior == nullptr ? 0 : (r.prior_dtype == 1 ? 2 : (r.prior_dtype == 2 ? 3 : 1));
    if (rg == 1) return launch_rr<1>(a, r.base_dtype, pk, nwg, s);
    const hipError_t e = launch_rr<2>(a, r.base_dtype, pk, nwg, s);
    return e != hipSuccess ? e : launch_rollout_ordered(r, ws, s);
}

}  // namespace dels
