// Fused low-rank LM-head combine + vocabulary argmax for 17 to 64 rows per
// pass over B: the streaming kernel between the 16-row GEMV kernel and the
// MFMA-tiled one, and the general one for more rows wherever the tiled kernel
// does not apply (row-major B, unaligned rows, a rank it does not take).
//
// Semantics as the GEMV kernel (code/kernel/dels.py:42-138):
//     s[m, v] = fma(-beta_m, prior[v], fma(fp32(rank_m . B[v]), alpha_m, base[m, v]))
// and per row the lowest v attaining max_v s[m, v].  The contraction sums the
// same MFMA K steps in the same order, so scores equal the GEMV kernel's bit
// for bit.
//
// Bound by streaming B from HBM once, so every 16-row vocabulary tile that a
// wave loads serves all the rows of its workgroup, RG groups of 16, instead of
// being read again for every 16 rows.  The groups' rank operands lie in LDS in
// operand order (RG * r * 32 bytes: 64 KiB for 64 rows at r = 512; each read is
// one bank-conflict-free KiB, which feeds one MFMA: at 64 rows the LDS and the
// matrix cores are each busy for 8 of the ~27 us the stream takes), which leaves
// the registers to the stream: two waves per SIMD with two tiles each in flight.
// (With the operands in registers, one wave per SIMD: 40 / 48 rows 38.5 / 39.7
// us a launch, 33.9 / 34.7 here at r = 512, V = 151936; 40 rows in the GEMV
// kernel, 104.)  The
// tile is the MFMA's A operand and the rank its B operand: lane l ends with row
// l % 16 of each group and the four consecutive columns 4 (l / 16) .. + 3, so
// that a lane's base logits are one 8- or 16-byte load per group, its prior
// values one load for all groups, and the running argmax takes one (score,
// index) pair per group.  Unaligned rows and vocabularies take the same loads
// at element alignment (load_quad_any: with four element loads instead, 63 rows
// at V = 50257 took 18.5 / 21.2 / 26.8 us at r = 128 / 256 / 512, more than the
// GEMV kernel's 13.8 / 17.4 / 24.8; as quads 11.7 / 14.2 / 18.3).  Tiles are
// walked wave-strided through two register sets, refills unconditional, as in the
// GEMV kernel.
#pragma once

#include <mutex>

#include "fused_argmax_gemv.h"
#include "fused_argmax_tiled.h"

namespace dels {

namespace rows {

constexpr int kWaves = 8;
constexpr int kThreads = kWaves * 64;

// The four consecutive values a lane takes from a row per tile, as loaded: two
// words of 16-bit values, four of fp32.
template <typename T>
constexpr int quad_words() { return sizeof(T) == 2 ? 2 : 4; }
template <typename T>
using Quad = uint32_t[quad_words<T>()];

// Row offsets (bytes) fit 32 bits with VEC, so that a row costs one register.
template <bool VEC>
using RowOff = typename std::conditional<VEC, uint32_t, int64_t>::type;

// Columns v .. v + 3 of a row of four or more, at any alignment: one load at
// element alignment, taken back into the row at its end (shift_quad puts its
// elements in place when it is used).  Four element loads instead touch each of
// a wave's 16 rows four times.
template <typename T>
__device__ __forceinline__ void load_quad_any(const T* row, int v, int V, Quad<T>& w) {
    const T* p = row + min(v, V - 4);
    if constexpr (sizeof(T) == 2) {
        typedef uint64_t __attribute__((aligned(2))) u64_a2;
        const uint64_t x = *reinterpret_cast<const u64_a2*>(p);
        w[0] = (uint32_t)x; w[1] = (uint32_t)(x >> 32);
    } else {
        typedef u32x4 __attribute__((aligned(4))) u32x4_a4;
        const u32x4 x = *reinterpret_cast<const u32x4_a4*>(p);
#pragma unroll
        for (int q = 0; q < 4; ++q) w[q] = x[q];
    }
}

// The quad of columns v .. v + 3 from one that was taken back to V - 4 (columns
// past V are not used).
template <typename T>
__device__ __forceinline__ void shift_quad(Quad<T>& w, int v, int V) {
    const int d = V >= 4 ? min(max(v - (V - 4), 0), 3) : 0;
    if constexpr (sizeof(T) == 2) {
        const uint64_t x = (((uint64_t)w[1] << 32) | w[0]) >> (16 * d);
        w[0] = (uint32_t)x; w[1] = (uint32_t)(x >> 32);
    } else {
#pragma unroll
        for (int q = 0; q < 3; ++q)
#pragma unroll
            for (int o = 1; q + o < 4; ++o) w[q] = d == o ? w[q + o] : w[q];
    }
}

// VEC: aligned quads, V a multiple of 4.
template <typename T, bool VEC>
__device__ __forceinline__ void load_quad(const void* base, RowOff<VEC> row, int v, int V, Quad<T>& w) {
    const char* p = static_cast<const char*>(base);
    if constexpr (VEC) {
        const uint32_t o = row + (uint32_t)min(v, V - 4) * (uint32_t)sizeof(T);   // V a multiple of 4: whole quads
        if constexpr (sizeof(T) == 2) {
            const u32x2 x = __builtin_nontemporal_load(reinterpret_cast<const u32x2*>(p + o));
            w[0] = x[0]; w[1] = x[1];
        } else {
            const u32x4 x = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p + o));
#pragma unroll
            for (int q = 0; q < 4; ++q) w[q] = x[q];
        }
    } else {
        load_quad_any<T>(reinterpret_cast<const T*>(p + row), v, V, w);
    }
}

// Value q of a quad, widened.
template <typename T>
__device__ __forceinline__ float quad_at(const Quad<T>& w, int q) {
    if constexpr (sizeof(T) == 2) return tiled::half_at<T>(w[q >> 1], q & 1);
    else return widen_raw<T>(w[q]);
}

}  // namespace rows

// Ranks the kernel takes: whole MFMA K steps, no masked operands.
inline bool rows_rank_ok(int r) { return r == 128 || r == 256 || r == 512; }

template <int RG, int KSTEPS, typename BaseT, typename PriorT>
struct RowsTile {
    bf16x8 b[KSTEPS];
    rows::Quad<BaseT> base[RG];
    rows::Quad<PriorT> prior;
};

// End of a workgroup's share of the argmax over the rows m0 .. m0 + 16 RG - 1:
// each lane's running (score, index) pairs over the quads of columns and the
// waves, then across workgroups.
template <int RG>
__device__ __forceinline__ void rows_finish(const ArgmaxKArgs& a, float (&best)[RG], int (&bidx)[RG], int m0,
                                            float (&s_val)[rows::kWaves][16 * RG], int (&s_idx)[rows::kWaves][16 * RG],
                                            int& s_last) {
    constexpr int kRows = 16 * RG;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int col = lane & 15, kg = lane >> 4;
#pragma unroll
    for (int g = 0; g < RG; ++g) {
#pragma unroll
        for (int off = 16; off < 64; off <<= 1) {
            const float ov = __shfl_xor(best[g], off, 64);
            const int oi = __shfl_xor(bidx[g], off, 64);
            if (argmax_better(ov, oi, best[g], bidx[g])) {
                best[g] = ov;
                bidx[g] = oi;
            }
        }
        if (kg == 0) {
            s_val[wave][16 * g + col] = best[g];
            s_idx[wave][16 * g + col] = bidx[g];
        }
    }
    __syncthreads();
    int fin_m[1] = {-1};
    unsigned long long fin_key[1] = {0ull};
    if (threadIdx.x < kRows) {
        const int mi = threadIdx.x;
        float bv = s_val[0][mi];
        int bi = s_idx[0][mi];
#pragma unroll
        for (int w = 1; w < rows::kWaves; ++w) {
            if (argmax_better(s_val[w][mi], s_idx[w][mi], bv, bi)) {
                bv = s_val[w][mi];
                bi = s_idx[w][mi];
            }
        }
        if (m0 + mi < a.M) fin_m[0] = m0 + mi;
        fin_key[0] = bi == INT_MAX ? 0ull : pack_argmax(bv, (uint32_t)bi);
    }
    tiled_argmax_finish(a, fin_m, fin_key, &s_last);
}

// HAS_PRIOR false: the prior term is absent (PriorT is then BaseT and unused).
template <int RG, int KSTEPS, bool ROWMAJOR, typename BaseT, typename PriorT, bool VEC, bool HAS_PRIOR>
__global__ __launch_bounds__(rows::kThreads) void fused_argmax_rows_kernel(ArgmaxKArgs a) {
#pragma clang fp contract(off)
    using namespace rows;
    constexpr int kRows = 16 * RG;
    extern __shared__ __attribute__((aligned(16))) char s_rank[];   // [KSTEPS][RG][64 lanes][16 bytes]
    __shared__ float s_val[kWaves][kRows];
    __shared__ int s_idx[kWaves][kRows];
    __shared__ int s_last;

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // uniform: scalar loop control
    const int col = lane & 15;     // row of the lane within each group
    const int kg = lane >> 4;      // K octet of the operands / quad of columns of the results
    const int m0 = blockIdx.y * kRows;

    // Rank operands of the groups' rows, K step by K step; rows past M repeat row
    // 0 (their results are not written).  The loads go out before the stream's.
    constexpr int kPieces = RG * KSTEPS * 64 / kThreads;   // 16-byte pieces per thread
    static_assert(kPieces * kThreads == RG * KSTEPS * 64, "whole pieces per thread");
    u32x4 rp[kPieces];
#pragma unroll
    for (int i = 0; i < kPieces; ++i) {
        const int p = threadIdx.x + kThreads * i;          // piece of the LDS image: step, group, lane
        const int l = p & 63, g = (p >> 6) % RG, s = (p >> 6) / RG;
        const int m = m0 + 16 * g + (l & 15);
        rp[i] = *reinterpret_cast<const u32x4*>(
            a.rank + rank_row_of(a.rank_rows, a.rank_rows_stride, a.rank_rows_count, m < a.M ? m : 0) * a.ldrank +
            s * 32 + (l >> 4) * 8);
    }
    float al[RG], nbe[RG], best[RG];
    int bidx[RG];
    bool use_prior[RG];
    RowOff<VEC> brow[RG];
#pragma unroll
    for (int g = 0; g < RG; ++g) {
        const int m = m0 + 16 * g + col;
        const int mc = m < a.M ? m : 0;
        al[g] = a.alpha[(int64_t)mc * a.alpha_stride];
        const float be = a.beta[(int64_t)mc * a.beta_stride];
        nbe[g] = -be;
        use_prior[g] = HAS_PRIOR && be != 0.f;
        brow[g] = (RowOff<VEC>)((int64_t)mc * a.ldbase * (int64_t)sizeof(BaseT));
        best[g] = -__builtin_inff();
        bidx[g] = INT_MAX;
    }

    using Tile = RowsTile<RG, KSTEPS, BaseT, PriorT>;
    // live (uniform) false: not one of the wave's tiles -- the same loads, of one line each
    auto load = [&](int t, bool live, Tile& tr) {
        // ROWMAJOR: the lane's K octets of vocabulary row t * 16 + col; else MFMA-16 blocks
        const uint16_t* bp = ROWMAJOR ? a.B + (int64_t)(live ? min(t * 16 + col, a.V - 1) : 0) * a.ldb + kg * 8
                                      : a.B + (int64_t)t * (KSTEPS * 512) + (live ? lane * 8 : 0);
#pragma unroll
        for (int s = 0; s < KSTEPS; ++s) tr.b[s] = load_bf16x8_nt(bp + s * (ROWMAJOR ? 32 : 512));
        const int v = live ? t * 16 + 4 * kg : 0;
#pragma unroll
        for (int g = 0; g < RG; ++g) load_quad<BaseT, VEC>(a.base, live ? brow[g] : 0, v, a.V, tr.base[g]);
        if constexpr (HAS_PRIOR) load_quad<PriorT, VEC>(a.prior, 0, v, a.V, tr.prior);
    };
    auto consume = [&](Tile& tr, int t) {
        // the operands are read from LDS tile by tile: through the empty asm statement the
        // compiler cannot take them for loop invariants and hold them in registers
        int lo = lane * 16;
        asm volatile("" : "+v"(lo));
        f32x4 acc[RG];
#pragma unroll
        for (int g = 0; g < RG; ++g) acc[g] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < KSTEPS; ++s)
#pragma unroll
            for (int g = 0; g < RG; ++g)
                acc[g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                    tr.b[s], *reinterpret_cast<const bf16x8*>(s_rank + (s * RG + g) * 1024 + lo), acc[g], 0, 0, 0);
        const int v = t * 16 + 4 * kg;
        if constexpr (!VEC) {
            if (t * 16 + 16 > a.V) {   // wave-uniform
#pragma unroll
                for (int g = 0; g < RG; ++g) shift_quad<BaseT>(tr.base[g], v, a.V);
                if constexpr (HAS_PRIOR) shift_quad<PriorT>(tr.prior, v, a.V);
            }
        }
#pragma unroll
        for (int q = 3; q >= 0; --q) {
            const bool in = v + q < a.V;
            float pv = 0.f;
            if constexpr (HAS_PRIOR) pv = quad_at<PriorT>(tr.prior, q);
#pragma unroll
            for (int g = 0; g < RG; ++g) {
                float sc = __builtin_fmaf(acc[g][q], al[g], quad_at<BaseT>(tr.base[g], q));
                if constexpr (HAS_PRIOR) sc = use_prior[g] ? __builtin_fmaf(nbe[g], pv, sc) : sc;
                // a lane's candidates arrive in decreasing column order: ">=" ends at the lowest index,
                // that of a first score of -inf among them
                const bool take = in & (sc >= best[g]);
                best[g] = take ? sc : best[g];
                bidx[g] = take ? v + q : bidx[g];
            }
        }
    };

    // the wave's tiles t, t + nwaves, .. (cnt of them), the last one first, through two
    // register sets (see the GEMV kernel)
    const int ntiles = (a.V + 15) >> 4;
    const int nwaves = gridDim.x * kWaves;
    const int t = blockIdx.x * kWaves + wave;
    const int cnt = t < ntiles ? (ntiles - 1 - t) / nwaves + 1 : 0;
    const int te = t + (cnt - 1) * nwaves;
    Tile tr0, tr1;
    // the first two whether or not the wave has them, so that the waits below are exact
    load(cnt > 0 ? te : 0, cnt > 0, tr0);
    load(cnt > 1 ? te - nwaves : 0, cnt > 1, tr1);
#pragma unroll
    for (int i = 0; i < kPieces; ++i)
        *reinterpret_cast<u32x4*>(s_rank + (threadIdx.x + kThreads * i) * 16) = rp[i];
    lds_barrier();   // the stream's loads stay in flight
    int k = 0;
    for (; k + 4 <= cnt; k += 2) {
        consume(tr0, te - k * nwaves);
        load(te - (k + 2) * nwaves, true, tr0);
        consume(tr1, te - (k + 1) * nwaves);
        load(te - (k + 3) * nwaves, true, tr1);
    }
    if (k < cnt) consume(tr0, te - k * nwaves);
    if (k + 2 < cnt) load(te - (k + 2) * nwaves, true, tr0);
    if (k + 1 < cnt) consume(tr1, te - (k + 1) * nwaves);
    if (k + 2 < cnt) consume(tr0, te - (k + 2) * nwaves);

    rows_finish<RG>(a, best, bidx, m0, s_val, s_idx, s_last);
}

template <int RG, int KSTEPS, bool ROWMAJOR, typename BaseT, typename PriorT, bool VEC, bool HAS_PRIOR>
hipError_t launch_rows_inst(const ArgmaxKArgs& ka, hipStream_t s) {
    const int ntiles = (ka.V + 15) / 16;
    const int groups = (ka.M + 16 * RG - 1) / (16 * RG);
    const int cus = device_cu_count();
    const int gx = std::max(1, std::min((ntiles + rows::kWaves - 1) / rows::kWaves, (cus + groups - 1) / groups));
    constexpr size_t kLds = (size_t)RG * KSTEPS * 1024;
    // more than 64 KiB of dynamic LDS is allowed once per kernel instance (see launch_domino_inst)
    static std::once_flag once;
    static hipError_t attr_err = hipSuccess;
    std::call_once(once, [] {
        attr_err = hipFuncSetAttribute(
            reinterpret_cast<const void*>(
                &fused_argmax_rows_kernel<RG, KSTEPS, ROWMAJOR, BaseT, PriorT, VEC, HAS_PRIOR>),
            hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLds);
    });
    if (attr_err != hipSuccess) return attr_err;
    hipLaunchKernelGGL((fused_argmax_rows_kernel<RG, KSTEPS, ROWMAJOR, BaseT, PriorT, VEC, HAS_PRIOR>),
                       dim3(gx, groups, 1), dim3(rows::kThreads), kLds, s, ka);
    return hipGetLastError();
}

// Whether launch_rows_* takes a prior of this kind beside base logits of BaseT:
// none, the base's own dtype, or fp32.
inline bool rows_prior_ok(int base_dtype, int prior_kind) {
    return prior_kind == 0 || prior_kind == 1 || prior_kind == (base_dtype == 1 ? 2 : base_dtype == 2 ? 3 : 1);
}

// Dispatch over row groups, K steps / B layout, prior and vector loads for one
// base dtype (rows_rank_ok).  `vec`: every row of base (and the prior) allows
// aligned loads of four elements, V is a multiple of 4 and base spans under 4 GiB.
template <typename BaseT>
hipError_t launch_rows_for_base(const ArgmaxKArgs& ka, bool packed, int prior_kind, bool vec, hipStream_t s) {
    using True = std::true_type;
    using False = std::false_type;
    auto by_shape = [&](auto prior_tag, auto has_tag, auto vec_tag) -> hipError_t {
        using PriorT = decltype(prior_tag);
        constexpr bool HP = decltype(has_tag)::value;
        constexpr bool VEC = decltype(vec_tag)::value;
        auto by_rows = [&](auto ks_tag, auto rm_tag) -> hipError_t {
            constexpr int KS = decltype(ks_tag)::value;
            constexpr bool RM = decltype(rm_tag)::value;
            if (ka.M <= 32) return launch_rows_inst<2, KS, RM, BaseT, PriorT, VEC, HP>(ka, s);
            // three groups where their operands split evenly over the threads; eight, past
            // 64 rows, where their base logits fit the registers and B is long (200 rows,
            // row-major, r = 512, V = 151936: 141 us with four, 114 with eight; on a short
            // one the longer fill of the LDS is not made up: 80 rows, V = 24000, r = 256, 13 %
            // more with eight; V = 65536, 3 % less, at r = 128 13 % more; V = 128000 10 % less)
            if constexpr (VEC) {
                if constexpr (KS >= 8)
                    if (ka.M <= 48) return launch_rows_inst<3, KS, RM, BaseT, PriorT, VEC, HP>(ka, s);
                if constexpr (sizeof(BaseT) == 2)
                    if (ka.M > 64 && ka.V >= (KS >= 8 ? 49152 : 114688))
                        return launch_rows_inst<8, KS, RM, BaseT, PriorT, VEC, HP>(ka, s);
            }
            return launch_rows_inst<4, KS, RM, BaseT, PriorT, VEC, HP>(ka, s);
        };
        auto by_layout = [&](auto ks_tag) -> hipError_t {
            return packed ? by_rows(ks_tag, False{}) : by_rows(ks_tag, True{});
        };
        if (ka.r == 512) return by_layout(std::integral_constant<int, 16>{});
        if (ka.r == 256) return by_layout(std::integral_constant<int, 8>{});
        return by_layout(std::integral_constant<int, 4>{});
    };
    auto by_vec = [&](auto prior_tag, auto has_tag) -> hipError_t {
        return vec ? by_shape(prior_tag, has_tag, True{}) : by_shape(prior_tag, has_tag, False{});
    };
    if (prior_kind == 0) return by_vec(BaseT{}, False{});
    if (prior_kind == 1) return by_vec(float{}, True{});
    return by_vec(BaseT{}, True{});
}

hipError_t launch_rows_f32(const ArgmaxKArgs& ka, bool packed, int prior_kind, bool vec, hipStream_t s);
hipError_t launch_rows_bf16(const ArgmaxKArgs& ka, bool packed, int prior_kind, bool vec, hipStream_t s);
hipError_t launch_rows_f16(const ArgmaxKArgs& ka, bool packed, int prior_kind, bool vec, hipStream_t s);

}  // namespace dels
