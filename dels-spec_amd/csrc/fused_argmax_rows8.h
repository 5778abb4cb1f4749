// The e4m3 form of the kernel that shares each tile of B among several groups
// of 16 rows (fused_argmax_rows.h), for 17 to 64 rows per pass over B.
//
// Semantics as the e4m3 GEMV kernel (fused_argmax_fp8.h): the rank is quantised
// per row in the kernel, dot = fp32(R_q . B_q[v]) * sR[m] * sB[v] (two
// roundings, in that order), then the common combine and argmax; the same MFMA
// steps in the same order, so scores equal that kernel's bit for bit.
//
// Bound by streaming B (half the bytes of bf16) and the base logits.  The
// quantised rank of all rows lies in LDS in operand order (RG * r * 16 bytes:
// 32 KiB for 64 rows at r = 512); a tile is half of the bf16 kernel's registers,
// so three of them per wave are in flight at two waves per SIMD.  The GEMV
// kernel reads B once per 16 rows and keeps the sizes where that costs little
// (rows8_eligible).  r = 512, V = 151936, bf16 base logits: 24 rows 23.8 -> 20.3 us,
// 40 rows 60.5 -> 25.2; V = 32000, 40 rows 20.3 -> 14.8; r = 256, V = 65536, 40 / 63
// rows 16.5 / 18.6 -> 14.4 / 15.0; 200 rows of an unaligned vocabulary of 50257, r =
// 512, 73.0 -> 28.0.  (Above 63
// rows aligned rows go to the tiled kernel: 96 rows 30 us there, 41 in a variant
// of this one with eight groups.)
#pragma once

#include <mutex>

#include "fp8.h"
#include "fused_argmax_rows.h"

namespace dels {

template <int RG, int KS8, typename BaseT, typename PriorT>
struct Rows8Tile {
    i32x8 b[KS8];
    rows::Quad<BaseT> base[RG];
    rows::Quad<PriorT> prior;
    rows::Quad<float> bscale;
};

// HAS_PRIOR false: the prior term is absent (PriorT is then BaseT and unused).
template <int RG, int KS8, typename BaseT, typename PriorT, bool VEC, bool HAS_PRIOR>
__global__ __launch_bounds__(rows::kThreads) void fused_argmax_rows8_kernel(ArgmaxKArgs a) {
#pragma clang fp contract(off)
    using namespace rows;
    constexpr int kRows = 16 * RG;
    // tiles in flight per wave: three where they fit the registers
    constexpr int kND = !VEC && RG == 4 && sizeof(BaseT) == 4 ? 2 : 3;
    extern __shared__ __attribute__((aligned(16))) char s_rank[];   // [KS8][RG][2][64 lanes][16 bytes]
    __shared__ float s_rsc[kRows];
    __shared__ float s_val[kWaves][kRows];
    __shared__ int s_idx[kWaves][kRows];
    __shared__ int s_last;

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // uniform: scalar loop control
    const int col = lane & 15;     // row of the lane within each group
    const int kg = lane >> 4;      // K part of the operands / quad of columns of the results
    const int m0 = blockIdx.y * kRows;

    // Sixteen threads per rank row (RG / 2 rows each), KS8 * 8 consecutive values
    // per thread: their loads go out before the stream's.  Rows past M repeat row 0.
    constexpr int kParts = kRows * 16 / kThreads;
    static_assert(kParts * kThreads == kRows * 16, "whole rows per thread");
    const int seg = threadIdx.x & 15;
    u32x4 rk[kParts][KS8];
#pragma unroll
    for (int i = 0; i < kParts; ++i) {
        const int m = m0 + (int)(threadIdx.x >> 4) + i * (kThreads / 16);
        const uint16_t* p = a.rank + (int64_t)(m < a.M ? m : 0) * a.ldrank + seg * (KS8 * 8);
#pragma unroll
        for (int e = 0; e < KS8; ++e) rk[i][e] = *reinterpret_cast<const u32x4*>(p + 8 * e);
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
    asm volatile("" ::: "memory");   // these loads stay ahead of the stream's

    using Tile = Rows8Tile<RG, KS8, BaseT, PriorT>;
    // live (uniform) false: not one of the wave's tiles -- the same loads, of one line each
    auto load = [&](int t, bool live, Tile& tr) {
        const uint8_t* bp = reinterpret_cast<const uint8_t*>(a.B) + (int64_t)t * KS8 * kFp8K128Block + (live ? lane * 16 : 0);
#pragma unroll
        for (int j = 0; j < KS8; ++j) {
            const u32x4 lo = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(bp + j * kFp8K128Block));
            const u32x4 hi = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(bp + j * kFp8K128Block + 1024));
            tr.b[j] = i32x8{(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3], (int)hi[0], (int)hi[1], (int)hi[2], (int)hi[3]};
        }
        const int v = live ? t * 16 + 4 * kg : 0;
#pragma unroll
        for (int g = 0; g < RG; ++g) load_quad<BaseT, VEC>(a.base, live ? brow[g] : 0, v, a.V, tr.base[g]);
        if constexpr (HAS_PRIOR) load_quad<PriorT, VEC>(a.prior, 0, v, a.V, tr.prior);
        load_quad<float, VEC>(a.b_scale, 0, v, a.V, tr.bscale);
    };
    float rsc[RG];
    auto consume = [&](Tile& tr, int t) {
        // operands tile by tile from LDS (see the bf16 kernel)
        int lo = lane * 16;
        asm volatile("" : "+v"(lo));
        f32x4 acc[RG];
#pragma unroll
        for (int g = 0; g < RG; ++g) acc[g] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < KS8; ++j)
#pragma unroll
            for (int g = 0; g < RG; ++g) {
                const char* p = s_rank + (j * RG + g) * 2048 + lo;
                const u32x4 x = *reinterpret_cast<const u32x4*>(p), y = *reinterpret_cast<const u32x4*>(p + 1024);
                acc[g] = mfma_e4m3_16x16x128(tr.b[j], i32x8{(int)x[0], (int)x[1], (int)x[2], (int)x[3], (int)y[0],
                                                            (int)y[1], (int)y[2], (int)y[3]}, acc[g]);
            }
        const int v = t * 16 + 4 * kg;
        if constexpr (!VEC) {
#pragma unroll
            for (int g = 0; g < RG; ++g) shift_quad<BaseT>(tr.base[g], v, a.V);
            if constexpr (HAS_PRIOR) shift_quad<PriorT>(tr.prior, v, a.V);
            shift_quad<float>(tr.bscale, v, a.V);
        }
#pragma unroll
        for (int q = 3; q >= 0; --q) {
            const bool in = v + q < a.V;
            const float bs = __uint_as_float(tr.bscale[q]);
            float pv = 0.f;
            if constexpr (HAS_PRIOR) pv = quad_at<PriorT>(tr.prior, q);
#pragma unroll
            for (int g = 0; g < RG; ++g) {
                float dot = acc[g][q] * rsc[g];
                dot = dot * bs;
                float sc = __builtin_fmaf(dot, al[g], quad_at<BaseT>(tr.base[g], q));
                if constexpr (HAS_PRIOR) sc = use_prior[g] ? __builtin_fmaf(nbe[g], pv, sc) : sc;
                // a lane's candidates arrive in decreasing column order: ">=" ends at the lowest index,
                // that of a first score of -inf among them
                const bool take = in & (sc >= best[g]);
                best[g] = take ? sc : best[g];
                bidx[g] = take ? v + q : bidx[g];
            }
        }
    };

    // the wave's tiles t, t + nwaves, .. (cnt of them), the last one first, through kND
    // register sets (see the GEMV kernel)
    const int ntiles = (a.V + 15) >> 4;
    const int nwaves = gridDim.x * kWaves;
    const int t = blockIdx.x * kWaves + wave;
    const int cnt = t < ntiles ? (ntiles - 1 - t) / nwaves + 1 : 0;
    const int te = t + (cnt - 1) * nwaves;
    Tile tr[kND];
    // the first ones whether or not the wave has them, so that the waits below are exact
#pragma unroll
    for (int u = 0; u < kND; ++u) load(u < cnt ? te - u * nwaves : 0, u < cnt, tr[u]);

    // the rank rows, quantised by the rule of quantize_rank_coop, into operand
    // order: a thread's bytes are whole 16-byte pieces of one K128 block
#pragma unroll
    for (int i = 0; i < kParts; ++i) {
        const int row = (int)(threadIdx.x >> 4) + i * (kThreads / 16);
        float amax = 0.f;
#pragma unroll
        for (int e = 0; e < KS8; ++e)
#pragma unroll
            for (int h = 0; h < 4; ++h) {
                amax = __builtin_fmaxf(amax, __builtin_fabsf(__uint_as_float(rk[i][e][h] << 16)));
                amax = __builtin_fmaxf(amax, __builtin_fabsf(__uint_as_float(rk[i][e][h] & 0xffff0000u)));
            }
#pragma unroll
        for (int off = 1; off < 16; off <<= 1) amax = __builtin_fmaxf(amax, __shfl_xor(amax, off, 64));
        const float inv = amax > 0.f ? kE4M3Max / amax : 1.f;
#pragma unroll
        for (int e = 0; e < KS8 / 2; ++e) {
            u32x4 w;
#pragma unroll
            for (int h = 0; h < 4; ++h) {
                const uint32_t x0 = rk[i][2 * e + (h >> 1)][2 * (h & 1)], x1 = rk[i][2 * e + (h >> 1)][2 * (h & 1) + 1];
                w[h] = f32x4_to_e4m3(__uint_as_float(x0 << 16) * inv, __uint_as_float(x0 & 0xffff0000u) * inv,
                                     __uint_as_float(x1 << 16) * inv, __uint_as_float(x1 & 0xffff0000u) * inv);
            }
            const int k = seg * (KS8 * 8) + 16 * e, j = k >> 7, kb = k & 127;   // first value, its block, byte in it
            *reinterpret_cast<u32x4*>(s_rank + ((j * RG + (row >> 4)) * 2 + ((kb >> 4) & 1)) * 1024 +
                                      ((row & 15) + 16 * (kb >> 5)) * 16) = w;
        }
        if (seg == 0) s_rsc[row] = amax > 0.f ? amax / kE4M3Max : 1.f;
    }
    lds_barrier();   // the stream's loads stay in flight
#pragma unroll
    for (int g = 0; g < RG; ++g) rsc[g] = s_rsc[16 * g + col];

    int k = 0;
    for (; k + 2 * kND <= cnt; k += kND) {
#pragma unroll
        for (int u = 0; u < kND; ++u) {
            consume(tr[u], te - (k + u) * nwaves);
            load(te - (k + u + kND) * nwaves, true, tr[u]);
        }
    }
#pragma unroll
    for (int u = 0; u < kND; ++u) {
        if (k + u < cnt) consume(tr[u], te - (k + u) * nwaves);
        if (k + u + kND < cnt) load(te - (k + u + kND) * nwaves, true, tr[u]);
    }
#pragma unroll
    for (int u = 0; u < kND; ++u)
        if (k + u + kND < cnt) consume(tr[u], te - (k + u + kND) * nwaves);

    rows_finish<RG>(a, best, bidx, m0, s_val, s_idx, s_last);
}

template <int RG, int KS8, typename BaseT, typename PriorT, bool VEC, bool HAS_PRIOR>
hipError_t launch_rows8_inst(const ArgmaxKArgs& ka, hipStream_t s) {
    const int ntiles = (ka.V + 15) / 16;
    const int groups = (ka.M + 16 * RG - 1) / (16 * RG);
    const int cus = device_cu_count();
    const int gx = std::max(1, std::min((ntiles + rows::kWaves - 1) / rows::kWaves, (cus + groups - 1) / groups));
    constexpr size_t kLds = (size_t)RG * KS8 * 2048;
    static_assert(kLds <= 64 * 1024, "within the dynamic LDS a launch may have without an attribute");
    hipLaunchKernelGGL((fused_argmax_rows8_kernel<RG, KS8, BaseT, PriorT, VEC, HAS_PRIOR>), dim3(gx, groups, 1),
                       dim3(rows::kThreads), kLds, s, ka);
    return hipGetLastError();
}

// Ranks the kernel takes.
inline bool rows8_rank_ok(int r) { return r == 256 || r == 512; }

// Dispatch for one base dtype; `vec` as for the bf16 kernel, with the B scales
// aligned for four-element loads too.
template <typename BaseT>
hipError_t launch_rows8_for_base(const ArgmaxKArgs& ka, int prior_kind, bool vec, hipStream_t s) {
    auto by_rows = [&](auto prior_tag, auto has_tag, auto vec_tag, auto ks_tag) -> hipError_t {
        using PriorT = decltype(prior_tag);
        constexpr bool HP = decltype(has_tag)::value;
        constexpr bool VEC = decltype(vec_tag)::value;
        constexpr int KS8 = decltype(ks_tag)::value;
        if (ka.M <= 32) return launch_rows8_inst<2, KS8, BaseT, PriorT, VEC, HP>(ka, s);
        return launch_rows8_inst<4, KS8, BaseT, PriorT, VEC, HP>(ka, s);
    };
    auto by_shape = [&](auto prior_tag, auto has_tag) -> hipError_t {
        using K2 = std::integral_constant<int, 2>;
        using K4 = std::integral_constant<int, 4>;
        if (vec) return ka.r == 512 ? by_rows(prior_tag, has_tag, std::true_type{}, K4{})
                                    : by_rows(prior_tag, has_tag, std::true_type{}, K2{});
        return ka.r == 512 ? by_rows(prior_tag, has_tag, std::false_type{}, K4{})
                           : by_rows(prior_tag, has_tag, std::false_type{}, K2{});
    };
    if (prior_kind == 0) return by_shape(BaseT{}, std::false_type{});
    if (prior_kind == 1) return by_shape(float{}, std::true_type{});
    return by_shape(BaseT{}, std::true_type{});
}

hipError_t launch_rows8_f32(const ArgmaxKArgs& ka, int prior_kind, bool vec, hipStream_t s);
hipError_t launch_rows8_bf16(const ArgmaxKArgs& ka, int prior_kind, bool vec, hipStream_t s);
hipError_t launch_rows8_f16(const ArgmaxKArgs& ka, int prior_kind, bool vec, hipStream_t s);

}  // namespace dels
