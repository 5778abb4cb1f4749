// Domino correction step: f(z + s) . fc2^T (+ fc2 bias), scaled by the
// guidance alpha, plus the base logits, then the vocabulary argmax -- the
// fused kernel of the Domino runner (code/kernel/domino.py:58-173: its
// _fused_mlp_bias_argmax_kernel and _reduce_argmax_kernel in one launch; f is
// SiLU there, and any of the middle layers of DELS_MIDDLE_* here, which the
// reference runs as its unfused step, 404-431).
//
// For row m (< 16 per row group) and vocabulary index v:
//     mid[m, k] = f(p),  p = fp32(z[m, k]) + fp32(s[m, k])                (fp32, never rounded)
//                 (SiLU: p * sigmoid(p))
//     dot[m, v] = sum_k fp32(fc2[v, k]) * mid[m, k]                       (fp32 accumulate)
//     score     = fma(dot (+ bias[v]), alpha, base[m, v])
// and per row the lowest v attaining the maximum.
//
// mid stays fp32 in the reference, but the matrix cores take bf16 operands,
// so each value is split into two bf16 parts, hi = bf16(mid) and
// lo = bf16(mid - hi) (|mid - hi - lo| <= 2^-17 |mid|), and every K step runs
// two v_mfma_f32_16x16x32_bf16 on the same fc2 operand: the products are exact
// in fp32, so the dot is that of mid to within 2^-17 relative per term -- well
// inside the fp32 accumulation-order freedom the reference already has.
//
// One workgroup of eight waves per CU builds the hi/lo operands of its 16 rows
// in LDS (64 * E bytes, E <= 2048; rows past M are zero), then its waves stream
// 16-row tiles of fc2 (MFMA-16 block layout, one contiguous KiB per K step)
// through two register sets of up to 16 K steps, walking (tile, K chunk) units
// so any E streams with the same register budget.  The cross-workgroup argmax
// is that of the other kernels (row keys and an arrival counter).
//
// Bound by streaming fc2 from HBM (311 MB at E = 1024, V = 151936), so the
// stream must not start late or end in a queue: a workgroup's loads of z and s
// go out first (a CU returns its loads in order), then the first two units of
// every wave, and the operands are computed while those travel.  One row at
// E = 1024, V = 151936: 65.9 -> about 54 us a launch (5.8 TB/s), the 14-step
// rollout 1071 -> 905 us, with no waits on loads inside the stream either (see
// EXACT) and one operand build and one arrival per CU instead of two.
#include <algorithm>
#include <climits>
#include <mutex>

#include "../../include/dels.h"
#include "dels_device.h"
#include "dels_internal.h"
#include "fused_argmax_gemv.h"

namespace dels {

namespace {

constexpr int kDomKC = 16;   // K steps (of 32) per register set

// The middle layer f of the correction MLP in fp32 (DELS_MIDDLE_*; `middle` is
// uniform over the launch).  GELU is x/2 (1 + erf(x / sqrt 2)) and its tanh
// form x/2 (1 + tanh(sqrt(2/pi) (x + 0.044715 x^3))), as nn.GELU defines them.
template <int MIDDLE>
__device__ __forceinline__ float domino_middle(float p) {
#pragma clang fp contract(off)
    if constexpr (MIDDLE == DELS_MIDDLE_IDENTITY) return p;
    else if constexpr (MIDDLE == DELS_MIDDLE_RELU) return p > 0.f ? p : (p == p ? 0.f : p);
    else if constexpr (MIDDLE == DELS_MIDDLE_GELU) return 0.5f * p * (1.f + erff(p * 0.70710678118654752f));
    else if constexpr (MIDDLE == DELS_MIDDLE_GELU_TANH)
        return 0.5f * p * (1.f + tanhf(0.79788456080286536f * (p + 0.044715f * (p * p * p))));
    else if constexpr (MIDDLE == DELS_MIDDLE_TANH) return tanhf(p);
    else if constexpr (MIDDLE == DELS_MIDDLE_SIGMOID) return sigmoid_f32(p);
    else return p * sigmoid_f32(p);   // DELS_MIDDLE_SILU
}

constexpr int kDomWaves = 8;
constexpr int kDomThreads = kDomWaves * 64;
// Pieces of eight values of one row that a thread turns into operands; those
// of E <= 1024 are held in registers while the first units are put in flight.
constexpr int kDomPieces = 16 * 1024 / 8 / kDomThreads;

// Eight values of z and s as loaded.
struct DomPiece {
    u32x4 z, s;
};

// z and s rows need no more than their elements' alignment: the copy states
// that, and the compiler picks loads that are legal at it.
__device__ __forceinline__ u32x4 load_eight(const uint16_t* p) {
    u32x4 r;
    __builtin_memcpy(&r, p, sizeof(r));
    return r;
}

// Piece i: row i / (kpad / 8) of the 16, values k .. k + 7.  Rows past M and the
// K padding are zero.
__device__ __forceinline__ bool domino_piece_at(const DominoArgs& a, int m0, int kpad, int i, int& row, int& k) {
    row = i / (kpad / 8);
    k = (i - row * (kpad / 8)) * 8;
    return m0 + row < a.M && k < a.E;
}
__device__ __forceinline__ void domino_load_piece(const DominoArgs& a, int m0, int kpad, int i, DomPiece& p) {
    int row, k;
    const bool live = i < 2 * kpad && domino_piece_at(a, m0, kpad, i, row, k);
    // a piece without values loads the first row's first eight (in bounds) and is not used
    const int64_t m = live ? m0 + row : m0;
    p.z = load_eight(a.z + m * a.ldz + (live ? k : 0));
    p.s = load_eight(a.s + m * a.lds + (live ? k : 0));
}

// mid = f(z + s) of a piece into the hi/lo operand layout in LDS (see the kernel).
template <int MIDDLE>
__device__ __forceinline__ void domino_store_piece(const DominoArgs& a, int m0, int kpad, int i, const DomPiece& p,
                                                   uint16_t* ops) {
#pragma clang fp contract(off)
    if (i >= 2 * kpad) return;
    int row, k;
    const bool live = domino_piece_at(a, m0, kpad, i, row, k);
    u32x4 hi = {0u, 0u, 0u, 0u}, lo = {0u, 0u, 0u, 0u};
    if (live) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int sh = 16 * (e & 1);
            const float mid = domino_middle<MIDDLE>(bf16_bits_to_f32((p.z[e >> 1] >> sh) & 0xffffu) +
                                                    bf16_bits_to_f32((p.s[e >> 1] >> sh) & 0xffffu));
            const uint32_t h = f32_to_bf16_bits(mid);
            hi[e >> 1] |= h << sh;
            lo[e >> 1] |= (uint32_t)f32_to_bf16_bits(mid - bf16_bits_to_f32(h)) << sh;
        }
    }
    const int ks = k >> 5, ln = row + 16 * ((k & 31) >> 3);
    *reinterpret_cast<u32x4*>(&ops[((ks * 2 + 0) * 64 + ln) * 8]) = hi;
    *reinterpret_cast<u32x4*>(&ops[((ks * 2 + 1) * 64 + ln) * 8]) = lo;
}

// All pieces of the workgroup: the first kDomPieces per thread from registers,
// the rest (E > 1024) loaded here.  One instance per middle layer, so none
// carries a branch on it.
template <int MIDDLE>
__device__ __forceinline__ void domino_fill_operands(const DominoArgs& a, int m0, int kpad, const DomPiece (&pc)[kDomPieces], uint16_t* ops) {
#pragma unroll
    for (int j = 0; j < kDomPieces; ++j)
        domino_store_piece<MIDDLE>(a, m0, kpad, (int)threadIdx.x + kDomThreads * j, pc[j], ops);
    for (int i = threadIdx.x + kDomThreads * kDomPieces; i < 2 * kpad; i += kDomThreads) {
        DomPiece p;
        domino_load_piece(a, m0, kpad, i, p);
        domino_store_piece<MIDDLE>(a, m0, kpad, i, p, ops);
    }
}

template <typename BaseT, typename BiasT>
struct DomRegs {
    bf16x8 b[kDomKC];
    uint32_t base[4];   // as loaded (load_raw), widened at use
    uint32_t bias;
};

// EXACT: E is a whole number of register sets (a multiple of 512), so no operand
// of fc2 is masked: a mask applied to a load would wait for it right there, and
// the unit that is contracted meanwhile would be the only one in flight.
template <typename BaseT, typename BiasT, bool EXACT>
__global__ __launch_bounds__(kDomThreads) void domino_argmax_kernel(DominoArgs a, ArgmaxKArgs fin) {
#pragma clang fp contract(off)
    extern __shared__ __attribute__((aligned(16))) char dyn_lds[];   // [ksteps][2][64 lanes][16 bytes]
    __shared__ float s_val[kDomWaves][16];
    __shared__ int s_idx[kDomWaves][16];
    __shared__ int s_last;

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane & 15;
    const int kg = lane >> 4;
    const int m0 = blockIdx.y * 16;
    const int ksteps = a.E / 32;

    // mid = f(z + s) of the 16 rows, split into bf16 hi/lo A operands: K step
    // ks, part p (0 hi, 1 lo) is the KiB at ((ks * 2 + p) * 64 + lane) * 16 with
    // lane = row + 16 * (k % 32 / 8), element k % 8.  K is padded with zeros to
    // whole register sets (and rows past M are zero), so the contraction below
    // runs every step of a set unconditionally: padded steps multiply zeros.
    uint16_t* ops = reinterpret_cast<uint16_t*>(dyn_lds);
    const int kpad = ((ksteps + kDomKC - 1) / kDomKC) * kDomKC * 32;
    DomPiece pc[kDomPieces];
#pragma unroll
    for (int j = 0; j < kDomPieces; ++j)
        domino_load_piece(a, m0, kpad, (int)threadIdx.x + kDomThreads * j, pc[j]);
    asm volatile("" ::: "memory");   // these loads stay ahead of the stream's

    float al[4], best[4];
    int bidx[4];
    const BaseT* brow[4];
    const BaseT* base = static_cast<const BaseT*>(a.base);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int m = m0 + 4 * kg + q;
        const bool mok = m < a.M;
        al[q] = a.alpha;
        brow[q] = base + (int64_t)(mok ? m : 0) * a.ldbase;
        best[q] = -__builtin_inff();
        bidx[q] = INT_MAX;
    }

    const int ntiles = (a.V + 15) >> 4;
    const int nch = (ksteps + kDomKC - 1) / kDomKC;
    const int nwaves = gridDim.x * kDomWaves;
    const int t0 = blockIdx.x * kDomWaves + wave;
    const int cnt = t0 < ntiles ? (ntiles - 1 - t0) / nwaves + 1 : 0;
    const int units = cnt * nch;
    const BiasT* bias = static_cast<const BiasT*>(a.bias);

    auto load_unit = [&](int u, DomRegs<BaseT, BiasT>& tr) {
        // the first two units are loaded whether or not the wave has them (the last tile again)
        const int t = min(t0 + (u / nch) * nwaves, ntiles - 1);
        const int c = u % nch;
        const int v = t * 16 + col;
        const int vc = v < a.V ? v : a.V - 1;
        const uint16_t* bp = a.W + ((int64_t)t * ksteps + c * kDomKC) * 512 + lane * 8;
#pragma unroll
        for (int i = 0; i < kDomKC; ++i) {
            if constexpr (EXACT) {
                tr.b[i] = load_bf16x8_nt(bp + i * 512);
                continue;
            }
            const bool ok = c * kDomKC + i < ksteps;
            tr.b[i] = masked_bf16x8(__builtin_nontemporal_load(reinterpret_cast<const u32x4*>(bp + (ok ? i : 0) * 512)),
                                    ok ? 0xffffffffu : 0u);
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) tr.base[q] = load_raw(brow[q] + vc);
        if constexpr (!is_no_prior<BiasT>::value) tr.bias = load_raw(bias + vc);
        else tr.bias = 0u;
    };
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    auto consume = [&](const DomRegs<BaseT, BiasT>& tr, int u) {
        const int t = t0 + (u / nch) * nwaves;
        const int c = u % nch;
        const char* ap = dyn_lds + (size_t)(c * kDomKC) * 2048 + lane * 16;
#pragma unroll
        for (int i = 0; i < kDomKC; ++i) {
            const bf16x8 hi = *reinterpret_cast<const bf16x8*>(ap + i * 2048);
            const bf16x8 lo = *reinterpret_cast<const bf16x8*>(ap + i * 2048 + 1024);
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(hi, tr.b[i], acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(lo, tr.b[i], acc, 0, 0, 0);
        }
        if (c == nch - 1) {
            const int v = t * 16 + col;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                float dot = acc[q];
                if constexpr (!is_no_prior<BiasT>::value) dot = dot + widen_raw<BiasT>(tr.bias);
                const float sc = __builtin_fmaf(dot, al[q], widen_raw<BaseT>(tr.base[q]));
                const bool take = (v < a.V) & argmax_better(sc, v, best[q], bidx[q]);
                best[q] = take ? sc : best[q];
                bidx[q] = take ? v : bidx[q];
            }
            acc = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    };
    // two register sets, refills unconditional inside the loop, the tail peeled
    DomRegs<BaseT, BiasT> tr0, tr1;
    load_unit(0, tr0);
    load_unit(1, tr1);
    switch (a.middle) {   // uniform
        case DELS_MIDDLE_IDENTITY: domino_fill_operands<DELS_MIDDLE_IDENTITY>(a, m0, kpad, pc, ops); break;
        case DELS_MIDDLE_RELU: domino_fill_operands<DELS_MIDDLE_RELU>(a, m0, kpad, pc, ops); break;
        case DELS_MIDDLE_GELU: domino_fill_operands<DELS_MIDDLE_GELU>(a, m0, kpad, pc, ops); break;
        case DELS_MIDDLE_GELU_TANH: domino_fill_operands<DELS_MIDDLE_GELU_TANH>(a, m0, kpad, pc, ops); break;
        case DELS_MIDDLE_TANH: domino_fill_operands<DELS_MIDDLE_TANH>(a, m0, kpad, pc, ops); break;
        case DELS_MIDDLE_SIGMOID: domino_fill_operands<DELS_MIDDLE_SIGMOID>(a, m0, kpad, pc, ops); break;
        default: domino_fill_operands<DELS_MIDDLE_SILU>(a, m0, kpad, pc, ops); break;
    }
    lds_barrier();   // the operands; the stream's loads stay in flight
    int u = 0;
    for (; u + 4 <= units; u += 2) {
        consume(tr0, u);
        load_unit(u + 2, tr0);
        consume(tr1, u + 1);
        load_unit(u + 3, tr1);
    }
    if (u < units) consume(tr0, u);
    if (u + 2 < units) load_unit(u + 2, tr0);
    if (u + 1 < units) consume(tr1, u + 1);
    if (u + 2 < units) consume(tr0, u + 2);

    argmax_wg_finish<kDomWaves>(fin, best, bidx, m0, s_val, s_idx, s_last, nullptr);
}

template <typename BaseT, typename BiasT, bool EXACT>
hipError_t launch_domino_inst(const DominoArgs& a, const ArgmaxKArgs& fin, int gx, int gy, size_t lds, hipStream_t s) {
    // the operands of E = 2048 take 128 KiB of dynamic LDS: allow it once per kernel instance (the
    // attribute belongs to the function, not to a device); call_once makes concurrent first launches
    // from several host threads safe, and every caller sees the call's result
    static std::once_flag once;
    static hipError_t attr_err = hipSuccess;
    std::call_once(once, [] {
        attr_err = hipFuncSetAttribute(reinterpret_cast<const void*>(&domino_argmax_kernel<BaseT, BiasT, EXACT>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)domino_lds_bytes(kDominoMaxE));
    });
    if (attr_err != hipSuccess) return attr_err;
    hipLaunchKernelGGL((domino_argmax_kernel<BaseT, BiasT, EXACT>), dim3(gx, gy, 1), dim3(kDomThreads), lds, s, a, fin);
    return hipGetLastError();
}

template <typename BaseT>
hipError_t launch_domino_for_base(const DominoArgs& a, const ArgmaxKArgs& fin, int gx, int gy, size_t lds,
                                  hipStream_t s) {
    auto by_bias = [&](auto exact_tag) -> hipError_t {
        constexpr bool EXACT = decltype(exact_tag)::value;
        if (a.bias == nullptr) return launch_domino_inst<BaseT, no_prior_t, EXACT>(a, fin, gx, gy, lds, s);
        if (a.bias_dtype == 1) return launch_domino_inst<BaseT, bf16_t, EXACT>(a, fin, gx, gy, lds, s);
        if (a.bias_dtype == 2) return launch_domino_inst<BaseT, f16_t, EXACT>(a, fin, gx, gy, lds, s);
        return launch_domino_inst<BaseT, float, EXACT>(a, fin, gx, gy, lds, s);
    };
    return a.E % (32 * kDomKC) == 0 ? by_bias(std::true_type{}) : by_bias(std::false_type{});
}

}  // namespace

size_t domino_lds_bytes(int64_t E) {
    const int64_t ksteps = (E + 31) / 32;
    return (size_t)((ksteps + kDomKC - 1) / kDomKC) * kDomKC * 2048;
}

bool domino_supported(int64_t M, int64_t E, int64_t V) {
    return M >= 1 && M <= kMaxKeyRows && E >= 32 && E <= kDominoMaxE && E % 32 == 0 && V >= 1;
}

hipError_t launch_domino_argmax(const DominoArgs& a, void* ws, hipStream_t s) {
    char* w = static_cast<char*>(ws);
    ArgmaxKArgs fin{};
    fin.M = a.M; fin.V = a.V;
    fin.out_ids = a.out_ids; fin.out_score = a.out_score; fin.ld_out = a.ld_out;
    fin.counter = reinterpret_cast<unsigned int*>(w + kCountersOff);
    fin.keys = reinterpret_cast<unsigned long long*>(w + kKeysOff);
    fin.key_stride = (int64_t)a.M * 128 <= (int64_t)(kCtrlBytes - kKeysOff) ? 16 : 1;
    const int ntiles = (a.V + 15) / 16;
    const int groups = (a.M + 15) / 16;
    const size_t lds = domino_lds_bytes(a.E);
    const int gx = std::max(1, std::min((ntiles + kDomWaves - 1) / kDomWaves, (device_cu_count() + groups - 1) / groups));
    if (a.base_dtype == 1) return launch_domino_for_base<bf16_t>(a, fin, gx, groups, lds, s);
    if (a.base_dtype == 2) return launch_domino_for_base<f16_t>(a, fin, gx, groups, lds, s);
    return launch_domino_for_base<float>(a, fin, gx, groups, lds, s);
}

}  // namespace dels
