// Temperature sampling of rows of logits: sample() at temperature > 0
// (code/dflash.py:31-38: softmax(logits / T) then torch.multinomial), as a
// Gumbel-max in one pass that never writes probabilities.
//
// For row m and vocabulary index v:
//     y[m, v] = round_T(fp32(x[m, v]) / T)          # logits / temperature, in the logits' dtype
//     u[m, v] = ((bits >> 9) + 0.5) * 2^-23          # in (0, 1), exact in fp32
//     g[m, v] = -log(-log(u[m, v]))                  # standard Gumbel noise
//     id_m    = argmax_v (y[m, v] + g[m, v])         # distributed as softmax(y[m, :])
// where `bits` is word v%4 of Philox4x32-10 (Salmon et al., "Parallel random
// numbers: as easy as 1, 2, 3", SC 2011) at counter (v/4, m, offset_lo,
// offset_hi) and key (seed_lo, seed_hi).  Every element has its own counter,
// so the result depends only on (seed, offset, m, v): any grid, any chunking
// and any later call with the same arguments give the same ids.
//
// What bounds it: vector arithmetic, not memory.  Philox costs ~25 instruction
// slots per element (20 wide multiplies per call at a quarter of the rate, four
// elements per call) and the two logarithms with their argument handling and
// the division about as much again.  The logarithms and the division are only
// taken where they can matter: for each group of four elements the kernel forms
// an upper bound of every candidate -- -log(u) >= 1 - u, so g <= -log(1 - u), one
// hardware log2 of an exact argument, and y <= x / T widened by its rounding --
// and evaluates exactly, as above, only candidates whose bound passes the best
// value the workgroup has seen (kept in LDS).  The bound is tight where u is
// near 1, which is where winners are: a candidate that passes is almost always
// a new maximum.  Everything that is compared or returned is the exact value.
// 120 rows of 151936 bf16 logits, whole call: 65.3 -> 29.3 us, and with one wide
// multiply per Philox product and one bitop3 per pair of xors 26.6, with few
// lanes at the LDS atomics 23 (18.2 M candidates; their 36 MB take 7.3 us at the
// rate of a large copy).
//
// Reduction: one 64-bit key per candidate (order(score) << 32 | ~index, NaN
// above +inf), a device-scope atomic max per workgroup into the row's key, and
// an arrival counter per row; the row's last workgroup decodes its key and
// returns key and counter to zero.  (One counter for the whole grid queued
// every workgroup's arrival on one address, ~12 ns each.)
#include <algorithm>

#include "dels_device.h"
#include "dels_internal.h"

namespace dels {

namespace {

constexpr uint32_t kPhiloxM0 = 0xD2511F53u, kPhiloxM1 = 0xCD9E8D57u;
constexpr uint32_t kPhiloxW0 = 0x9E3779B9u, kPhiloxW1 = 0xBB67AE85u;

__device__ __forceinline__ uint32_t xor3(uint32_t a, uint32_t b, uint32_t c) {
    return __builtin_amdgcn_bitop3_b32(a, b, c, 0x96);   // truth table of a ^ b ^ c
}

// Ten rounds of Philox4x32 on counter c with key (k0, k1).
__device__ __forceinline__ void philox4x32_10(uint32_t (&c)[4], uint32_t k0, uint32_t k1) {
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        // one wide multiply gives both halves of a product, one bitop3 the two xors
        const uint64_t p0 = (uint64_t)kPhiloxM0 * c[0], p1 = (uint64_t)kPhiloxM1 * c[2];
        const uint32_t n0 = xor3((uint32_t)(p1 >> 32), c[1], k0), n2 = xor3((uint32_t)(p0 >> 32), c[3], k1);
        c[0] = n0; c[1] = (uint32_t)p1; c[2] = n2; c[3] = (uint32_t)p0;
        k0 += kPhiloxW0;
        k1 += kPhiloxW1;
    }
}

// Gumbel noise from 32 random bits: u = ((bits >> 9) + 0.5) * 2^-23 lies in
// [2^-24, 1 - 2^-24] and is exact in fp32, so both logarithms are finite.
__device__ __forceinline__ float gumbel_from_bits(uint32_t bits) {
    const float u = ((float)(bits >> 9) + 0.5f) * 0x1p-23f;
    return -logf(-logf(u));
}

// logits / temperature rounded to the logits' dtype, as torch divides a
// bf16/fp16 tensor by a Python float (fp32 arithmetic, one rounding).
__device__ __forceinline__ float tempered(float x, float t, float) { return x / t; }
__device__ __forceinline__ float tempered(float x, float t, bf16_t) { return round_bf16(x / t); }
__device__ __forceinline__ float tempered(float x, float t, f16_t) { return (float)(_Float16)(x / t); }

__device__ __forceinline__ unsigned long long sample_key(float v, uint32_t idx) {
    return pack_argmax(v != v ? __uint_as_float(0x7fc00000u) : v, idx);
}

__device__ __forceinline__ unsigned long long shfl_xor_u64(unsigned long long x, int off) {
    const uint32_t lo = __shfl_xor((uint32_t)x, off, 64);
    const uint32_t hi = __shfl_xor((uint32_t)(x >> 32), off, 64);
    return ((unsigned long long)hi << 32) | lo;
}

// Relative slack of x * (1/T) against tempered(x, T): the rounding to the
// logits' dtype, with room for the fp32 product's own.
template <typename T> constexpr float tempered_slack() { return 0x1p-20f; }
template <> constexpr float tempered_slack<bf16_t>() { return 0x1p-7f; }
template <> constexpr float tempered_slack<f16_t>() { return 0x1p-9f; }

// The value of the lane K below in the DPP row of 16 lanes (0 where there is none).
template <int K>
__device__ __forceinline__ uint32_t row_shr(uint32_t x) {
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0x110 + K, 0xf, 0xf, true);
}

// Four logits as loaded: one 8- or 16-byte load where the rows allow it (VEC),
// else four element loads, clamped to the row.
template <typename T, bool VEC>
__device__ __forceinline__ u32x4 load4_raw(const T* row, int g, int v1) {
    if constexpr (VEC && sizeof(T) == 4) {
        return __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(row + g));
    } else if constexpr (VEC) {
        const u32x2 w = __builtin_nontemporal_load(reinterpret_cast<const u32x2*>(row + g));
        return u32x4{w[0] & 0xffffu, w[0] >> 16, w[1] & 0xffffu, w[1] >> 16};
    } else {
        u32x4 r;
#pragma unroll
        for (int q = 0; q < 4; ++q) r[q] = load_raw(row + min(g + q, v1 - 1));
        return r;
    }
}

constexpr int kSampleThreads = 256;
constexpr int kSampleWGs = 2048;   // workgroups per launch (8 per CU)
constexpr float kLn2 = 0.693147180559945309f;
// Absolute slack of the bounds: the hardware log2 (about 1e-6 at these
// magnitudes) and the rounding of the exact value (its terms are at most 17).
constexpr float kBoundSlack = 1e-4f;

// Grid (chunks, M); a chunk is a multiple of 4 elements, a thread takes groups
// of 4 (one Philox call each).  VEC: V, the chunk and the row stride multiples
// of 4, rows aligned for four-element loads.
template <typename T, bool VEC>
__global__ __launch_bounds__(kSampleThreads) void sample_rows_kernel(
    const T* __restrict__ x, int64_t ldx, int M, int V, int chunk, float temperature, uint32_t k0, uint32_t k1,
    uint32_t off_lo, uint32_t off_hi, unsigned long long* keys, int64_t key_stride, unsigned int* counters,
    int64_t counter_stride, int64_t* out_ids, float* out_score, int64_t ld_out) {
    __shared__ unsigned long long s_key[kSampleThreads / 64];
    __shared__ uint32_t s_thr;        // order key of the best value seen (exact, or a lower bound of one)
    const int m = blockIdx.y;
    const int v0 = blockIdx.x * chunk;
    const int v1 = min(V, v0 + chunk);
    const T* row = x + (int64_t)m * ldx;
    if (threadIdx.x == 0) s_thr = 0u;
    __syncthreads();

    // x * s_a and x * s_b bracket tempered(x, T) (whichever is larger bounds it
    // from above); +inf where a 16-bit quotient may round to infinity
    const float rt = 1.0f / temperature;
    const float s_a = rt * (1.f + tempered_slack<T>()), s_b = rt * (1.f - tempered_slack<T>());
    auto y_upper = [&](float xv) {
        float y = __builtin_fmaxf(xv * s_a, xv * s_b);
        if constexpr (std::is_same<T, f16_t>::value) y = y > 65000.f ? __builtin_inff() : y;
        return xv != xv ? xv : y;   // NaN stays NaN: such a candidate is always evaluated
    };

    unsigned long long best = 0ull;   // below every candidate's key
    // One group per thread: no threshold would serve a later one, so every candidate
    // is evaluated (V = 1000, one row: 6.9 us when they took bounds and a threshold
    // too, 4.6 without).
    const bool bounded = chunk > 4 * kSampleThreads;
    bool first = true;
    int g = v0 + 4 * (int)threadIdx.x;
    u32x4 next = {0u, 0u, 0u, 0u};
    if (g < v1) next = load4_raw<T, VEC>(row, g, v1);
    while (g < v1) {
        const u32x4 raw = next;
        const bool more = v1 - g > 4 * kSampleThreads;
        if (more) next = load4_raw<T, VEC>(row, g + 4 * kSampleThreads, v1);
        uint32_t c[4] = {(uint32_t)g >> 2, (uint32_t)m, off_lo, off_hi};
        philox4x32_10(c, k0, k1);
        float xv[4], lu[4], up[4];    // logits; log2(2^23 (1 - u)), its argument exact; upper bounds
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            xv[q] = widen_raw<T>(raw[q]);
            lu[q] = 0.f;
            up[q] = __builtin_inff();
            if (bounded) {
                lu[q] = __builtin_amdgcn_logf((float)(0x7fffffu - (c[q] >> 9)) + 0.5f);
                up[q] = __builtin_fmaf(lu[q], -kLn2, 23.f * kLn2 + kBoundSlack) + y_upper(xv[q]);
            }
            if constexpr (!VEC) up[q] = g + q < v1 ? up[q] : -__builtin_inff();
        }
        if (first && bounded) {
            // a first threshold: -log(u) <= (1 - u) / u bounds the noise from below
            first = false;
            uint32_t low = 0u;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                float y = __builtin_fminf(xv[q] * s_a, xv[q] * s_b);
                // a float16 quotient may round to -inf (as for y_upper)
                if constexpr (std::is_same<T, f16_t>::value) y = y < -65000.f ? -__builtin_inff() : y;
                const float lo = __builtin_fmaf(__builtin_amdgcn_logf((float)(c[q] >> 9) + 0.5f) - lu[q], kLn2,
                                                y - kBoundSlack);
                const bool use = (xv[q] == xv[q]) & (lo == lo) & (VEC || g + q < v1);
                low = use ? max(low, f32_order_key(lo)) : low;
            }
            // the 16 lanes of each DPP row, then one lane of each: an LDS atomic of all 64
            // lanes costs a round per lane (120 rows of 151936 bf16 logits 27.5 us, 23.7 so).
            // A row whose last lane has no group adds nothing: a lower threshold.
            low = max(low, row_shr<1>(low));
            low = max(low, row_shr<2>(low));
            low = max(low, row_shr<4>(low));
            low = max(low, row_shr<8>(low));
            if ((threadIdx.x & 15) == 15) atomicMax(&s_thr, low);
        }
        // candidates at or below the threshold cannot win (their exact value is
        // below their bound); it stays under +inf, so that equal infinities are
        // all evaluated and the lowest index wins
        const uint32_t tk = *(volatile uint32_t*)&s_thr;
        const float thr = tk == 0u ? -__builtin_inff() : __builtin_fminf(f32_from_order_key(tk), 3.402823466e38f);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if (!(up[q] <= thr)) {
                const float val = tempered(xv[q], temperature, T{}) + gumbel_from_bits(c[q]);
                const unsigned long long k = sample_key(val, (uint32_t)(g + q));
                // -inf is no candidate: not every such element is evaluated, and a row of
                // nothing else gives id 0 without one
                best = val != -__builtin_inff() && k > best ? k : best;
                if (bounded && val == val) atomicMax(&s_thr, f32_order_key(val));
            }
        }
        if (!more) break;
        g += 4 * kSampleThreads;
    }
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const unsigned long long o = shfl_xor_u64(best, off);
        best = o > best ? o : best;
    }
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) s_key[wave] = best;
    __syncthreads();
    if (threadIdx.x != 0) return;
    unsigned long long seen = 0;
    for (int w = 1; w < kSampleThreads / 64; ++w) best = s_key[w] > best ? s_key[w] : best;
    unsigned long long* key = keys + (int64_t)m * key_stride;
    unsigned int* counter = counters + (int64_t)m * counter_stride;
    if (best != 0ull) seen = __hip_atomic_fetch_max(key, best, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    // the returned value orders the count after the update
    const unsigned prev = __hip_atomic_fetch_add(counter, seen == ~0ull ? 2u : 1u, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT);
    if (prev != gridDim.x - 1) return;
    const unsigned long long k = __hip_atomic_exchange(key, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_exchange(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    uint32_t idx = ~(uint32_t)(k & 0xffffffffull);
    float val = f32_from_order_key((uint32_t)(k >> 32));
    if (k == 0ull || idx >= (uint32_t)V) {   // no candidate (every logit -inf)
        idx = 0;
        val = -__builtin_inff();
    }
    out_ids[(int64_t)m * ld_out] = (int64_t)idx;
    if (out_score) out_score[(int64_t)m * ld_out] = val;
}

}  // namespace

hipError_t launch_sample_rows(const void* x, int64_t ldx, int dtype, int M, int V, float temperature, uint64_t seed,
                              uint64_t offset, int64_t* out_ids, float* out_score, int64_t ld_out, void* ws,
                              hipStream_t s) {
    char* w = static_cast<char*>(ws);
    auto* counters = reinterpret_cast<unsigned int*>(w + kCountersOff);
    auto* keys = reinterpret_cast<unsigned long long*>(w + kKeysOff);
    const int64_t key_stride = (int64_t)M * 128 <= (int64_t)(kCtrlBytes - kKeysOff) ? 16 : 1;
    // a 128-byte line per row's counter while they fit below the line that persists, else packed
    const int64_t counter_stride = (int64_t)M * 32 <= kMaxCounters ? 32 : 1;
    // Chunks per row: about kSampleWGs workgroups in all, so that a workgroup's
    // threshold serves many groups, and at least one group per thread (M = 1
    // then runs V / 1024 workgroups).
    const int gx_max = std::max(1, (V + 4 * kSampleThreads - 1) / (4 * kSampleThreads));
    const int gx = std::max(1, std::min(gx_max, kSampleWGs / std::max(M, 1)));
    const int chunk = ((V + gx - 1) / gx + 3) & ~3;
    const dim3 grid((V + chunk - 1) / chunk, M);
    const uint32_t k0 = (uint32_t)seed, k1 = (uint32_t)(seed >> 32);
    const uint32_t o0 = (uint32_t)offset, o1 = (uint32_t)(offset >> 32);
    const size_t quad = dtype == 0 ? 16 : 8;   // bytes of four logits
    const bool vec = reinterpret_cast<uintptr_t>(x) % quad == 0 && ldx % 4 == 0 && V % 4 == 0;
    auto go = [&](auto tag, auto vec_tag) {
        using T = decltype(tag);
        hipLaunchKernelGGL((sample_rows_kernel<T, decltype(vec_tag)::value>), grid, dim3(kSampleThreads), 0, s,
                           static_cast<const T*>(x), ldx, M, V, chunk, temperature, k0, k1, o0, o1, keys, key_stride,
                           counters, counter_stride, out_ids, out_score, ld_out);
    };
    auto by_vec = [&](auto tag) {
        if (vec) go(tag, std::integral_constant<bool, true>{});
        else go(tag, std::integral_constant<bool, false>{});
    };
    if (dtype == 1) by_vec(bf16_t{});
    else if (dtype == 2) by_vec(f16_t{});
    else by_vec(float{});
    return hipGetLastError();
}

}  // namespace dels
