// moe_prefill.h -- what the prefill kernels of both tile widths share: the
// staging of a row as FP16 planes, the tile descriptors and SwiGLU.
#pragma once

#include <utility>

#include "kquant_frag.h"
#include "moe_decode.h"

namespace mqh {

typedef float f32x4 __attribute__((ext_vector_type(4)));

template <int... Ms, class F>
__device__ __forceinline__ void pf_unroll(std::integer_sequence<int, Ms...>, F&& f) {
    (f(std::integral_constant<int, Ms>{}), ...);
}

__device__ __forceinline__ float pf_silu_mul(float g, float u) {
    const float e = __builtin_amdgcn_exp2f(-g * 1.4426950408889634f);
    return (g * __builtin_amdgcn_rcpf(1.0f + e)) * u;
}

__device__ __forceinline__ float pf_wave_max(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
    return v;
}

__device__ __forceinline__ float pf_wave_sum(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// ------------------------------------------------------------ token staging
//
// One wave stages token row `row` of src (K values, FP32 or BF16) as LDS column
// j of the B operand: high plane xh[j][K + PF_PAD], low plane xl (SPLIT only),
// and the 32-column sub-block sums / 32 as [block][j][hi 0..7 | lo 0..7] in xs
// (block-major, so the 16 token columns of one block sit in distinct banks).
// A lane owns 8 consecutive values per 512-column pass.  The loads
// (pf_stage_load) and the rest (pf_stage_finish, or pf_stage_planes into
// device memory) are separate.
template <int K, bool BF16>
struct PfStageRaw {
    static constexpr int NIT = K >= 512 ? K / 512 : 1;
    uint4 r[NIT][BF16 ? 1 : 2];
};

// live = false (a token column past the tile's count): every lane reads the
// row's first values, one request per instruction instead of a row's worth
template <int K, bool BF16>
__device__ __forceinline__ void pf_stage_load(const void* src, int64_t row, bool live, PfStageRaw<K, BF16>& raw) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int it = 0; it < PfStageRaw<K, BF16>::NIT; ++it) {
        // lanes past K (K = 256) read the row's first values again (in bounds, unused)
        const int c = live ? (512 * it + 8 * lane) % K : 0;
        if constexpr (BF16) {
            raw.r[it][0] = *(const uint4*)((const uint16_t*)src + row * K + c);
        } else {
            raw.r[it][0] = *(const uint4*)((const float*)src + row * K + c);
            raw.r[it][1] = *(const uint4*)((const float*)src + row * K + c + 4);
        }
    }
}

// The values of pass `it` (8 per lane) from the loaded words; zero past K
template <int K, bool BF16>
__device__ __forceinline__ void pf_raw_vals(const PfStageRaw<K, BF16>& raw, int it, int c, float v[8]) {
    if constexpr (BF16) {
        const uint32_t w[4] = {raw.r[it][0].x, raw.r[it][0].y, raw.r[it][0].z, raw.r[it][0].w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            v[2 * e] = __uint_as_float(w[e] << 16);
            v[2 * e + 1] = __uint_as_float(w[e] & 0xFFFF0000u);
        }
    } else {
        const uint4 a = raw.r[it][0], b = raw.r[it][1];
        v[0] = __uint_as_float(a.x); v[1] = __uint_as_float(a.y); v[2] = __uint_as_float(a.z); v[3] = __uint_as_float(a.w);
        v[4] = __uint_as_float(b.x); v[5] = __uint_as_float(b.y); v[6] = __uint_as_float(b.z); v[7] = __uint_as_float(b.w);
    }
    if (c >= K) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = 0.0f;
    }
}

// The row's scale exponent k (its max |value| to [2^13, 2^14), frag_exp); with
// gvec set, also x_row . gvec (FP32, unscaled) in every lane, else 0.
template <int K, bool BF16>
__device__ __forceinline__ int pf_row_exp(const PfStageRaw<K, BF16>& raw, const float* gvec, float& gdot_out) {
    constexpr int NIT = PfStageRaw<K, BF16>::NIT;
    const int lane = threadIdx.x & 63;
    float amax = 0.0f, gdot = 0.0f;
#pragma unroll
    for (int it = 0; it < NIT; ++it) {
        const int c = 512 * it + 8 * lane;
        float v[8];
        pf_raw_vals(raw, it, c, v);
#pragma unroll
        for (int e = 0; e < 8; ++e) amax = fmaxf(amax, fabsf(v[e]));
        if (gvec != nullptr && c < K) {
            const float4 g0 = *(const float4*)(gvec + c), g1 = *(const float4*)(gvec + c + 4);
            gdot = fmaf(v[0], g0.x, gdot); gdot = fmaf(v[1], g0.y, gdot);
            gdot = fmaf(v[2], g0.z, gdot); gdot = fmaf(v[3], g0.w, gdot);
            gdot = fmaf(v[4], g1.x, gdot); gdot = fmaf(v[5], g1.y, gdot);
            gdot = fmaf(v[6], g1.z, gdot); gdot = fmaf(v[7], g1.w, gdot);
        }
    }
    gdot_out = pf_wave_sum(gdot);
    return frag_exp(pf_wave_max(amax));
}

// Pass `it` of the row at scale 2^-k: the lane's 8 values as FP16 high and low
// parts, and the sum of its 32-column sub-block (the same in lanes 4m .. 4m+3)
// as an FP16 (high, low) pair.
template <int K, bool BF16>
__device__ __forceinline__ void pf_split_pass(const PfStageRaw<K, BF16>& raw, int it, int k, h8_t& hi, h8_t& lo,
                                              _Float16& sh, _Float16& sl) {
    const int c = 512 * it + 8 * (threadIdx.x & 63);
    float v[8];
    pf_raw_vals(raw, it, c, v);
    float s = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        _Float16 h, l;
        frag_split(v[e], k, h, l);
        hi[e] = h;
        lo[e] = l;
        s += ldexpf(v[e], -k);
    }
    s += __shfl_xor(s, 1, 64);
    s += __shfl_xor(s, 2, 64);
    frag_split(s, 5, sh, sl);
}

// Planes in device memory: [rows x K] FP16 high and low parts at scale 2^-exp,
// the 32-column sums [rows x K / 32] as (high, low) FP16 pairs, exp [rows]
struct PfPlanePtrs {
    uint16_t *hi, *lo;
    uint32_t* sum;
    int* exp;
};

// The same staging of row `t` into planes in device memory (the route pass makes
// the tokens' once per token; every gate/up workgroup of the token's tiles then
// copies them into LDS with no arithmetic).  Returns the row's product with gvec.
template <int K, bool BF16, bool SPLIT>
__device__ __forceinline__ float pf_stage_planes(const PfStageRaw<K, BF16>& raw, int64_t t, const PfPlanePtrs& d,
                                                 const float* gvec) {
    constexpr int NIT = PfStageRaw<K, BF16>::NIT;
    const int lane = threadIdx.x & 63;
    float gdot;
    const int k = pf_row_exp(raw, gvec, gdot);
#pragma unroll
    for (int it = 0; it < NIT; ++it) {
        const int c = 512 * it + 8 * lane;
        h8_t hi, lo;
        _Float16 sh, sl;
        pf_split_pass(raw, it, k, hi, lo, sh, sl);
        if (c < K) {
            *(h8_t*)((_Float16*)d.hi + t * K + c) = hi;
            if constexpr (SPLIT) *(h8_t*)((_Float16*)d.lo + t * K + c) = lo;
            if ((lane & 3) == 0)
                d.sum[t * (K / 32) + (c >> 5)] =
                    (uint32_t)__builtin_bit_cast(uint16_t, sh) | (uint32_t)__builtin_bit_cast(uint16_t, sl) << 16;
        }
    }
    if (lane == 0) d.exp[t] = k;
    return gdot;
}

hipError_t launch_prefill_wide(const PrefillParams& p, hipStream_t s, const KernelEvents& ev);

}  // namespace mqh
