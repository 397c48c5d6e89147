// router.hip -- top-k expert routing on the GPU (ExpertRouter.route).
//
// Replaces src/flash_moe/router.py:140-170 for tokens already in HBM, so a
// decode step needs no host round trip between the router and the experts:
//   scores = x . W       FP32; W is the layer's ffn_gate_inp as the GGUF file
//                        stores it, n_experts rows of hidden floats (the
//                        reference keeps its transpose, router.py:39-59,101-135)
//   ids    = top-k of scores in descending order (argsort, last k, reversed)
//   w      = float64 softmax over the selected scores, then FP32 (the combine
//            multiplies by fl32(w), moe_layer.py:70,85-86); a non-finite or
//            non-positive exponential sum gives 1/k each (router.py:161-166).
//
// Two launches.  k_route_scores: each workgroup owns 4/SPLIT experts and a group
// of tokens; SPLIT waves share one expert row, each summing a contiguous share of
// the hidden dimension with 16-byte loads (a lane's chain, then a fixed DPP tree
// over the wave), and the shares are added in wave order, so the summation order
// of a score is fixed for a given SPLIT.  k_route_scores_mfma, for more scores
// than that kernel makes in one round of the chip (route_on_matrix): the same
// FP32 products and sums as a matrix product on the FP32 matrix instructions,
// also in a fixed order.
// k_route_select: one wavefront per token takes the top k by k rounds of a
// wave maximum over (score, expert) keys (route_topk.h): NaN ranks above every
// number, as np.argsort places NaN last (a NaN among the selected then makes
// the softmax sum NaN and the weights uniform, as in the reference); equal
// scores, and NaNs among themselves, are taken in ascending expert order
// (NumPy's order for ties is unspecified); -0.0 and +0.0 count as equal.
// The routed decode runs the select step inside its gate/up kernel instead
// (moe_fast.hip) when the experts number at most 256.

#include <hip/hip_runtime.h>

#include <cstdint>

#include "moe_decode.h"
#include "route_topk.h"

namespace mqh {

constexpr int RS_WAVES = 4;    // waves per scores workgroup
constexpr int SEL_WAVES = 4;   // tokens per select workgroup, one wave each

template <int CTRL, int ROW_MASK>
__device__ __forceinline__ float dpp_f32(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(v), __float_as_int(v), CTRL, ROW_MASK, 0xF, false));
}

// Sum over the wavefront in a fixed order (quads, half rows, rows, then
// (row3 + row2) + (row1 + row0)); the total lands in lane 63.
__device__ __forceinline__ float wave_sum_to_lane63(float v) {
    v += dpp_f32<0xB1, 0xF>(v);    // quad_perm [1,0,3,2]
    v += dpp_f32<0x4E, 0xF>(v);    // quad_perm [2,3,0,1]
    v += dpp_f32<0x141, 0xF>(v);   // row_half_mirror
    v += dpp_f32<0x140, 0xF>(v);   // row_mirror
    const float a = dpp_f32<0x142, 0xA>(v);   // row_bcast:15 into rows 1 and 3
    v = (threadIdx.x & 16) ? v + a : v;
    const float b = dpp_f32<0x143, 0xC>(v);   // row_bcast:31 into rows 2 and 3
    return (threadIdx.x & 32) ? v + b : v;
}

template <int SPLIT, int TT>
__global__ __launch_bounds__(64 * RS_WAVES) void k_route_scores(const float* __restrict__ x, int n_tokens, int hidden,
                                                                const float* __restrict__ w, int n_experts,
                                                                float* __restrict__ scores) {
    constexpr int EPG = RS_WAVES / SPLIT;   // experts per workgroup
    __shared__ float part[RS_WAVES][TT];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int e = blockIdx.x * EPG + wave / SPLIT, piece = wave % SPLIT;
    const int t0 = blockIdx.y * TT, nt = min(TT, n_tokens - t0);
    const int n4 = hidden >> 2;
    const int per = (n4 + SPLIT - 1) / SPLIT;
    const int j0 = piece * per, j1 = min(n4, j0 + per);

    float acc[TT];
#pragma unroll
    for (int t = 0; t < TT; ++t) acc[t] = 0.0f;
    if (e < n_experts) {
        const float4* wr = reinterpret_cast<const float4*>(w + (int64_t)e * hidden);
        const float4* xr = reinterpret_cast<const float4*>(x + (int64_t)t0 * hidden);
        // two 16-byte columns per lane per pass, both loads issued before
        // either is used; a second column past j1 re-reads the first's and is
        // not accumulated
        for (int j = j0 + lane; j < j1; j += 128) {
            const int j2 = j + 64 < j1 ? j + 64 : j;
            const float4 wv = wr[j], wv2 = wr[j2];
            float4 xv[TT], xv2[TT];
#pragma unroll
            for (int t = 0; t < TT; ++t) {
                const int64_t row = (int64_t)min(t, nt - 1) * n4;   // rows past nt repeat the last
                xv[t] = xr[row + j];
                xv2[t] = xr[row + j2];
            }
#pragma unroll
            for (int t = 0; t < TT; ++t)
                acc[t] = fmaf(xv[t].w, wv.w, fmaf(xv[t].z, wv.z, fmaf(xv[t].y, wv.y, fmaf(xv[t].x, wv.x, acc[t]))));
            if (j + 64 < j1) {
#pragma unroll
                for (int t = 0; t < TT; ++t)
                    acc[t] = fmaf(xv2[t].w, wv2.w,
                                  fmaf(xv2[t].z, wv2.z, fmaf(xv2[t].y, wv2.y, fmaf(xv2[t].x, wv2.x, acc[t]))));
            }
        }
    }
#pragma unroll
    for (int t = 0; t < TT; ++t) {
        const float v = wave_sum_to_lane63(acc[t]);
        if (lane == 63) part[wave][t] = v;
    }
    __syncthreads();
    const int le = threadIdx.x / TT, t = threadIdx.x % TT;
    const int oe = blockIdx.x * EPG + le;
    if (le < EPG && t < nt && oe < n_experts) {
        float s = part[le * SPLIT][t];
#pragma unroll
        for (int p = 1; p < SPLIT; ++p) s += part[le * SPLIT + p][t];
        scores[(int64_t)(t0 + t) * n_experts + oe] = s;
    }
}

// Scores of many tokens on v_mfma_f32_32x32x2_f32 (FP32 in, FP32 sums).  A
// workgroup owns 32 TB tokens x 32 experts; its sixteen waves share the hidden
// dimension, each a contiguous slice of a multiple of 32 columns, and read their
// operands straight into registers: the instruction takes row l % 32 of both
// operands at column l / 32, so with the columns of a group of eight dealt as
// 0..3 to the low and 4..7 to the high half of the wave (the same for both
// operands) a lane's 16-byte load feeds four instructions.  No LDS staging and
// no barrier before the waves' partial tiles are added.
//
// Summation order: chains of CH columns, joined as a tree over each 32 (TB = 1) or
// added in turn, then the sixteen waves' sums as a tree.  The vector kernel's
// chains are H / 64 columns under six tree levels.  CH = 16 from H = 1536 on and
// 8 from 512 on is no less accurate (relative error against 64 bits at 512 tokens
// x 256 experts, vector and matrix kernel: 1.23e-7 and 1.04e-7 at H = 2048,
// 1.00e-7 and 0.90e-7 at 1024, 0.86e-7 both at 512); below 512 the vector
// kernel's chains are shorter still (0.78e-7 and 0.81e-7 at 256) and it stays.
// Bound by the FP32 matrix rate (2 T E H operations, 14 us for 2048 x 256 scores
// of 2048 columns) and, below some 256 tiles, by one workgroup's own chain (17 us
// there).  That size: 133 -> 34 us; 512 x 256 x 2048: 37.6 -> 17.2 us.
typedef float f32x16 __attribute__((ext_vector_type(16)));
constexpr int RM_WAVES = 16;
constexpr int RM_STEP = 32;   // columns of a pass

// Columns C0 .. C0 + N - 1 of a pass (in the order the lanes hold them): chains
// of CH, joined as a tree.  MFMA c of group s takes columns 8 s + c and 8 s + 4 + c.
template <int C0, int N, int CH>
__device__ __forceinline__ f32x16 rm_tree(const float4 (&av)[RM_STEP / 8], const float4 (&bv)[RM_STEP / 8]) {
    if constexpr (N > CH) {
        const f32x16 l = rm_tree<C0, N / 2, CH>(av, bv);
        return l + rm_tree<C0 + N / 2, N / 2, CH>(av, bv);
    } else {
        f32x16 p;
#pragma unroll
        for (int i = 0; i < 16; ++i) p[i] = 0.0f;
#pragma unroll
        for (int c = C0; c < C0 + N; c += 2)
            p = __builtin_amdgcn_mfma_f32_32x32x2f32(((const float*)&av[c / 8])[c % 8 / 2],
                                                     ((const float*)&bv[c / 8])[c % 8 / 2], p, 0, 0, 0);
        return p;
    }
}

template <int TB, int CH>
__global__ __launch_bounds__(64 * RM_WAVES) void k_route_scores_mfma(const float* __restrict__ x, int n_tokens,
                                                                     int hidden, const float* __restrict__ w,
                                                                     int n_experts, float* __restrict__ scores,
                                                                     int per, int n_etiles) {
    __shared__ float part[RM_WAVES][TB][32][32];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, half = lane >> 5, l32 = lane & 31;
    // workgroup i runs on XCD i % 8: the expert tiles of one token tile have
    // indices that agree mod 8, so its rows are read into one XCD's L2
    const int j = blockIdx.x / 8;
    const int et = j % n_etiles, tt = (j / n_etiles) * 8 + blockIdx.x % 8;
    const int t0 = tt * 32 * TB, e0 = et * 32;
    if (t0 >= n_tokens) return;
    // rows past the last repeat it and are not stored
    const float* wr = w + (int64_t)min(e0 + l32, n_experts - 1) * hidden + 4 * half;
    const float* xr[TB];
#pragma unroll
    for (int b = 0; b < TB; ++b) xr[b] = x + (int64_t)min(t0 + 32 * b + l32, n_tokens - 1) * hidden + 4 * half;

    f32x16 acc[TB];
#pragma unroll
    for (int b = 0; b < TB; ++b)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[b][i] = 0.0f;
    const int k1 = min(hidden, (wave + 1) * per);
    for (int k = wave * per; k < k1; k += RM_STEP) {
        float4 bv[RM_STEP / 8], av[TB][RM_STEP / 8];
#pragma unroll
        for (int s = 0; s < RM_STEP / 8; ++s) {
            // columns past the last enter as zeros (of both operands)
            const bool in = k + 8 * s + 4 * half < k1;
            const int o = in ? k + 8 * s : 0;
            const float4 z = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            const float4 bw = *(const float4*)(wr + (in ? o : -4 * half));
            bv[s] = in ? bw : z;
#pragma unroll
            for (int b = 0; b < TB; ++b) {
                const float4 ax = *(const float4*)(xr[b] + (in ? o : -4 * half));
                av[b][s] = in ? ax : z;
            }
        }
        if constexpr (TB == 1) {
            acc[0] += rm_tree<0, RM_STEP, CH>(av[0], bv);
        } else {   // the token blocks' chains in turn (the tree's registers would spill)
#pragma unroll
            for (int c0 = 0; c0 < RM_STEP; c0 += CH) {
                f32x16 p[TB];
#pragma unroll
                for (int b = 0; b < TB; ++b)
#pragma unroll
                    for (int i = 0; i < 16; ++i) p[b][i] = 0.0f;
#pragma unroll
                for (int c = c0; c < c0 + CH; c += 2)
#pragma unroll
                    for (int b = 0; b < TB; ++b)
                        p[b] = __builtin_amdgcn_mfma_f32_32x32x2f32(((const float*)&av[b][c / 8])[c % 8 / 2],
                                                                    ((const float*)&bv[c / 8])[c % 8 / 2], p[b], 0, 0, 0);
#pragma unroll
                for (int b = 0; b < TB; ++b) acc[b] += p[b];
            }
        }
    }
    // D layout: register 4 g + i of lane l holds row 8 g + 4 (l / 32) + i, column l % 32
#pragma unroll
    for (int b = 0; b < TB; ++b)
#pragma unroll
        for (int i = 0; i < 16; ++i) part[wave][b][8 * (i / 4) + 4 * half + i % 4][l32] = acc[b][i];
    __syncthreads();
#pragma unroll
    for (int b = 0; b < TB; ++b) {
        const int row = threadIdx.x >> 5, col = threadIdx.x & 31;
        const int t = t0 + 32 * b + row, e = e0 + col;
        float v[RM_WAVES];
#pragma unroll
        for (int i = 0; i < RM_WAVES; ++i) v[i] = part[i][b][row][col];
#pragma unroll
        for (int d = 1; d < RM_WAVES; d *= 2)
#pragma unroll
            for (int i = 0; i < RM_WAVES; i += 2 * d) v[i] += v[i + d];
        if (t < n_tokens && e < n_experts) scores[(int64_t)t * n_experts + e] = v[0];
    }
}

template <int NM>
__global__ __launch_bounds__(64 * SEL_WAVES) void k_route_select(const float* __restrict__ scores, int n_tokens,
                                                                 int n_experts, int top_k, int32_t* __restrict__ ids,
                                                                 float* __restrict__ weights) {
    const int lane = threadIdx.x & 63;
    const int t = blockIdx.x * SEL_WAVES + (threadIdx.x >> 6);
    if (t >= n_tokens) return;   // the whole wave leaves: no workgroup barrier below
    uint32_t ord[NM];
    route_ords<NM>(scores + (int64_t)t * n_experts, n_experts, lane, ord);
    float mine = 0.0f;   // lane r keeps the r-th selected score
    for (int r = 0; r < top_k; ++r) {
        uint32_t best;
        const int win = route_next<NM>(ord, lane, best);
        if (lane == r) mine = ord_score(best);
        if (lane == 0) ids[(int64_t)t * top_k + r] = win;
    }
    const float w = route_weight(mine, top_k, lane);
    if (lane < top_k) weights[(int64_t)t * top_k + lane] = w;
}

template <int SPLIT, int TT>
static void launch_scores(const float* x, int n_tokens, int hidden, const float* w, int n_experts, float* scores,
                          hipStream_t stream) {
    constexpr int EPG = RS_WAVES / SPLIT;
    const dim3 grid((n_experts + EPG - 1) / EPG, (n_tokens + TT - 1) / TT);
    hipLaunchKernelGGL((k_route_scores<SPLIT, TT>), grid, dim3(64 * RS_WAVES), 0, stream, x, n_tokens, hidden, w,
                       n_experts, scores);
}

template <int TB>
static void launch_scores_mfma(const float* x, int n_tokens, int hidden, const float* w, int n_experts, float* scores,
                               hipStream_t stream) {
    const int n_etiles = (n_experts + 31) / 32, n_ttiles = (n_tokens + 32 * TB - 1) / (32 * TB);
    const int per = ((hidden + RM_WAVES - 1) / RM_WAVES + RM_STEP - 1) / RM_STEP * RM_STEP;
    const dim3 grid((unsigned)((n_ttiles + 7) / 8 * 8 * n_etiles)), block(64 * RM_WAVES);
    if (hidden >= 1536)
        hipLaunchKernelGGL((k_route_scores_mfma<TB, 16>), grid, block, 0, stream, x, n_tokens, hidden, w, n_experts,
                           scores, per, n_etiles);
    else
        hipLaunchKernelGGL((k_route_scores_mfma<TB, 8>), grid, block, 0, stream, x, n_tokens, hidden, w, n_experts,
                           scores, per, n_etiles);
}

template <int NM>
static void launch_select(const float* scores, int n_tokens, int n_experts, int top_k, int32_t* ids, float* weights,
                          hipStream_t stream) {
    hipLaunchKernelGGL((k_route_select<NM>), dim3((n_tokens + SEL_WAVES - 1) / SEL_WAVES), dim3(64 * SEL_WAVES), 0,
                       stream, scores, n_tokens, n_experts, top_k, ids, weights);
}

// Few tokens: four waves per expert row, so the n_experts x 4 waves spread
// over the chip, and as many token accumulators as there are tokens (up to 8).
// Above 32 tokens (us, the two kernels in turn):
//   up to 8192 scores the same, eight tokens at a time, against one wave per
//     expert over 16 tokens, which reads each row once per 16 tokens (4096 with
//     fewer than 16 experts of hidden 1025 to 4096).  Hidden 2048: 64 x 16 3.3/7.2, 33
//     x 256 5.7/7.7, 64 x 256 7.9/7.7; hidden 1536, 4096 x 2 13.1/10.1
//   then that kernel, while its workgroups (4 experts x 16 tokens) are few enough
//     for the chip to hold at once, four a CU, and with so few experts that most
//     columns of a matrix tile are empty: fewer than 8, or than 12 below hidden
//     1536.  Against the matrix kernel: 192 x 256 at hidden 1024 13.1/15.6, 2048
//     19.8/20.7, 7168 52.7/68.3; 24576 x 2 at hidden 768 21/36; 8192 x 8 at hidden
//     2048 27.8/22.3, 12288 x 8 at 768 20.1/23.8, 8000 x 12 at 768 22.8/17.6
//   the matrix kernel from there on: 260 x 256 at hidden 512 13.4/12.2, 1024
//     18.0/16.7, 2048 27.2/20.8; 128 x 512 and hidden 1024 or less 92-105 % of the
//     other's time, and at fewer than 96 tokens (of more than 700 experts) up to
//     107 %.  The vector kernel's fourth workgroup a CU already costs a round: there
//     the matrix kernel is ahead from hidden 1536 on (256 x 256 at 1536 0.87, at
//     2048 0.87) but for its long chains and idle XCDs with few tokens (768 or 1024
//     experts 1.01-1.08, hidden 7168 up to 1.05), and with one tile of experts
//     (4000 x 16 0.64-0.96 at every hidden size; up to 24 experts from hidden 1536
//     on already with the third, 3072 x 16 at 2048 23.1/19.7)
// The matrix kernel takes 64 tokens a workgroup where 32 would give well over one
// workgroup a CU (2048 x 256 at hidden 1024: 20.8, 32 tokens 26.9; 1024 x 256:
// 17.2 and 14.7), except under 16 experts (16384 x 8 at hidden 1536: 44.6 and 32.4).
static int64_t route_few_scores(int hidden, int n_experts) {
    return n_experts < 16 && hidden > 1024 && hidden <= 4096 ? 4096 : 8192;
}
static bool route_on_matrix(int n_tokens, int hidden, int n_experts) {
    if (hidden < 512 || n_experts < (hidden >= 1536 ? 8 : 12)) return false;
    const int64_t wg = (int64_t)((n_experts + 3) / 4) * ((n_tokens + 15) / 16);   // the vector kernel's
    if (wg > 4 * 256) return hidden >= 1536 || n_tokens >= 96;
    if (n_experts <= 24 && hidden >= 1536) return wg >= 3 * 256;
    return wg > 3 * 256 && (n_experts <= 32 || (hidden >= 1536 && n_experts <= (hidden <= 4096 ? 512 : 128)));
}
constexpr int64_t RM_WIDE_TILES = 384;
hipError_t launch_route_scores(const float* x, int n_tokens, int hidden, const float* w, int n_experts, float* scores,
                               hipStream_t stream) {
    const int64_t n = (int64_t)n_tokens * n_experts;
    if (n_tokens == 1) launch_scores<4, 1>(x, n_tokens, hidden, w, n_experts, scores, stream);
    else if (n_tokens == 2) launch_scores<4, 2>(x, n_tokens, hidden, w, n_experts, scores, stream);
    else if (n_tokens <= 4) launch_scores<4, 4>(x, n_tokens, hidden, w, n_experts, scores, stream);
    else if (n_tokens <= 32 || n <= route_few_scores(hidden, n_experts))
        launch_scores<4, 8>(x, n_tokens, hidden, w, n_experts, scores, stream);
    else if (!route_on_matrix(n_tokens, hidden, n_experts))
        launch_scores<1, 16>(x, n_tokens, hidden, w, n_experts, scores, stream);
    else if (hidden >= 1024 && n_experts >= 16 &&
             (int64_t)((n_tokens + 31) / 32) * ((n_experts + 31) / 32) > RM_WIDE_TILES)
        launch_scores_mfma<2>(x, n_tokens, hidden, w, n_experts, scores, stream);
    else launch_scores_mfma<1>(x, n_tokens, hidden, w, n_experts, scores, stream);
    return hipGetLastError();
}

hipError_t launch_route_select(const float* scores, int n_tokens, int n_experts, int top_k, int32_t* ids,
                               float* weights, hipStream_t stream) {
    const int nm = (n_experts + 63) / 64;
    if (nm <= 1) launch_select<1>(scores, n_tokens, n_experts, top_k, ids, weights, stream);
    else if (nm <= 2) launch_select<2>(scores, n_tokens, n_experts, top_k, ids, weights, stream);
    else if (nm <= 4) launch_select<4>(scores, n_tokens, n_experts, top_k, ids, weights, stream);
    else if (nm <= 8) launch_select<8>(scores, n_tokens, n_experts, top_k, ids, weights, stream);
    else launch_select<16>(scores, n_tokens, n_experts, top_k, ids, weights, stream);
    return hipGetLastError();
}

hipError_t launch_route(const float* x, int n_tokens, int hidden, const float* w, int n_experts, int top_k,
                        float* scores, int32_t* ids, float* weights, hipStream_t stream) {
    const hipError_t e = launch_route_scores(x, n_tokens, hidden, w, n_experts, scores, stream);
    if (e != hipSuccess) return e;
    return launch_route_select(scores, n_tokens, n_experts, top_k, ids, weights, stream);
}

}  // namespace mqh
