// moe_decode.hip -- fused quantized-expert decode for a few tokens (GEMV regime).
//
// Computes, for each token t and each of its routed slots s (expert ids[t,s],
// routing weight w[t,s]) plus an optional shared expert:
//   y_s  = W_down (silu(W_gate x) * (W_up x))            (moe_quant_dot.cpp:189-211)
//   y[t] = sum_s fl32(w_s) * y_s  (+ sigmoid(x . g_inp) * y_shared)
//                                                    (moe_layer.py:70-106,
//                                                     shared_expert.py:221-251)
// straight from the GGUF-quantized expert slices resident in HBM; experts are
// addressed through an index gather into the stacked [n_experts x slice]
// tensors, so one launch pair covers every expert of every token.
//
// Generic path (this file): every type and any multiple of the block size, with
// FP32 activations and FP32 sums.  Kernel A (gate/up/act), then kernel B (down
// and weighted combine).  The unit a lane decodes is 8 consecutive values of a
// row (decode8); a row of `cols` columns has cols/8 units, dealt to the L lanes
// of a row in turn (L = 64, or 32 with two rows a wave where that leaves no
// lane without a unit).
//
// Graph modes: fp16_graph=1 reproduces the reference's FP16 graph on the
// routed experts (x, weights, g, u, sigmoid, silu, act and y rounded to FP16
// at the points of moe_quant_dot.cpp:192-209); the shared expert always runs
// the FP32 graph, as the reference's NumPy shared expert does.
#include <hip/hip_ext.h>

#include "kquant_device.h"
#include "moe_decode.h"

namespace mqh {

__device__ __forceinline__ float sigmoid_ref(float g) { return 1.0f / (1.0f + expf(-g)); }

// Stable sigmoid of shared_expert.py:55-62.
__device__ __forceinline__ float sigmoid_stable(float v) {
    if (v >= 0.0f) return 1.0f / (1.0f + expf(-v));
    const float e = expf(v);
    return e / (1.0f + e);
}

// 32 bytes of FP32 values (a row may start at any 4-byte boundary)
__device__ __forceinline__ void ld_x8(const float* p, float (&v)[8]) {
    typedef float f4_a4 __attribute__((ext_vector_type(4), aligned(4)));
    const f4_a4 a = *(const f4_a4*)p, b = *(const f4_a4*)(p + 4);
    v[0] = a[0]; v[1] = a[1]; v[2] = a[2]; v[3] = a[3];
    v[4] = b[0]; v[5] = b[1]; v[6] = b[2]; v[7] = b[3];
}

// Lanes of a row: 64, or 32 (two rows a wave) where 64 would leave lanes idle
__host__ __device__ constexpr int gen_lanes(int cols) { return (cols >> 3) % 64 == 0 ? 64 : 32; }
// Units per lane and pass (1..4): all of them where there are at most four,
// else the passes' even share
static int gen_units(int cols) {
    const int n = ((cols >> 3) + gen_lanes(cols) - 1) / gen_lanes(cols), passes = (n + 3) / 4;
    return (n + passes - 1) / passes;
}

// Partial dot products of the lane's units (lp, lp + L, ...) of rows r0 of W0 and
// r1 of W1 (type T, 8 n8 columns) against the same values x, NJ units a pass.  A
// pass is straight-line code: the loads of all its units of both rows are issued
// before the first is used (one row and one unit at a time, behind a branch on
// the type per unit, left a wave with one load in flight).  Two sums a row, by
// the parity of the unit's place in the pass (with NJ = 1 one sum holds all).
template <int T, int NJ, bool RX, bool RW>
__device__ __forceinline__ void gen_dot2(const uint8_t* W0, int r0, const uint8_t* W1, int r1, const float* x, int n8,
                                         int lp, int L, float& out0, float& out1) {
    constexpr int UPB = block_size(T) / 8, PB = block_bytes(T);
    const int row_bytes = n8 / UPB * PB;   // (at most 65536 columns)
    const uint8_t* row0 = W0 + (int64_t)r0 * row_bytes;
    const uint8_t* row1 = W1 + (int64_t)r1 * row_bytes;
    float acc[2][2] = {{0.0f, 0.0f}, {0.0f, 0.0f}};
#pragma unroll 1
    for (int u0 = lp; u0 < n8; u0 += NJ * L) {
        float xv[NJ][8], w[2][NJ][8];
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            // a unit past the row's end re-reads the last one and is not summed
            const int u = min(u0 + j * L, n8 - 1);
            const int off = u / UPB * PB;
            ld_x8(x + 8 * u, xv[j]);
            decode8<T>(row0 + off, u % UPB, w[0][j]);
            decode8<T>(row1 + off, u % UPB, w[1][j]);
        }
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            if (j > 0 && u0 + j * L >= n8) break;
#pragma unroll
            for (int r = 0; r < 2; ++r)
#pragma unroll
                for (int k = 0; k < 8; ++k)
                    acc[r][j & 1] = fmaf(RW ? round16(w[r][j][k]) : w[r][j][k], RX ? round16(xv[j][k]) : xv[j][k],
                                         acc[r][j & 1]);
        }
    }
    out0 = acc[0][0] + acc[0][1];
    out1 = acc[1][0] + acc[1][1];
}

// The type is uniform over the wave: one branch a row pair.
template <int NJ, bool RX, bool RW>
__device__ __forceinline__ void gen_dot2_any(int type, const uint8_t* W0, int r0, const uint8_t* W1, int r1,
                                             const float* x, int n8, int lp, int L, float& a, float& b) {
    switch (type) {
        case T_Q8_0: gen_dot2<T_Q8_0, NJ, RX, RW>(W0, r0, W1, r1, x, n8, lp, L, a, b); break;
        case T_IQ4_NL: gen_dot2<T_IQ4_NL, NJ, RX, RW>(W0, r0, W1, r1, x, n8, lp, L, a, b); break;
        case T_Q3_K: gen_dot2<T_Q3_K, NJ, RX, RW>(W0, r0, W1, r1, x, n8, lp, L, a, b); break;
        case T_Q4_K: gen_dot2<T_Q4_K, NJ, RX, RW>(W0, r0, W1, r1, x, n8, lp, L, a, b); break;
        case T_Q5_K: gen_dot2<T_Q5_K, NJ, RX, RW>(W0, r0, W1, r1, x, n8, lp, L, a, b); break;
        default: gen_dot2<T_Q6_K, NJ, RX, RW>(W0, r0, W1, r1, x, n8, lp, L, a, b); break;
    }
}

constexpr int GEN_WAVES_A = 4;
constexpr int GEN_WAVES_B = 8;

// ------------------------------------------------------------ kernel A

// Grid (row groups + 1, slots, tokens): a wave takes one row (L = 64) or two
// (L = 32) of gate and up together.  The last x block of the shared slot sets
// its sigmoid gate instead (its own block: at the head of a row block it would
// lengthen the launch by its chain of loads).
// Bound by its chain of dependent loads and by the decoding arithmetic (FP32
// weights, about five operations a value).  Hidden 1536, intermediate 768, top-6
// of Q4_K/Q6_K and a shared expert, one token: 26.9 -> 12.2 us with the loads of
// a pass issued together, one wave a row instead of two row pairs in turn.
template <int NJ, bool F16>
__global__ __launch_bounds__(64 * GEN_WAVES_A) void k_gate_up(DecodeParams p) {
    const int t = blockIdx.z, s = blockIdx.y;
    const bool shared = (s == p.top_k);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const float* xt = p.x + (int64_t)t * p.hidden;
    if (blockIdx.x == gridDim.x - 1) {
        if (!shared || wave != 0) return;
        float sc = 1.0f;
        if (p.sh_gate_inp) {
            float acc[2] = {0.0f, 0.0f};
            const int n8 = p.hidden >> 3;
#pragma unroll 2
            for (int u = lane; u < n8; u += 64) {
                float a[8], b[8];
                ld_x8(xt + 8 * u, a);
                ld_x8(p.sh_gate_inp + 8 * u, b);
#pragma unroll
                for (int k = 0; k < 8; ++k) acc[k & 1] = fmaf(a[k], b[k], acc[k & 1]);
            }
            sc = sigmoid_stable(group_sum(acc[0] + acc[1], 64));
        }
        if (lane == 0) p.sh_scale[t] = sc;
        return;
    }
    const int L = gen_lanes(p.hidden), rpw = 64 / L;
    const int lp = lane & (L - 1);
    const int r = (blockIdx.x * GEN_WAVES_A + wave) * rpw + (L == 64 ? 0 : lane >> 5);
    float* at = p.act + ((int64_t)t * p.S + s) * p.Imax;
    // every argument either kind of slot needs, awaited together with the expert
    // id (loaded where they are used, each is a memory round trip of its own)
    const int id = shared ? 0 : p.ids[t * p.top_k + s];
    const uint8_t *gate = p.gate, *up = p.up, *sh_gate = p.sh_gate, *sh_up = p.sh_up;
    const int64_t geb = p.gate_eb, ueb = p.up_eb;
    const int gtr = p.gate_type, utr = p.up_type, gts = p.sh_gate_type, uts = p.sh_up_type;
    const int ir = p.inter, is = p.sh_inter;
    __asm__ volatile("" ::"s"(id), "s"(gate), "s"(up), "s"(sh_gate), "s"(sh_up), "s"(geb), "s"(ueb), "s"(gtr), "s"(utr),
                     "s"(gts), "s"(uts), "s"(ir), "s"(is));
    const int I = shared ? is : ir, gt = shared ? gts : gtr, ut = shared ? uts : utr;
    // nothing to do for a wave whose rows are all past this slot's intermediate
    // size (the grid is the larger one's, routed or shared), and for an expert id
    // out of range, which is flagged and contributes nothing
    const bool bad = id < 0 || (!shared && id >= p.n_experts);
    if (bad || (int)(blockIdx.x * GEN_WAVES_A + __builtin_amdgcn_readfirstlane(wave)) * rpw >= I) {
        if (bad && threadIdx.x == 0 && blockIdx.x == 0) atomicOr(&p.flags[FLAG_BAD_ID], 1);
        if (bad && r < I && lp == 0) at[r] = 0.0f;
        return;
    }
    const uint8_t* G = shared ? sh_gate : gate + (int64_t)id * geb;
    const uint8_t* U = shared ? sh_up : up + (int64_t)id * ueb;
    // (a lane past the last row computes that row again and stores nothing)
    const int rr = min(r, I - 1), n8 = p.hidden >> 3;
    const bool f16 = F16 && !shared;
    float g, u, unused;
    if (gt == ut) {
        if (f16) gen_dot2_any<NJ, F16, F16>(gt, G, rr, U, rr, xt, n8, lp, L, g, u);
        else gen_dot2_any<NJ, false, false>(gt, G, rr, U, rr, xt, n8, lp, L, g, u);
    } else if (f16) {
        gen_dot2_any<1, F16, F16>(gt, G, rr, G, rr, xt, n8, lp, L, g, unused);
        gen_dot2_any<1, F16, F16>(ut, U, rr, U, rr, xt, n8, lp, L, u, unused);
    } else {
        gen_dot2_any<1, false, false>(gt, G, rr, G, rr, xt, n8, lp, L, g, unused);
        gen_dot2_any<1, false, false>(ut, U, rr, U, rr, xt, n8, lp, L, u, unused);
    }
    g = group_sum(g, L);
    u = group_sum(u, L);
    if (r < I && lp == 0) {
        float a;
        if (f16) {
            g = round16(g); u = round16(u);
            const float sig = round16(sigmoid_ref(g));
            const float silu = round16(g * sig);
            a = round16(silu * u);
        } else {
            a = (g * sigmoid_ref(g)) * u;
        }
        at[r] = a;
    }
}

// ------------------------------------------------------------ kernel B

// Grid (row groups, tokens): a workgroup takes two rows (L = 64) or four (L =
// 32) of the output, a wave the slots wave, wave + waves, ... of them, and the
// slots' results are added in slot order from LDS (GEN_SLOT floats a slot).
// At the size above 51.3 -> 10.7 us: one wave over all slots in turn left 1.5
// waves a CU and a chain of seven slots' loads.
constexpr int GEN_MAX_SLOTS = 65;   // top_k <= 64 and the shared expert
constexpr int GEN_SLOT = 6;   // four rows' results, the routing weight, 1.0 if the slot counts
template <int NJ, bool F16>
__global__ __launch_bounds__(64 * GEN_WAVES_B) void k_down_combine(DecodeParams p, int rows_b) {
    __shared__ float s_slot[GEN_MAX_SLOTS * GEN_SLOT];
    const int t = blockIdx.y;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
    for (int s = __builtin_amdgcn_readfirstlane(wave); s < p.S; s += nw) {
        const bool shared = (s == p.top_k);
        const int slot = t * p.top_k + (shared ? 0 : s);
        const int id = shared ? 0 : p.ids[slot];
        const float w = shared ? p.sh_scale[t] : p.weights[slot];
        const uint8_t *down = p.down, *sh_down = p.sh_down;
        const int64_t deb = p.down_eb;
        const int dtr = p.down_type, dts = p.sh_down_type, ir = p.inter, is = p.sh_inter;
        __asm__ volatile("" ::"s"(id), "s"(w), "s"(down), "s"(sh_down), "s"(deb), "s"(dtr), "s"(dts), "s"(ir), "s"(is));
        if (id < 0 || (!shared && id >= p.n_experts)) {
            if (lane == 0) s_slot[s * GEN_SLOT + 5] = 0.0f;
            continue;
        }
        const uint8_t* D = shared ? sh_down : down + (int64_t)id * deb;
        const int dt = shared ? dts : dtr, I = shared ? is : ir;
        const float* at = p.act + ((int64_t)t * p.S + s) * p.Imax;
        const int L = gen_lanes(I), lp = lane & (L - 1);
        const bool f16 = F16 && !shared;
        // rows r0 and r0 + rpw of a pass of 2 rpw rows; the workgroup's rows are
        // rows_b whatever this slot's L is
        const int rpw = 64 / L, lr = L == 64 ? 0 : lane >> 5;
#pragma unroll 1
        for (int c = 0; c < rows_b; c += 2 * rpw) {
            const int r0 = blockIdx.x * rows_b + c + lr;
            const int ra = min(r0, p.hidden - 1), rb = min(r0 + rpw, p.hidden - 1);
            float a, b;
            if (f16) gen_dot2_any<NJ, false, F16>(dt, D, ra, D, rb, at, I >> 3, lp, L, a, b);
            else gen_dot2_any<NJ, false, false>(dt, D, ra, D, rb, at, I >> 3, lp, L, a, b);
            a = group_sum(a, L);
            b = group_sum(b, L);
            if (f16) {
                a = round16(a);
                b = round16(b);
            }
            if (lp == 0) {
                if ((r0 < p.hidden && !isfinite(a)) || (r0 + rpw < p.hidden && !isfinite(b)))
                    atomicOr(&p.flags[FLAG_NONFINITE], 1);
                if (c + lr < rows_b) s_slot[s * GEN_SLOT + c + lr] = a;
                if (c + lr + rpw < rows_b) s_slot[s * GEN_SLOT + c + lr + rpw] = b;
            }
        }
        if (lane == 0) {
            s_slot[s * GEN_SLOT + 4] = w;
            s_slot[s * GEN_SLOT + 5] = 1.0f;
        }
    }
    __syncthreads();
    const int r = blockIdx.x * rows_b + threadIdx.x;
    if (threadIdx.x < rows_b && r < p.hidden) {
        float acc = 0.0f;
        for (int s = 0; s < p.S; ++s) {
            const float* v = s_slot + s * GEN_SLOT;
            if (v[5] != 0.0f) acc = __fadd_rn(acc, __fmul_rn(v[4], v[threadIdx.x]));
        }
        p.y[(int64_t)t * p.hidden + r] = acc;
        if (!isfinite(acc)) atomicOr(&p.flags[FLAG_NONFINITE], 1);
    }
}

template <int NJ, bool F16>
static void launch_gen_a(const DecodeParams& p, dim3 grid, hipStream_t stream, const KernelEvents& ev) {
    if (ev.armed_a())
        hipExtLaunchKernelGGL((k_gate_up<NJ, F16>), grid, dim3(64 * GEN_WAVES_A), 0, stream, ev.a_start, ev.a_stop, 0, p);
    else
        hipLaunchKernelGGL((k_gate_up<NJ, F16>), grid, dim3(64 * GEN_WAVES_A), 0, stream, p);
}

template <int NJ, bool F16>
static void launch_gen_b(const DecodeParams& p, dim3 grid, int rows_b, hipStream_t stream, const KernelEvents& ev) {
    const dim3 block(64 * std::min(p.S, GEN_WAVES_B));
    if (ev.armed_b())
        hipExtLaunchKernelGGL((k_down_combine<NJ, F16>), grid, block, 0, stream, ev.b_start, ev.b_stop, 0, p, rows_b);
    else
        hipLaunchKernelGGL((k_down_combine<NJ, F16>), grid, block, 0, stream, p, rows_b);
}

template <bool F16>
static hipError_t launch_generic(const DecodeParams& p, hipStream_t stream, const KernelEvents& ev) {
    const int rows_a = GEN_WAVES_A * 64 / gen_lanes(p.hidden);
    const dim3 ga((p.Imax + rows_a - 1) / rows_a + 1, p.S, p.n_tokens);
    switch (gen_units(p.hidden)) {
        case 1: launch_gen_a<1, F16>(p, ga, stream, ev); break;
        case 2: launch_gen_a<2, F16>(p, ga, stream, ev); break;
        case 3: launch_gen_a<3, F16>(p, ga, stream, ev); break;
        default: launch_gen_a<4, F16>(p, ga, stream, ev); break;
    }
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess) return err;
    const int inter = p.top_k > 0 ? p.inter : p.sh_inter;
    const int rows_b = 2 * 64 / gen_lanes(inter);
    const dim3 gb((p.hidden + rows_b - 1) / rows_b, p.n_tokens);
    switch (gen_units(inter)) {
        case 1: launch_gen_b<1, F16>(p, gb, rows_b, stream, ev); break;
        case 2: launch_gen_b<2, F16>(p, gb, rows_b, stream, ev); break;
        case 3: launch_gen_b<3, F16>(p, gb, rows_b, stream, ev); break;
        default: launch_gen_b<4, F16>(p, gb, rows_b, stream, ev); break;
    }
    return hipGetLastError();
}

hipError_t launch_decode_generic(const DecodeParams& p, hipStream_t stream, const KernelEvents& ev) {
    return p.fp16 ? launch_generic<true>(p, stream, ev) : launch_generic<false>(p, stream, ev);
}

}  // namespace mqh
