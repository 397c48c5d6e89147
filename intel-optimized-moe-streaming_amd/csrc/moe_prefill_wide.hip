// moe_prefill_wide.hip -- the prefill GEMMs for many tokens per expert.
//
// The kernels of moe_prefill.hip build every weight operand once per 16 tokens
// and hold a tile's whole K in LDS; with 128 tokens an expert that rebuilds each
// operand eight times (a 4096-token prompt: gate/up 564 us, down 676 us, the
// matrix cores a tenth busy).  Here a tile is up to 64 tokens of one expert, in
// NS = 1, 2 or 4 column blocks of 16, and an operand built in registers serves all
// of them:
//
//   W1 k_prefill_gate_up_wide  128 intermediate rows x one tile a workgroup, 16
//                              gate rows and the same 16 up rows a wave, SwiGLU
//                              in registers
//   W2 k_prefill_act_planes    the activations as FP16 planes, once per row
//   W3 k_prefill_down_wide     256 output rows x one tile a workgroup, 32 a wave
//
// K goes by in stages of one super-block (256 columns): the tile's 64 x 512
// bytes of each plane are copied to LDS, two buffers, one barrier a stage; the
// loads of the next stage's tokens and weights are issued ahead of a stage's
// arithmetic.  A wave's two row blocks share each token operand it reads from
// LDS (one row block would read 1 KB of LDS per 16-cycle MFMA, twice what the
// LDS delivers to four SIMDs).  The arithmetic and its order are those of
// moe_prefill.hip, so results are the same bit for bit.  Q8_0 down projections
// (a scale per step, so no room in the registers) stay there.
//
// Bound by vector arithmetic (a stage's operands and scales take 1.5 times as
// long as its MFMAs) that two waves a SIMD do not fully overlap with the matrix
// cores; 4096 BF16 tokens, 256 experts, top-8 + shared, Q4_K/Q6_K: W1 564 -> 315
// us, W3 676 -> 510 us, W2 26 us.  (Four waves a SIMD on one row block each,
// 128 registers, spilling: 345 and 483.)
#include <hip/hip_ext.h>

#include "moe_prefill.h"

namespace mqh {

constexpr int PW_WAVES = 8;
constexpr int PW_THREADS = 64 * PW_WAVES;
constexpr int PW_ROWS_GU = 128;               // gate/up rows of a workgroup, 16 of each matrix a wave
constexpr int PW_ROWS_DOWN = 256;             // down rows of a workgroup, 32 a wave
constexpr int PW_TOK = PREFILL_WIDE;
constexpr int PW_ROW = 512;                   // LDS bytes of a token's stage of one plane
constexpr int PW_PLANE = PW_TOK * PW_ROW;     // of a tile's
constexpr int PW_SUMS = PW_TOK * 32;          // a tile's sub-block sums
static_assert(PW_TOK == 64, "the staging deals 64 x 32 16-byte pieces to 512 threads");

struct PwLds {
    uint8_t *xh, *xl, *xs;   // two buffers each
};

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// The planes the tile's rows are read from
struct PwSrc {
    const uint16_t *hi, *lo;
    const uint32_t* sum;
};

// Both planes of a token row go to LDS in 16-byte pieces, piece c of token t in
// slot c ^ (t & 15) of its row: the sixteen tokens of a column block read their
// pieces of one column from sixteen slots, all banks once.
template <int T, int NS, bool SPLIT, bool IP>
struct PwGemm {
    static constexpr int NW = FragGeo<T>::NW, BB = frag_unit_bytes<T>();
    static constexpr bool MIN = FragGeo<T>::MIN;
    uint32_t raw[2][2][NW];   // [stage parity][row block]
    u32x4 xr[NS];             // one plane's pieces on their way to LDS
    uint32_t xsr;
    uint32_t off[NS];         // this thread's staged rows: element offset in the planes
    uint32_t soff;            // and its sub-block sum (threads below 128 NS)

    // Rows of the planes for the thread's staged tokens: row(r) for tile column r
    template <class F>
    __device__ __forceinline__ void rows(int K, F&& row) {
        const int tid = threadIdx.x;
#pragma unroll
        for (int i = 0; i < NS; ++i) off[i] = (uint32_t)row((tid >> 5) + 16 * i) * K + 8 * (tid & 31);
        if constexpr (MIN) soff = (uint32_t)row(min(tid >> 3, 16 * NS - 1)) * (K / 32) + (tid & 7);
    }

    __device__ __forceinline__ void load_x(const uint16_t* plane, int kb) {
#pragma unroll
        for (int i = 0; i < NS; ++i) xr[i] = *(const u32x4*)(plane + 256 * kb + off[i]);
    }

    __device__ __forceinline__ void store_x(uint8_t* plane, int buf) {
        const int tid = threadIdx.x, r = tid >> 5;
        const int o = buf * PW_PLANE + r * PW_ROW + (((tid & 31) ^ (r & 15)) << 4);
#pragma unroll
        for (int i = 0; i < NS; ++i) *(u32x4*)(plane + o + 16 * PW_ROW * i) = xr[i];
    }

    __device__ __forceinline__ void load_sums(const PwSrc& x, int kb) {
        if constexpr (MIN) xsr = (x.sum + 8 * kb)[soff];
    }

    __device__ __forceinline__ void store_sums(const PwLds& s, int buf) {
        if constexpr (MIN) {
            // a token's 32 bytes: eight high halves, then the eight low ones
            const int tid = threadIdx.x;
            if (tid < 128 * NS) {
                uint8_t* d = s.xs + buf * PW_SUMS + (tid >> 3) * 32 + 2 * (tid & 7);
                *(uint16_t*)d = (uint16_t)xsr;
                *(uint16_t*)(d + 16) = (uint16_t)(xsr >> 16);
            }
        }
    }

    __device__ __forceinline__ void read_b(const uint8_t* plane, int o, h8_t (&b)[NS]) {
#pragma unroll
        for (int n = 0; n < NS; ++n) b[n] = *(const h8_t*)(plane + o + 16 * PW_ROW * n);
    }

    // A stage: one super-block of both row blocks against the columns in buffer
    // `par`, with the tokens of stage nx on their way to the other buffer.
    //
    // Software-pipelined by hand: the operands of a round of MFMAs were read from
    // LDS (and built from the weights) a round earlier.  Left to itself the
    // compiler read each token operand right before its MFMA and waited for it.
    __device__ __forceinline__ void stage(const PwSrc& x, const PwLds& s, int par, int nx, f32x4 (&acc)[2][NS]) {
        // (the lane's index anew in every stage: its many derived shifts and
        // addresses would otherwise stay in registers across the loop)
        int lane = threadIdx.x & 63;
        __asm__ volatile("" : "+v"(lane));
        const int tok = lane & 15, q = lane >> 4, qq = (q + 3) & 3;
        const uint32_t (&cur)[2][NW] = raw[par];
        // (the lane's and the step's pieces differ in other bits, so the step's
        // is one exclusive or)
        const int base = par * PW_PLANE + tok * PW_ROW + (((frag_lane_col<T>(qq) >> 3) ^ tok) << 4);
        FragPrep<T> sp[2];
        f32x4 P[2][NS];
        h8_t a[2][2][2];        // [step parity][row block][part]
        h8_t bh[2][NS];         // SPLIT: [0] high, [1] low; else by step parity
        read_b(s.xh, base ^ (2 * frag_col<T, 0>()), bh[0]);
#pragma unroll
        for (int mt = 0; mt < 2; ++mt) {
            frag_prep<T, IP>(cur[mt], q, sp[mt]);
            frag_step<T, 0, IP>(cur[mt], sp[mt], q, a[0][mt]);
#pragma unroll
            for (int n = 0; n < NS; ++n) P[mt][n] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        }
        __builtin_amdgcn_sched_barrier(0);
        // one round: every row block and column block, one MFMA each
        auto round = [&](const h8_t& a0, const h8_t& a1, const h8_t (&b)[NS]) {
#pragma unroll
            for (int n = 0; n < NS; ++n) {
                P[0][n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a0, b[n], P[0][n], 0, 0, 0);
                P[1][n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a1, b[n], P[1][n], 0, 0, 0);
            }
        };
        pf_unroll(std::make_integer_sequence<int, 8>{}, [&](auto mc) {
            constexpr int m = decltype(mc)::value, pm = m & 1, nm = m < 7 ? m + 1 : 7;
            constexpr int bi = SPLIT ? 0 : pm;
            const int o = base ^ (2 * frag_col<T, m>()), on = base ^ (2 * frag_col<T, nm>());
            if constexpr (SPLIT) {
                read_b(s.xl, o, bh[1]);
                round(a[pm][0][0], a[pm][1][0], bh[0]);
                if constexpr (FragGeo<T>::NA == 2) round(a[pm][0][1], a[pm][1][1], bh[0]);
                __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (m < 7) {
                read_b(s.xh, on, bh[SPLIT ? 0 : pm ^ 1]);
#pragma unroll
                for (int mt = 0; mt < 2; ++mt) frag_step<T, nm, IP>(cur[mt], sp[mt], q, a[pm ^ 1][mt]);
            }
            if constexpr (SPLIT) {
                round(frag_lo_operand<T>(a[pm][0]), frag_lo_operand<T>(a[pm][1]), bh[1]);
            } else {
                round(a[pm][0][0], a[pm][1][0], bh[bi]);
                if constexpr (FragGeo<T>::NA == 2) round(a[pm][0][1], a[pm][1][1], bh[bi]);
            }
            if constexpr (m < 7) {
                // the reads first, then the next operands' arithmetic among the MFMAs
                __builtin_amdgcn_sched_group_barrier(0x100, NS, 0);
                pf_unroll(std::make_integer_sequence<int, 2 * NS>{}, [&](auto) {
                    __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x2, FragGeo<T>::NA == 2 ? 7 : 4, 0);
                });
            }
            __builtin_amdgcn_sched_barrier(0);
            // the high plane is in by now: on to LDS, and the low one's loads
            if constexpr (SPLIT && m == 3) {
                store_x(s.xh, par ^ 1);
                load_x(x.lo, nx);
                __builtin_amdgcn_sched_barrier(0);
            }
        });
#pragma unroll
        for (int mt = 0; mt < 2; ++mt) {
            // d (and dmin) of D row 4q + i live in the header word of A lane 4q + i
            uint32_t hdr[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) hdr[i] = (uint32_t)__shfl((int)cur[mt][FragGeo<T>::HDR], 4 * q + i, 64);
#pragma unroll
            for (int n = 0; n < NS; ++n) {
                f32x4 Mn;
                if constexpr (MIN) {
                    const h4_t bs = *(const h4_t*)(s.xs + par * PW_SUMS + (16 * n + tok) * 32 + 8 * q);
                    Mn = __builtin_amdgcn_mfma_f32_16x16x16f16(frag_mins<T>(cur[mt], q), bs,
                                                               f32x4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    acc[mt][n][i] = fmaf(frag_d<T>(hdr[i]), P[mt][n][i], acc[mt][n][i]);
                    if constexpr (MIN) acc[mt][n][i] = fmaf(-frag_dmin(hdr[i]), Mn[i], acc[mt][n][i]);
                }
            }
        }
    }

    // all nb super-blocks (1, or even) of the rows at W0 and W1
    __device__ __forceinline__ void run(int nb, const uint8_t* W0, const uint8_t* W1, const PwSrc& x, const PwLds& s,
                                        f32x4 (&acc)[2][NS]) {
        const int q = (threadIdx.x & 63) >> 4;
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
#pragma unroll
            for (int n = 0; n < NS; ++n) acc[mt][n] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        load_x(x.hi, 0);
        load_sums(x, 0);
        frag_load<T>(W0, q, raw[0][0]);
        frag_load<T>(W1, q, raw[0][1]);
        __builtin_amdgcn_sched_barrier(0);
        store_x(s.xh, 0);
        store_sums(s, 0);
        if constexpr (SPLIT) {
            load_x(x.lo, 0);
            store_x(s.xl, 0);
        }
        __syncthreads();
#pragma unroll 1
        for (int b = 0; b < nb; b += 2)
#pragma unroll
            for (int par = 0; par < 2; ++par) {
                const int kb = b + par;
                if (kb >= nb) break;
                // (past the last stage: the last one again, in bounds and unused)
                const int nx = min(kb + 1, nb - 1);
                load_x(x.hi, nx);
                load_sums(x, nx);
                frag_load<T>(W0 + nx * BB, q, raw[par ^ 1][0]);
                frag_load<T>(W1 + nx * BB, q, raw[par ^ 1][1]);
                __builtin_amdgcn_sched_barrier(0);
                // (the other buffer was last read in the stage before this one's
                // barrier, so it is written while this stage still runs)
                stage(x, s, par, nx, acc);
                store_x(SPLIT ? s.xl : s.xh, par ^ 1);
                store_sums(s, par ^ 1);
                __syncthreads();
            }
    }
};

// Workgroup -> (tile, chunk).  Workgroup i runs on XCD i % 8; the chunks of a
// tile go to one XCD (its tokens are read into one L2), and so do PW_GROUP
// tiles in a row (an expert's tiles follow each other and share its weights).
constexpr int PW_XCDS = 8, PW_GROUP = 4;
__device__ __forceinline__ void pw_wg(int nch_log2, int& tile, int& chunk) {
    const int j = blockIdx.x / PW_XCDS, g = j >> nch_log2;
    chunk = j & ((1 << nch_log2) - 1);
    tile = g / PW_GROUP * (PW_XCDS * PW_GROUP) + (int)(blockIdx.x % PW_XCDS) * PW_GROUP + g % PW_GROUP;
}
static unsigned pw_grid(int nch, int max_tiles) {
    constexpr int R = PW_XCDS * PW_GROUP;
    return (unsigned)(nch * ((max_tiles + R - 1) / R * R));
}

// f with the tile's number of column blocks as a constant
template <class F>
__device__ __forceinline__ void pw_blocks(int cnt, F&& f) {
    if (cnt <= 16) f(std::integral_constant<int, 1>{});
    else if (cnt <= 32) f(std::integral_constant<int, 2>{});
    else f(std::integral_constant<int, 4>{});
}

// ------------------------------------------------------------ W1

template <int GT, int SGT, bool XBF16>
__global__ __launch_bounds__(PW_THREADS) void k_prefill_gate_up_wide(PrefillParams p, int nch_log2) {
    constexpr bool SPLIT = !XBF16;   // BF16 tokens are exact in the high plane
    __shared__ __attribute__((aligned(16))) uint8_t xh[2 * PW_PLANE];
    __shared__ __attribute__((aligned(16))) uint8_t xl[SPLIT ? 2 * PW_PLANE : 16];
    __shared__ __attribute__((aligned(16))) uint8_t xs[2 * PW_SUMS];
    int tile, chunk;
    pw_wg(nch_log2, tile, chunk);
    if (tile >= *p.n_tiles) return;
    const int4 td = ((const int4*)p.tiles)[tile];
    const int e = td.x, first = td.y, cnt = td.z;
    const int lane = threadIdx.x & 63, q = lane >> 4, tok = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int rbase = chunk * PW_ROWS_GU + wave * 16;
    const uint8_t* Wg = e < 0 ? p.sh_gate : p.gate + (int64_t)e * p.gate_eb;
    const uint8_t* Wu = e < 0 ? p.sh_up : p.up + (int64_t)e * p.up_eb;
    const int* tt = p.tile_tok + (int64_t)tile * PW_TOK;
    const int nb = p.hidden / 256;

    auto body = [&](auto tc, auto nc) {
        constexpr int T = decltype(tc)::value, NS = decltype(nc)::value;
        PwGemm<T, NS, SPLIT, false> g;
        const int64_t wo = (int64_t)(rbase + tok) * nb * frag_unit_bytes<T>();
        // (columns at or past cnt hold stale words: column 0 stands in)
        g.rows(p.hidden, [&](int r) { return tt[r < cnt ? r : 0]; });
        f32x4 acc[2][NS];
        g.run(nb, Wg + wo, Wu + wo, PwSrc{p.xhi, p.xlo, p.xsum}, PwLds{xh, xl, xs}, acc);
#pragma unroll
        for (int n = 0; n < NS; ++n) {
            const int col = 16 * n + tok;
            if (col < cnt) {
                const float sc = ldexpf(1.0f, p.xexp[tt[col]]);
                const f32x4 gv = acc[0][n], uv = acc[1][n];
                float4 o;
                o.x = pf_silu_mul(gv[0] * sc, uv[0] * sc);
                o.y = pf_silu_mul(gv[1] * sc, uv[1] * sc);
                o.z = pf_silu_mul(gv[2] * sc, uv[2] * sc);
                o.w = pf_silu_mul(gv[3] * sc, uv[3] * sc);
                *(float4*)(p.act + (int64_t)(first + col) * p.inter + rbase + 4 * q) = o;
            }
        }
    };
    pw_blocks(cnt, [&](auto nc) {
        if constexpr (SGT == GT) body(std::integral_constant<int, GT>{}, nc);
        else if (e < 0) body(std::integral_constant<int, SGT>{}, nc);   // (uniform: the workgroup's tile)
        else body(std::integral_constant<int, GT>{}, nc);
    });
}

// ------------------------------------------------------------ W2

// One wave a row of the activations (the row's scale needs all of its chunks,
// which are other workgroups' in W1).
constexpr int PW_ACT_WAVES = 4;
template <int NBI>
__global__ __launch_bounds__(64 * PW_ACT_WAVES) void k_prefill_act_planes(PrefillParams p, int64_t n_rows) {
    constexpr int I = NBI * 256;
    const int64_t r = (int64_t)blockIdx.x * PW_ACT_WAVES + (threadIdx.x >> 6);
    if (r >= n_rows) return;
    PfStageRaw<I, false> raw;
    pf_stage_load<I, false>(p.act, r, true, raw);
    pf_stage_planes<I, false, true>(raw, r, PfPlanePtrs{p.ahi, p.alo, p.asum, p.aexp}, nullptr);
}

// ------------------------------------------------------------ W3

template <int DT, int SDT>
__global__ __launch_bounds__(PW_THREADS) void k_prefill_down_wide(PrefillParams p, int nch_log2) {
    __shared__ __attribute__((aligned(16))) uint8_t xh[2 * PW_PLANE];
    __shared__ __attribute__((aligned(16))) uint8_t xl[2 * PW_PLANE];
    __shared__ __attribute__((aligned(16))) uint8_t xs[2 * PW_SUMS];
    int tile, chunk;
    pw_wg(nch_log2, tile, chunk);
    if (tile >= *p.n_tiles) return;
    const int4 td = ((const int4*)p.tiles)[tile];
    const int e = td.x, first = td.y, cnt = td.z;
    const int lane = threadIdx.x & 63, q = lane >> 4, tok = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int rbase = chunk * PW_ROWS_DOWN + wave * 32;
    const uint8_t* W0 = e < 0 ? p.sh_down : p.down + (int64_t)e * p.down_eb;
    const int* td_dst = p.tile_dst + (int64_t)tile * PW_TOK;
    const int nb = p.inter / 256;

    auto body = [&](auto tc, auto nc) {
        constexpr int T = decltype(tc)::value, NS = decltype(nc)::value;
        PwGemm<T, NS, true, true> g;
        const int row_bytes = nb * frag_unit_bytes<T>();
        const uint8_t* W = W0 + (int64_t)(rbase + tok) * row_bytes;
        g.rows(p.inter, [&](int r) { return first + min(r, cnt - 1); });
        f32x4 acc[2][NS];
        g.run(nb, W, W + 16 * row_bytes, PwSrc{p.ahi, p.alo, p.asum}, PwLds{xh, xl, xs}, acc);
#pragma unroll
        for (int n = 0; n < NS; ++n) {
            const int col = 16 * n + tok;
            if (col < cnt) {
                const float sc = ldexpf(1.0f, p.aexp[first + col]);
                float* y = p.ypair + (int64_t)td_dst[col] * p.hidden + rbase + 4 * q;
#pragma unroll
                for (int mt = 0; mt < 2; ++mt)
                    *(float4*)(y + 16 * mt) = make_float4(acc[mt][n][0] * sc, acc[mt][n][1] * sc, acc[mt][n][2] * sc,
                                                          acc[mt][n][3] * sc);
            }
        }
    };
    pw_blocks(cnt, [&](auto nc) {
        if constexpr (SDT == DT) body(std::integral_constant<int, DT>{}, nc);
        else if (e < 0) body(std::integral_constant<int, SDT>{}, nc);
        else body(std::integral_constant<int, DT>{}, nc);
    });
}

// ------------------------------------------------------------ host side

#define PW_LAUNCH(kernel, grid, armed, e0, e1, s, p, nch)                                                          \
    do {                                                                                                           \
        if (armed)                                                                                                 \
            hipExtLaunchKernelGGL(kernel, dim3(grid), dim3(PW_THREADS), 0, s, e0, e1, 0, p, __builtin_ctz(nch));   \
        else                                                                                                       \
            hipLaunchKernelGGL(kernel, dim3(grid), dim3(PW_THREADS), 0, s, p, __builtin_ctz(nch));                 \
    } while (0)

template <int GT, int SGT>
static void launch_w1(const PrefillParams& p, hipStream_t s, const KernelEvents& ev) {
    const int nch = p.inter / PW_ROWS_GU;
    const unsigned grid = pw_grid(nch, p.max_tiles);
    if (p.x_bf16) PW_LAUNCH((k_prefill_gate_up_wide<GT, SGT, true>), grid, ev.armed_a(), ev.a_start, ev.a_stop, s, p, nch);
    else PW_LAUNCH((k_prefill_gate_up_wide<GT, SGT, false>), grid, ev.armed_a(), ev.a_start, ev.a_stop, s, p, nch);
}

// a shared expert of another type is Q6_K (prefill_supported admits no other)
template <int GT>
static void launch_w1_t(const PrefillParams& p, hipStream_t s, const KernelEvents& ev) {
    if constexpr (GT != T_Q6_K) {
        if (p.has_shared && p.sh_gate_type != GT) {
            launch_w1<GT, T_Q6_K>(p, s, ev);
            return;
        }
    }
    launch_w1<GT, GT>(p, s, ev);
}

template <int DT>
static void launch_w3_t(const PrefillParams& p, hipStream_t s, const KernelEvents& ev) {
    const int nch = p.hidden / PW_ROWS_DOWN;
    const unsigned grid = pw_grid(nch, p.max_tiles);
    if constexpr (DT != T_Q6_K) {
        if (p.has_shared && p.sh_down_type != DT) {
            PW_LAUNCH((k_prefill_down_wide<DT, T_Q6_K>), grid, ev.armed_b(), ev.b_start, ev.b_stop, s, p, nch);
            return;
        }
    }
    PW_LAUNCH((k_prefill_down_wide<DT, DT>), grid, ev.armed_b(), ev.b_start, ev.b_stop, s, p, nch);
}

hipError_t launch_prefill_wide(const PrefillParams& p, hipStream_t s, const KernelEvents& ev) {
    switch (p.gate_type) {
        case T_Q4_K: launch_w1_t<T_Q4_K>(p, s, ev); break;
        case T_Q5_K: launch_w1_t<T_Q5_K>(p, s, ev); break;
        case T_Q6_K: launch_w1_t<T_Q6_K>(p, s, ev); break;
        default: launch_w1_t<T_Q3_K>(p, s, ev); break;
    }
    hipError_t err = hipGetLastError();
    if (err != hipSuccess) return err;
    const int64_t rows = (int64_t)p.n_tokens * p.S;
    const dim3 grid((unsigned)((rows + PW_ACT_WAVES - 1) / PW_ACT_WAVES)), block(64 * PW_ACT_WAVES);
    switch (p.inter) {
        case 256: hipLaunchKernelGGL((k_prefill_act_planes<1>), grid, block, 0, s, p, rows); break;
        case 512: hipLaunchKernelGGL((k_prefill_act_planes<2>), grid, block, 0, s, p, rows); break;
        case 1024: hipLaunchKernelGGL((k_prefill_act_planes<4>), grid, block, 0, s, p, rows); break;
        default: hipLaunchKernelGGL((k_prefill_act_planes<8>), grid, block, 0, s, p, rows); break;
    }
    if ((err = hipGetLastError()) != hipSuccess) return err;
    switch (p.down_type) {
        case T_Q4_K: launch_w3_t<T_Q4_K>(p, s, ev); break;
        case T_Q5_K: launch_w3_t<T_Q5_K>(p, s, ev); break;
        case T_Q6_K: launch_w3_t<T_Q6_K>(p, s, ev); break;
        default: launch_w3_t<T_Q3_K>(p, s, ev); break;
    }
    return hipGetLastError();
}

}  // namespace mqh
