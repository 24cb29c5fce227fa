// MatMul of several activation rows in the host backend's summation order (the dots of exact_order.hip, bit for bit), from 2 rows to
// whole prompts: weights in their native blocks, activations quantized to Q8_0 and laid out once as fp16.
//
// Q4_0 / Q8_0 (Dot<Q4_0,Q8_0>, Dot<Q8_0,Q8_0>; vec_dot.h:42-115): every output has eight accumulators, one per "word" of four
// elements of a block, and every block adds fma(d_w * d_x, float(integer sum of the word's four products), acc) to each.
//   * The integer sums come from v_mfma_f32_16x16x4_4b_f16 as floats (products and sums of small integers: exact): lane block q
//     (lanes 16q .. 16q + 15) supplies word q of 16 weight rows and of 16 activation rows, so one instruction yields one term of four
//     accumulators of a 16 x 16 tile.
//   * The scale products of four blocks come from ONE more such instruction: element 0 of lane block b is d_w resp. d_x of block b, the
//     rest is zero, and a product of two fp16 values is exact in fp32 (subnormal scales included).
//   * The vector units do one fma per term; that is what bounds the kernel: 4096 x 4096 x 2048 is 1.34e8 wave-fmas = 255 us at the
//     2.05 GHz the part holds under this load.
//   * A weight word is used by exactly one wave, which unpacks it itself (0x6400 | n is the fp16 1024 + n) and applies it to C groups
//     of 16 activation rows.  The accumulators of an output are split over two waves (words 0..3 | 4..7), which meet in hsum_float_8 at the
//     end: a wave's chain is half as long.
//   * Weights (in chunks of eight blocks) and activations (in stages of four) go from memory straight into rings of LDS slots
//     (global_load_lds), P stages ahead of their use, one workgroup barrier per stage.
// Measured against what these kernels replaced (operands packed as fp16 once per call, 64 x 64 tiles), packing included:
// 4096 x 4096 Q4_0: 16 rows 80 -> 15 us, 77 rows 104 -> 28, 512 rows 137 -> 88, 2048 rows 400 -> 313; 8 rows (one launch per row) 36 -> 15.
#include "common.cuh"
#include "exact_sum.cuh"
#include "gemm_tiles.h"
#include "xt_pack.cuh"

#include <type_traits>
#include <utility>

namespace {

typedef _Float16 xt_h2 __attribute__((ext_vector_type(2)));
typedef _Float16 xt_h4 __attribute__((ext_vector_type(4)));
typedef float xt_v16f __attribute__((ext_vector_type(16)));

// 16 (4) bytes per lane from base + off to LDS bytes lds .. in lane order; base and lds are uniform over the wave.  Written as
// instructions so that the compiler does not wait for them at the next LDS read; xt_wait_vm says when they have to be there.
// (m0 among the clobbers keeps the compiler's own uses of it, if it has any, apart from these; it warns that the register is a reserved one.)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void xt_dma16(const void *base, uint32_t off, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" :: "s"(lds), "v"(off), "s"(base) : "memory", "m0");
}
__device__ __forceinline__ void xt_dma4(const void *base, uint32_t off, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" :: "s"(lds), "v"(off), "s"(base) : "memory", "m0");
}
#pragma clang diagnostic pop
// at most N of the wave's requests are still on their way (they complete in order), and its LDS reads are done
template <int N> __device__ __forceinline__ void xt_wait_vm() { asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" :: "n"(N) : "memory"); }

__device__ __forceinline__ xt_v16f xt_mfma(uint32_t a0, uint32_t a1, uint32_t b0, uint32_t b1) {
    const xt_v16f c = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    return __builtin_amdgcn_mfma_f32_16x16x4f16(__builtin_bit_cast(xt_h4, make_uint2(a0, a1)), __builtin_bit_cast(xt_h4, make_uint2(b0, b1)), c, 0, 0, 0);
}
__device__ __forceinline__ uint32_t xt_sub(uint32_t v, uint32_t c) {
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(xt_h2, v) - __builtin_bit_cast(xt_h2, c));
}
__device__ __forceinline__ uint32_t xt_and_or(uint32_t v, uint32_t m, uint32_t o) {
    uint32_t r;
    asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(v), "s"(m), "v"(o));
    return r;
}

template <int WT> struct xt_w {
    static constexpr int BB = WT == SPY_HIP_Q4_0 ? 18 : 34, CB = 8 * BB, CU = CB / 16, PD = BB / 2;     // bytes of a block and of a chunk of a row, 16-byte units of that, dwords of a block pair
};
struct xt_args {
    const uint8_t *w[3];                           // up to three matrices of the same shape that share the activations (wq | wk | wv, gate | up)
    float *dst[3];
    const float *resid;                            // added to the result (matrix 0 only), or null
    int64_t w_row, d_row;                          // bytes per weight row; elements between the outputs of two activation rows
    int M, tiles, nst, ncg, T;                     // rows and row tiles per matrix, stages (K / 128), groups of 16 activation rows, activation rows
    int ncg_all;                                   // groups of the whole call of which this is a piece
    const uint8_t *xq, *xd;
};
// What the first requests of a launch need, ahead of the rest: the first 14 dwords of a kernel's arguments come in registers (Makefile).  K-quant tiles 1 % faster by it
// (4096 x 11008 x 100 Q4_K 71.3 -> 69.8 us, 8192 x 4096 x 17 25.5 -> 25.1).  Not xks_kernel and xn_kernel, the short ones: at two workgroups per compute unit
// 4096 x 4096 x 17 Q4_K 15.5 us without, 17.1 with, 8192 x 4096 x 8 16.7 and 17.9, 5120 x 5120 x 8 17.5 and 18.4; 4096 x 11008 x 17 Q6_K 48.9 and 50.2; xn_kernel 4096 x 11008 x 8 Q4_0
// 23.3 and 24.0; 1024 x 1024 of any type 0.1 more of 7.
#define XT_PARAMS const uint8_t *w0_, const uint8_t *w1_, const uint8_t *w2_, const uint8_t *xq_, const uint8_t *xd_, int64_t w_row_, int tiles_, int nst_, xt_args a
#define XT_HOT const xt_hot hot = {w0_, w1_, w2_, xq_, xd_, w_row_, tiles_, nst_}
#define XT_ARGS(a) (a).w[0], (a).w[1], (a).w[2], (a).xq, (a).xd, (a).w_row, (a).tiles, (a).nst, (a)
struct xt_hot {
    const uint8_t *w0, *w1, *w2, *xq, *xd;
    int64_t w_row;
    int tiles, nst;
    __device__ __forceinline__ int mat(int b) const { return (b >= tiles ? 1 : 0) + (b >= 2 * tiles ? 1 : 0); }      // matrix of a workgroup
    __device__ __forceinline__ const uint8_t *w(int m) const { return m == 0 ? w0 : m == 1 ? w1 : w2; }
};

// AS: waves that share the accumulators of a tile; RG: groups of 16 weight rows per workgroup; C: groups of 16 activation rows per
// wave; NXS, NWC: LDS slots for stages and chunks (powers of two); P: stages requested ahead
template <int WT, int C, int NXS, int P, int NWC>
__device__ __forceinline__ void xt_tile(const xt_hot &hot, const xt_args &a, int cg0) {
    constexpr int AS = 2, RG = 2;
    constexpr int NT = 64 * AS * RG, ROWS = 16 * RG;
    constexpr int CU = xt_w<WT>::CU, UW = ROWS * CU, NI = (UW + NT - 1) / NT, NXI = C * 256 / NT;
    constexpr int XB = C * (XT_XB + 256), WB = (UW + 63) / 64 * 1024;
    static_assert(NXI * NT == C * 256 && AS * RG >= C && NXS > P && NWC * 2 > P, "one request per thread and group, one wave per group's scales, slots for what is on its way");
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = wave % AS, rg = wave / AS, q = lane >> 4, r = lane & 15;
    const int mat = hot.mat((int)blockIdx.x), m0 = ((int)blockIdx.x - mat * hot.tiles) * ROWS;
    const int nst = hot.nst, ncg = a.ncg, M = a.M;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)smem;

    // what a wave requests: uniform bases that advance, per-lane offsets that stay.  Row groups and activation groups past the end
    // repeat the last one.
    // The last request of a chunk covers it with the first waves only; the others repeat the first wave's, the same bytes to the same place.  (With a spare
    // kilobyte for what they repeat a compute unit had room for two workgroups of the Q8_0 tile instead of three: 22016 x 4096 x 512 474 -> 448 us,
    // 4096 x 4096 x 2048 347 -> 326, 12288 x 4096 x 100 69.7 -> 61.8.)
    const int wl = wave * 64 + (NI - 1) * NT >= UW ? 0 : wave;
    const uint8_t *bx[NXI], *bd, *bw = hot.w(mat) + (int64_t)m0 * hot.w_row;
    uint32_t ow[NI];
#pragma unroll
    for (int i = 0; i < NXI; i++) bx[i] = hot.xq + (int64_t)min(cg0 + (i * NT + wave * 64) / 256, ncg - 1) * nst * XT_XB + (i * NT + wave * 64) % 256 * 16;
    bd = hot.xd + (int64_t)min(cg0 + min(wave, C - 1), ncg - 1) * nst * XT_XD;
#pragma unroll
    for (int i = 0; i < NI; i++) {
        const int u = min((i == NI - 1 ? wl * 64 + lane : tid) + i * NT, UW - 1);
        ow[i] = (uint32_t)(min(m0 + u / CU, M - 1) - m0) * (uint32_t)hot.w_row + (u % CU) * 16;
    }
    const uint32_t l16 = lane * 16, l4 = lane * 4;
    const uint32_t ldsx = __builtin_amdgcn_readfirstlane(lds0 + wave * 1024), ldsd = __builtin_amdgcn_readfirstlane(lds0 + C * XT_XB + min(wave, C - 1) * 256),
                   ldsw = __builtin_amdgcn_readfirstlane(lds0 + NXS * XB + wave * 1024), ldswl = __builtin_amdgcn_readfirstlane(lds0 + NXS * XB + wl * 1024);
    int is = 0;                                    // next stage to request; past the last one it is requested again (same count of requests, slot unused)
    auto issue_x = [&]() {
        const uint32_t o = (is & (NXS - 1)) * XB;
        const int adv = is + 1 < nst ? 1 : 0;
#pragma unroll
        for (int i = 0; i < NXI; i++) { xt_dma16(bx[i], l16, ldsx + o + i * NT * 16); bx[i] += adv * XT_XB; }
        xt_dma4(bd, l4, ldsd + o);
        bd += adv * XT_XD;
        is++;
    };
    auto issue_w = [&]() {
        const uint32_t o = ((is >> 1) & (NWC - 1)) * WB;
#pragma unroll
        for (int i = 0; i < NI; i++) xt_dma16(bw, ow[i], (i == NI - 1 ? ldswl : ldsw) + o + i * NT * 16);
        bw += is + 2 < nst ? xt_w<WT>::CB : 0;
    };
#pragma unroll
    for (int s = 0; s < P; s++) { if ((s & 1) == 0) issue_w(); issue_x(); }

    constexpr int NACC = 32 / AS;                  // accumulators per lane and activation group: [word of the wave][4 weight rows 4q .. 4q + 3], activation row r
    float acc[C][NACC];
#pragma unroll
    for (int c = 0; c < C; c++)
#pragma unroll
        for (int i = 0; i < NACC; i++) acc[c][i] = 0.0f;

    // Where a lane finds its operands: word 4g + q of one block per matrix instruction.  A Q4_0 block holds words 0..3 in the low nibbles and 4..7 in the
    // high nibbles of its four quant dwords (which start at byte 2: blocks at odd dword halves are read as two dwords).
    constexpr bool Q4 = WT == SPY_HIP_Q4_0;
    constexpr int PD = xt_w<WT>::PD, OD = Q4 ? 5 : 9, BB = xt_w<WT>::BB;
    const uint32_t wbase = (rg * 16 + r) * xt_w<WT>::CB +
                           4 * (q + (Q4 ? 0 : 4 * g));
    const int sh = Q4 ? 4 * g : 0;
    const uint32_t dbase = (rg * 16 + r) * xt_w<WT>::CB + q * BB;
    const uint32_t xbase = (2 * g + (q >> 1)) * 256 + r * 16 + (q & 1) * 8;
    const uint32_t c64 = 0x64006400u;

    auto compute = [&](int s, auto par_c) {
        constexpr int par = decltype(par_c)::value;                 // which half of the chunk
        const uint8_t *sx = smem + (s & (NXS - 1)) * XB, *sw = smem + NXS * XB + ((s >> 1) & (NWC - 1)) * WB;
        constexpr int NW = 4;                                       // weight operands of the stage
        uint32_t wa[NW], wb[NW];
        {
            const uint32_t *b = (const uint32_t *)(sw + wbase);
            uint32_t v[NW];
#pragma unroll
            for (int i = 0; i < 2; i++) {
                v[2 * i] = __builtin_amdgcn_alignbit(b[PD * (2 * par + i) + 1], b[PD * (2 * par + i)], 16);
                v[2 * i + 1] = b[PD * (2 * par + i) + OD];
            }
#pragma unroll
            for (int i = 0; i < NW; i++) {                          // elements 0, 2 and 1, 3 of the word
                if constexpr (Q4) {
                    wa[i] = xt_sub(xt_and_or(v[i] >> sh, 0x000F000Fu, c64), 0x64086408u);
                    wb[i] = xt_sub(xt_and_or(v[i] >> (sh + 8), 0x000F000Fu, c64), 0x64086408u);
                } else {
                    const uint32_t t = v[i] ^ 0x80808080u;
                    wa[i] = xt_sub(xt_and_or(t, 0x00FF00FFu, c64), 0x64806480u);
                    wb[i] = xt_sub(xt_and_or(t >> 8, 0x00FF00FFu, c64), 0x64806480u);
                }
            }
        }
        uint32_t dw = *(const uint16_t *)(sw + dbase + par * 4 * BB);
        dw = dw == 0xFFFFu ? 0u : dw;                               // conversion.h:39-41: the host's table has no entry for 0xFFFF
        const uint8_t *sd = sx + C * XT_XB + lane * 4;
        // steps (activation group, weight operand), pipelined by hand: the activations of step j + 2 are read and the matrix instruction of step
        // j + 1 is issued before the fmas on the result of step j
        constexpr int NJ = C * NW;
        auto rd = [&](int j) -> uint2 { return *(const uint2 *)(sx + (j / NW) * XT_XB + (j % NW) * 1024 + xbase); };
        uint2 xv[3];
        xt_v16f p[2], D[2];
        uint32_t dx = *(const uint32_t *)sd, dxn = 0;
        xv[0] = rd(0);
        xv[1] = rd(1);
        if (C > 1) dxn = *(const uint32_t *)(sd + 256);
        D[0] = xt_mfma(dw, 0u, dx, 0u);
        p[0] = xt_mfma(wa[0], wb[0], xv[0].x, xv[0].y);
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            const int c = j / NW, i = j % NW;
            if (j + 2 < NJ) xv[(j + 2) % 3] = rd(j + 2);
            if (j + 1 < NJ) {
                const int c1 = (j + 1) / NW, i1 = (j + 1) % NW;
                if (i1 == 0) {
                    D[c1 & 1] = xt_mfma(dw, 0u, dxn, 0u);
                    if (c1 + 1 < C) dxn = *(const uint32_t *)(sd + (c1 + 1) * 256);
                }
                p[(j + 1) & 1] = xt_mfma(wa[i1], wb[i1], xv[(j + 1) % 3].x, xv[(j + 1) % 3].y);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int n = 0; n < 16; n++) acc[c][n] = fmaf(D[c & 1][4 * i + (n & 3)], p[j & 1][n], acc[c][n]);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // A stage: its data are there (of the requests only those of the P - 1 stages after it may be on their way), every wave is past the
    // stage before (whose slot is requested into next), the request, the sums.
    constexpr int N0 = (P - 1) * NXI + (P - 1), CE = (P - 1) / 2, CO = P / 2;       // chunks among the P - 1 stages after an even / odd stage
    auto ready = [&](auto odd) {
        constexpr int n = decltype(odd)::value ? CO : CE;
        xt_wait_vm<N0 + n * NI>();
        __builtin_amdgcn_s_barrier();
    };
    for (int s = 0; s < nst; s += 2) {
        ready(std::integral_constant<int, 0>{});
        if ((P & 1) == 0) issue_w();
        issue_x();
        compute(s, std::integral_constant<int, 0>{});
        ready(std::integral_constant<int, 1>{});
        if ((P & 1) == 1) issue_w();
        issue_x();
        compute(s + 1, std::integral_constant<int, 1>{});
    }
    xt_wait_vm<0>();
    __builtin_amdgcn_s_barrier();
    // hsum_float_8 (vec_util.h:75-81): r_k = word k + word k + 4, (r0 + r2) + (r1 + r3); the other waves' accumulators come through LDS
    float *ex = (float *)smem + (rg * (AS - 1)) * (C * NACC * 64);
    if (g > 0) {
#pragma unroll
        for (int c = 0; c < C; c++)
#pragma unroll
            for (int n = 0; n < NACC; n++) ex[(((g - 1) * C + c) * NACC + n) * 64 + lane] = acc[c][n];
    }
    __syncthreads();
    if (g > 0) return;
    const int row = m0 + rg * 16 + 4 * q;
    float *dst = a.dst[mat];
#pragma unroll
    for (int c = 0; c < C; c++) {
        float o[4];
#pragma unroll
        for (int v = 0; v < 4; v++) {
            float rr[4];
#pragma unroll
            for (int k = 0; k < 4; k++) rr[k] = ex[(c * NACC + 4 * k + v) * 64 + lane] + acc[c][4 * k + v];
            const float s0 = rr[0] + rr[2], s1 = rr[1] + rr[3];
            o[v] = s0 + s1;
        }
        const int t = (cg0 + c) * 16 + r;
        if (t < a.T) {
            const int64_t at = (int64_t)t * a.d_row + row;
            if (row + 3 < M) {
                if (a.resid) { const float4 z = *(const float4 *)(a.resid + at); o[0] += z.x; o[1] += z.y; o[2] += z.z; o[3] += z.w; }
                *(float4 *)(dst + at) = make_float4(o[0], o[1], o[2], o[3]);
            }
        }
    }
}

template <int WT, int C, int NXS, int P, int NWC>
__global__ __launch_bounds__(256, 3) void xt_kernel(XT_PARAMS) { XT_HOT; xt_tile<WT, C, NXS, P, NWC>(hot, a, (int)blockIdx.y * C); }
// Tiles of four activation groups and, behind them in the grid, one of the R groups that remain: the sums of groups that do not exist cost as much
// as those of groups that do (22016 x 4096 Q4_0: 77 rows 98 -> 85 us, 140 rows 161 -> 135, 200 rows 224 -> 188, 900 rows 831 -> 796)
template <int WT, int R>
__global__ __launch_bounds__(256, 3) void xt_mixed_kernel(XT_PARAMS) {
    XT_HOT;
    const int full = a.ncg / 4;
    if ((int)blockIdx.y < full) xt_tile<WT, 4, 2, 1, 2>(hot, a, (int)blockIdx.y * 4);
    else xt_tile<WT, R, R < 3 ? 4 : 2, R < 3 ? 2 : 1, 2>(hot, a, full * 4);
}

// Few activation rows: one group of them and 16 weight rows per workgroup, the accumulators of the tile over its four waves (words 2g, 2g + 1 to wave g).
// With a wave or two on a SIMD what bounds it is the chain barrier, LDS read, unpack, matrix instruction, fmas: it is walked once per chunk of eight
// blocks, and the operands of the next chunk are read from LDS before the fmas of this one.  NS: LDS slots for chunks, all of them on their way: four where
// a compute unit has one or two workgroups, whose weights come from memory (two: 20 % slower there); two, 24 KB, where it has more (four: up to
// 20 % slower).  32 weight rows and eight waves per workgroup: 30 % slower with 4096.  From four workgroups on a compute unit the tiles of 32 rows are faster (xt_choose).
// Against one stage of four blocks per barrier, weights from memory, in us, packing of the activations (4 us) included: 8 rows, Q4_0 4096 x 4096 14.4 -> 12.1,
// 4096 x 11008 30.6 -> 23.6, 12288 x 4096 21.0 -> 17.7, Q8_0 14.4 -> 12.5, 30.3 -> 24.3, 22.5 -> 20.8; 48 rows, Q4_0 4096 x 4096 21.2 -> 17.8, 4096 x 11008 47.5 -> 37.3.
template <int WT, int NS>
__global__ __launch_bounds__(256, 2) void xn_kernel(xt_args a) {
    constexpr int NT = 256, ROWS = 16, CU = xt_w<WT>::CU, UW = ROWS * CU, NI = (UW + NT - 1) / NT, NXI = 2;
    constexpr int XB = 2 * (XT_XB + 256), WB = (UW + 63) / 64 * 1024, NREQ = NXI + 1 + NI;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = wave, q = lane >> 4, r = lane & 15;
    const int mat = (int)blockIdx.x / a.tiles, m0 = ((int)blockIdx.x - mat * a.tiles) * ROWS, cg = (int)blockIdx.y;
    const int nch = a.nst / 2, M = a.M;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)smem;
    // requests as in xt_tile: uniform bases that advance by a chunk, per-lane offsets that stay; waves 0 and 1 bring the scales of the chunk's stages (the others repeat them)
    const uint8_t *bx = a.xq + (int64_t)cg * a.nst * XT_XB + wave * 1024, *bd = a.xd + ((int64_t)cg * a.nst + min(wave, 1)) * XT_XD, *bw = a.w[mat] + (int64_t)m0 * a.w_row;
    uint32_t ow[NI];
#pragma unroll
    for (int i = 0; i < NI; i++) {
        const int u = min(tid + i * NT, UW - 1);
        ow[i] = (uint32_t)(min(m0 + u / CU, M - 1) - m0) * (uint32_t)a.w_row + (u % CU) * 16;
    }
    const bool spare = wave * 64 + (NI - 1) * NT >= UW;
    const uint32_t lds_spare = __builtin_amdgcn_readfirstlane(lds0 + NS * (XB + WB));
    const uint32_t l16 = lane * 16, l4 = lane * 4;
    const uint32_t ldsx = __builtin_amdgcn_readfirstlane(lds0 + wave * 1024), ldsd = __builtin_amdgcn_readfirstlane(lds0 + 2 * XT_XB + min(wave, 1) * 256),
                   ldsw = __builtin_amdgcn_readfirstlane(lds0 + NS * XB + wave * 1024);
    int is = 0;                                    // next chunk to request; past the last one it is requested again (same count of requests, slot unused)
    auto issue = [&]() {
        const uint32_t slot = is & (NS - 1);
        const int adv = is + 1 < nch ? 1 : 0;
#pragma unroll
        for (int i = 0; i < NI; i++) xt_dma16(bw, ow[i], i == NI - 1 && spare ? lds_spare : ldsw + slot * WB + i * NT * 16);
#pragma unroll
        for (int i = 0; i < NXI; i++) xt_dma16(bx + i * NT * 16, l16, ldsx + slot * XB + i * NT * 16);
        xt_dma4(bd, l4, ldsd + slot * XB);
        bw += adv * xt_w<WT>::CB;
        bx += adv * 2 * XT_XB;
        bd += adv * 2 * XT_XD;
        is++;
    };
#pragma unroll
    for (int s = 0; s < NS; s++) issue();

    float acc[8];                                  // [word 2g, 2g + 1][weight rows 4q .. 4q + 3], activation row r
#pragma unroll
    for (int i = 0; i < 8; i++) acc[i] = 0.0f;
    // Where a lane finds its operands: lane block q holds word 2g + (q & 1) of block 2i + (q >> 1), so one instruction takes two blocks.  A Q4_0 block holds
    // words 0..3 in the low nibbles and 4..7 in the high nibbles of its four quant dwords (which start at byte 2: blocks at odd dword halves are read as two dwords).
    constexpr bool Q4 = WT == SPY_HIP_Q4_0;
    constexpr int PD = xt_w<WT>::PD, OD = Q4 ? 5 : 9, BB = xt_w<WT>::BB;
    const int odd = q >> 1;
    const uint32_t wbase = r * xt_w<WT>::CB + 4 * (odd * OD + (q & 1) + (Q4 ? 2 * (g & 1) : 2 * g));
    const uint32_t al = odd ? 0 : 16;
    const int sh = Q4 ? 4 * (g >> 1) : 0;
    const uint32_t dbase = r * xt_w<WT>::CB + q * BB, xbase = odd * 1024 + g * 256 + r * 16 + (q & 1) * 8;
    const uint32_t c64 = 0x64006400u;
    struct operands { uint32_t w0[4], w1[4], dw[2], dx[2]; uint2 x[4]; };
    auto read = [&](int s, operands &o) {
        const uint8_t *sx = smem + (s & (NS - 1)) * XB, *sw = smem + NS * XB + (s & (NS - 1)) * WB;
        const uint32_t *b = (const uint32_t *)(sw + wbase);
#pragma unroll
        for (int i = 0; i < 4; i++) { o.w0[i] = b[PD * i]; o.w1[i] = b[PD * i + 1]; }
#pragma unroll
        for (int h = 0; h < 2; h++) {
            o.dw[h] = *(const uint16_t *)(sw + dbase + h * 4 * BB);
            o.dx[h] = *(const uint32_t *)(sx + 2 * XT_XB + h * 256 + lane * 4);
        }
#pragma unroll
        for (int i = 0; i < 4; i++) o.x[i] = *(const uint2 *)(sx + i * 2048 + xbase);
    };
    auto compute = [&](const operands &o) {
        uint32_t wa[4], wb[4], dw[2];
#pragma unroll
        for (int i = 0; i < 4; i++) {                               // elements 0, 2 and 1, 3 of the word
            const uint32_t v = __builtin_amdgcn_alignbit(o.w1[i], o.w0[i], al);
            if constexpr (Q4) {
                wa[i] = xt_sub(xt_and_or(v >> sh, 0x000F000Fu, c64), 0x64086408u);
                wb[i] = xt_sub(xt_and_or(v >> (sh + 8), 0x000F000Fu, c64), 0x64086408u);
            } else {
                const uint32_t t = v ^ 0x80808080u;
                wa[i] = xt_sub(xt_and_or(t, 0x00FF00FFu, c64), 0x64806480u);
                wb[i] = xt_sub(xt_and_or(t >> 8, 0x00FF00FFu, c64), 0x64806480u);
            }
        }
#pragma unroll
        for (int h = 0; h < 2; h++) dw[h] = o.dw[h] == 0xFFFFu ? 0u : o.dw[h];         // conversion.h:39-41: the host's table has no entry for 0xFFFF
        // the matrix instruction of step j + 1 before the fmas on the result of step j
        xt_v16f p[2], D[2];
        D[0] = xt_mfma(dw[0], 0u, o.dx[0], 0u);
        p[0] = xt_mfma(wa[0], wb[0], o.x[0].x, o.x[0].y);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            if (j == 1) D[1] = xt_mfma(dw[1], 0u, o.dx[1], 0u);
            if (j < 3) p[(j + 1) & 1] = xt_mfma(wa[j + 1], wb[j + 1], o.x[j + 1].x, o.x[j + 1].y);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int b = 0; b < 2; b++)
#pragma unroll
                for (int n = 0; n < 8; n++) acc[n] = fmaf(D[j >> 1][4 * (2 * (j & 1) + b) + (n & 3)], p[j & 1][8 * b + n], acc[n]);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    operands A, B;
    xt_wait_vm<(NS - 1) * NREQ>();
    __builtin_amdgcn_s_barrier();
    read(0, A);
    auto body = [&](int s, operands &now, operands &next) {
        xt_wait_vm<(NS - 2) * NREQ>();             // chunk s + 1 is there (the requests of the NS - 2 chunks after it may be on their way), and this wave has read chunk s
        __builtin_amdgcn_s_barrier();
        issue();                                   // chunk s + NS, where chunk s was
        read(s + 1, next);                         // (past the last chunk: what the slot holds, not used)
        __builtin_amdgcn_sched_barrier(0);
        compute(now);
    };
    int s = 0;
    for (; s + 2 <= nch; s += 2) { body(s, A, B); body(s + 1, B, A); }
    if (s < nch) body(s, A, B);
    xt_wait_vm<0>();
    __builtin_amdgcn_s_barrier();
    // hsum_float_8, as in xt_tile
    float *ex = (float *)smem;
    if (g > 0) {
#pragma unroll
        for (int n = 0; n < 8; n++) ex[((g - 1) * 8 + n) * 64 + lane] = acc[n];
    }
    __syncthreads();
    if (g > 0) return;
    const int row = m0 + 4 * q, t = cg * 16 + r;
    float o[4];
#pragma unroll
    for (int v = 0; v < 4; v++) {
        float rr[4];
#pragma unroll
        for (int k = 0; k < 2; k++) {
            rr[k] = ex[(8 + 4 * k + v) * 64 + lane] + acc[4 * k + v];
            rr[2 + k] = ex[(16 + 4 * k + v) * 64 + lane] + ex[(4 * k + v) * 64 + lane];
        }
        const float s0 = rr[0] + rr[2], s1 = rr[1] + rr[3];
        o[v] = s0 + s1;
    }
    if (t < a.T && row + 3 < M) {
        const int64_t at = (int64_t)t * a.d_row + row;
        if (a.resid) { const float4 z = *(const float4 *)(a.resid + at); o[0] += z.x; o[1] += z.y; o[2] += z.z; o[3] += z.w; }
        *(float4 *)(a.dst[mat] + at) = make_float4(o[0], o[1], o[2], o[3]);
    }
}
template <int WT, int NS>
int xn_launch(hipStream_t st, xt_args a, int nmat) {
    constexpr size_t lds = NS * (2 * (XT_XB + 256) + (16 * xt_w<WT>::CU + 63) / 64 * 1024) + 1024;
    static_assert(lds <= 64 * 1024 && lds >= 3 * 8 * 256, "no raised LDS limit; room for the exchange of the accumulators");
    a.tiles = (a.M + 15) / 16;
    xn_kernel<WT, NS><<<dim3((unsigned)(a.tiles * nmat), (unsigned)a.ncg), dim3(256), lds, st>>>(a);
    return SPY_LAUNCH_RC();
}

// f32 rows -> packed activations.  Rows past T become zeros.  8 lanes per block; a workgroup takes 16 rows and two blocks.
__global__ __launch_bounds__(256) void xt_pack_kernel(const uint8_t *__restrict__ x, int64_t x_stride, int T, int nst, uint8_t *__restrict__ xq, uint8_t *__restrict__ xd) {
    const int tid = threadIdx.x, e = tid & 7, c = (tid >> 3) & 15, b = (int)blockIdx.x * 2 + (tid >> 7), cg = blockIdx.y;
    const int t = cg * 16 + c;
    float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (t < T) v = *(const float4 *)(x + (int64_t)t * x_stride + (b * 32 + e * 4) * 4);
    xt_store4(v, cg, nst, b, c, e, xq, xd);
}

// ---- producers: the operators in front of a MatMul, ending in its packed activations, in the host's order ---------------------------------
// Two words (eight elements) per lane, four lanes per block: quantize and store.  xq, xd: the bases of the lane's block for activation row 0 of the group
__device__ __forceinline__ void xt_store8(const float (&y)[8], int sub, uint8_t *xq, uint8_t *xd, int row) {
    float amax = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; i++) amax = fmaxf(amax, fabsf(y[i]));
    amax = fmaxf(amax, __shfl_xor(amax, 1, SPY_WAVE));
    amax = fmaxf(amax, __shfl_xor(amax, 2, SPY_WAVE));
    const float d = amax / 127.0f, id = (amax != 0.0f) ? 127.0f / amax : 0.0f;
    int sum = 0;
    uint32_t h[8];
#pragma unroll
    for (int i = 0; i < 8; i++) {
        int q = (int)rintf(y[i] * id);
        q = q < -128 ? -128 : (q > 127 ? 127 : q);
        sum += q;
        h[i] = __builtin_bit_cast(uint16_t, (_Float16)(float)q);
    }
    sum += __shfl_xor(sum, 1, SPY_WAVE);
    sum += __shfl_xor(sum, 2, SPY_WAVE);
    *(uint4 *)(xq + sub * 256 + row * 16) = make_uint4(h[0] | (h[2] << 16), h[1] | (h[3] << 16), h[4] | (h[6] << 16), h[5] | (h[7] << 16));
    if (sub == 0) {
        *(uint32_t *)(xd + row * 4) = f2h(d);
        *(float *)(xd + 256 + row * 4) = (float)sum;
    }
}

// NormRMS (non-linear.cpp:194-223) -> Mul by the norm weights -> packed activations; one workgroup per row.  The sum of squares is the host's
// std::transform_reduce: groups of four, (x0^2 + x1^2) + (x2^2 + x3^2), added to one running sum (xg_segment_sum).  Rows past T of the last
// group are written as zeros.  OWN: the sum in this backend's own order, by the thread pattern of norm_rms_kernel, from a copy of the row in LDS.
template <int NV, bool OWN>        // K <= 2048 * NV
__global__ __launch_bounds__(256) void xt_norm_pack_kernel(const float *__restrict__ x, const float *__restrict__ w, float eps, int K, int T, int nst,
                                                           uint8_t *__restrict__ xq, uint8_t *__restrict__ xd) {
    __shared__ __align__(16) float g[OWN ? 2048 * NV : 640 * NV];      // OWN: the row; else the group sums as xg_segment_sum reads them
    __shared__ float s_sum;
    // the 16 rows of a group write pieces of the same lines: consecutive workgroups go to the eight XCDs in turn, so every eighth one is of the same group and
    // the pieces meet in one L2 (rows in the order of the workgroups: 2048 rows of 4096 25.0 -> 18.4 us, 77 rows 6.6 -> 5.6; OWN, 1000 rows, 11.9 -> 9.1)
    const int tid = threadIdx.x, cg = (int)(blockIdx.x >> 7) * 8 + (blockIdx.x & 7), row = (blockIdx.x >> 3) & 15, t = cg * 16 + row, n8 = K / 8;
    if (cg * 16 >= T) return;
    const float4 *xr = (const float4 *)(x + (int64_t)min(t, T - 1) * K);
    float4 v[NV][2], wv[NV][2];
#pragma unroll
    for (int j = 0; j < NV; j++) {
        const int i = min(j * 256 + tid, n8 - 1);
        v[j][0] = xr[2 * i]; v[j][1] = xr[2 * i + 1];
    }
#pragma unroll
    for (int j = 0; j < NV; j++) {
        const int i = min(j * 256 + tid, n8 - 1);
        wv[j][0] = ((const float4 *)w)[2 * i]; wv[j][1] = ((const float4 *)w)[2 * i + 1];
        if (j * 256 + tid < n8) {
#pragma unroll
            for (int k = 0; k < 2; k++) {
                const float4 z = v[j][k];
                if constexpr (OWN) ((float4 *)g)[2 * i + k] = z;
                else {
                    const float a0 = z.x * z.x, a1 = z.y * z.y, a2 = z.z * z.z, a3 = z.w * z.w, v1 = a0 + a1, v2 = a2 + a3;
                    g[xg_seg_at(2 * i + k)] = v1 + v2;               // K / 4 is a multiple of 64: no segment is left open
                }
            }
        }
    }
    __syncthreads();
    if constexpr (OWN) {
        __shared__ float part[4];
        float acc = 0.0f;
        for (int i = tid; i < K; i += 256) acc = fmaf(g[i], g[i], acc);
        acc = wave_sum(acc);
        if ((tid & 63) == 0) part[tid >> 6] = acc;
        __syncthreads();
        if (tid == 0) s_sum = (part[0] + part[1]) + (part[2] + part[3]);
    } else if (tid < 64) {
        const float sum = xg_segment_sum<NV / 2>(g, K / 4);
        if (tid == 0) s_sum = sum;
    }
    __syncthreads();
    const float mean = s_sum / (float)K, scale = 1.0f / sqrtf(mean + eps);
#pragma unroll
    for (int j = 0; j < NV; j++) {
        const int i = j * 256 + tid;
        if (i < n8) {                                                // n8 is a multiple of 32: the four lanes of a block stay together
            const float4 w0 = wv[j][0], w1 = wv[j][1], v0 = v[j][0], v1 = v[j][1];
            float y[8] = {(v0.x * scale) * w0.x, (v0.y * scale) * w0.y, (v0.z * scale) * w0.z, (v0.w * scale) * w0.w,
                          (v1.x * scale) * w1.x, (v1.y * scale) * w1.y, (v1.z * scale) * w1.z, (v1.w * scale) * w1.w};
            if (t >= T) {
#pragma unroll
                for (int k = 0; k < 8; k++) y[k] = 0.0f;
            }
            const int b = i >> 2;
            xt_store8(y, i & 3, xq + ((int64_t)cg * nst + (b >> 2)) * XT_XB + (b & 3) * 1024, xd + ((int64_t)cg * nst + (b >> 2)) * XT_XD + (b & 3) * 64, row);
        }
    }
}

// Silu by the host's table (lut == nullptr: of this backend, v / (1 + exp(-v)) of the fp16-rounded argument) -> Mul (up * silu(gate)) -> packed
// activations (non-linear.cpp:11-14,57-77); a workgroup takes 16 rows and four blocks
__global__ __launch_bounds__(256) void xt_silu_pack_kernel(const float *__restrict__ gate, const float *__restrict__ up, const float *__restrict__ lut, int F, int T, int nst,
                                                           uint8_t *__restrict__ xq, uint8_t *__restrict__ xd) {
    const int tid = threadIdx.x, sub = tid & 3, bl = (tid >> 2) & 3, row = tid >> 4, b = (int)blockIdx.x * 4 + bl, cg = blockIdx.y, t = cg * 16 + row;
    float y[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    if (t < T) {
        const int64_t at = (int64_t)t * F + b * 32 + sub * 8;
        const float4 g0 = *(const float4 *)(gate + at), g1 = *(const float4 *)(gate + at + 4), u0 = *(const float4 *)(up + at), u1 = *(const float4 *)(up + at + 4);
        const float ga[8] = {g0.x, g0.y, g0.z, g0.w, g1.x, g1.y, g1.z, g1.w}, ua[8] = {u0.x, u0.y, u0.z, u0.w, u1.x, u1.y, u1.z, u1.w};
#pragma unroll
        for (int k = 0; k < 8; k++) {
            float sl;
            if (lut) sl = lut[65536 + f2h(ga[k])];
            else { const float v = h2f(f2h(ga[k])); sl = v / (1.0f + expf(-v)); }
            y[k] = ua[k] * sl;
        }
    }
    xt_store8(y, sub, xq + ((int64_t)cg * nst + blockIdx.x) * XT_XB + bl * 1024, xd + ((int64_t)cg * nst + blockIdx.x) * XT_XD + bl * 64, row);
}

// The same for many rows by the host's table, whose entries for 2^-11 <= |v| < 32 a workgroup of 1024 threads keeps in LDS: a gather of 64 entries takes the compute
// unit's address unit 64 cycles from memory and an LDS read of them about ten.  A thread's next operands are on their way while it works on these.
// F = 11008, operands from memory: 2048 rows 95.4 -> 46.3 us (4.9 TB/s), 512 rows 25.5 -> 16.1.  The 128 KB of table are 3 us: 150 rows (3.4 groups of four blocks
// per compute unit) 8.6 -> 7.4, 77 rows (1.7) 5.0 -> 6.9, hence the line at three.
constexpr uint32_t SL_LO = 0x1000, SL_N = 0x4000;                                // fp16 patterns without the sign
__global__ __launch_bounds__(1024) void xt_silu_pack_many_kernel(const float *__restrict__ gate, const float *__restrict__ up, const float *__restrict__ lut, int F, int T, int nst, int tiles,
                                                                 uint8_t *__restrict__ xq, uint8_t *__restrict__ xd) {
    extern __shared__ __attribute__((aligned(16))) float s_silu[];                // [sign][SL_N]
    const int tid = threadIdx.x, sub = tid & 3, bl = (tid >> 2) & 3, row = (tid >> 4) & 15, step = (int)gridDim.x * 4;
    int tile = (int)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(tid >> 8);
    float4 n[4];
    auto fetch = [&](int i) {
        const int cg = i / nst, b = (i - cg * nst) * 4 + bl;
        const int64_t at = (int64_t)min(cg * 16 + row, T - 1) * F + b * 32 + sub * 8;
        n[0] = *(const float4 *)(gate + at); n[1] = *(const float4 *)(gate + at + 4); n[2] = *(const float4 *)(up + at); n[3] = *(const float4 *)(up + at + 4);
    };
    fetch(min(tile, tiles - 1));
#pragma unroll
    for (int k = 0; k < (int)SL_N / 2048; k++) {
        const int i = k * 1024 + tid, neg = i >= (int)SL_N / 4;
        ((float4 *)s_silu)[i] = ((const float4 *)(lut + 65536 + neg * 0x8000 + SL_LO))[i - neg * (int)(SL_N / 4)];
    }
    __syncthreads();
    for (; tile < tiles; tile += step) {
        const float ga[8] = {n[0].x, n[0].y, n[0].z, n[0].w, n[1].x, n[1].y, n[1].z, n[1].w}, ua[8] = {n[2].x, n[2].y, n[2].z, n[2].w, n[3].x, n[3].y, n[3].z, n[3].w};
        fetch(min(tile + step, tiles - 1));
        const int cg = tile / nst, st = tile - cg * nst;
        const bool in = cg * 16 + row < T;
        float y[8];
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const uint32_t h = f2h(ga[k]), m = (h & 0x7FFFu) - SL_LO;
            float sl = s_silu[(h >> 15) * SL_N + min(m, SL_N - 1)];
            if (m >= SL_N) sl = lut[65536 + h];
            y[k] = in ? ua[k] * sl : 0.0f;
        }
        xt_store8(y, sub, xq + ((int64_t)cg * nst + st) * XT_XB + bl * 1024, xd + ((int64_t)cg * nst + st) * XT_XD + bl * 64, row);
    }
}

template <int WT, int C, int NXS, int NWC> constexpr size_t xt_lds() {
    constexpr size_t ring = NXS * C * (XT_XB + 256) + NWC * ((32 * xt_w<WT>::CU + 63) / 64) * 1024, ex = (size_t)2 * C * 16 * 256, lds = ring > ex ? ring : ex;
    static_assert(lds <= 64 * 1024, "no raised LDS limit");
    return lds;
}
template <int WT, int C, int NXS, int P, int NWC>
int xt_launch(hipStream_t st, xt_args a, int nmat) {
    a.tiles = (a.M + 31) / 32;
    xt_kernel<WT, C, NXS, P, NWC><<<dim3((unsigned)(a.tiles * nmat), (unsigned)((a.ncg + C - 1) / C)), dim3(256), xt_lds<WT, C, NXS, NWC>(), st>>>(XT_ARGS(a));
    return SPY_LAUNCH_RC();
}
template <int WT, int R>
int xt_launch_mixed(hipStream_t st, xt_args a, int nmat) {
    a.tiles = (a.M + 31) / 32;
    constexpr size_t l4 = xt_lds<WT, 4, 2, 2>(), lr = xt_lds<WT, R, R < 3 ? 4 : 2, 2>();
    xt_mixed_kernel<WT, R><<<dim3((unsigned)(a.tiles * nmat), (unsigned)(a.ncg / 4 + 1)), dim3(256), l4 > lr ? l4 : lr, st>>>(XT_ARGS(a));
    return SPY_LAUNCH_RC();
}

// ---- Q4_K / Q6_K ------------------------------------------------------------------------------------------------------------------------
// These dots keep ONE accumulator per output and add one term per sub-block of 32 elements (the order this project defines; exact_order.hip):
//   Q4_K:  acc = fma(d_x, d * float(sc * isum) - dmin * float(m * bsum), acc)       Q6_K:  acc = fma(d_x * d, float(sc0 * isum0 + sc1 * isum1), acc)
// so the integer sums of a whole sub-block come from v_mfma_f32_16x16x32_f16 -- lane (q, r): elements 8q .. 8q + 7 of row r -- and the outer products of a
// term (Q4_K dmin * m by bsum, Q6_K d by d_x) for two sub-blocks and two groups of activation rows from one instruction of four blocks (v_mfma_f32_16x16x1_4b_f32,
// whose single product rounds once as the multiplication does, and v_mfma_f32_16x16x4_4b_f16, exact).  Left for the vector units are 12 (Q4_K) or 4 (Q6_K)
// instructions per 16 x 16 tile and sub-block where the tile kernel of exact_order.hip had 64 and 56:
//   * small integers are fp16 subnormals as they are (the bit pattern n is n * 2^-24): unpacking a pair of nibbles is one AND.  The factor
//     2^24 goes into the weights' scale; every product and sum below is still exact.
//   * d * sc, dmin * m and d_w * d_x have at most 22 significant bits: they are exact in fp32, so (d * sc) * isum rounds once, as d * (sc * isum) does.
//   * Q6_K: q - 32 = l + 16 (h - 2) with the low four and the high two bits, and sc * l, 16 * sc * (h - 2) are exact in fp16: the scales of the
//     two halves of a sub-block ride on the operands, and two matrix instructions leave sc0 * isum0 + sc1 * isum1 (below 2^24).
//   * Q6_K: the 2^24 stays out until the end: accumulators are multiples of 2^-72, so no sum below it is rounded otherwise.
// A wave takes 16 weight rows, which it reads straight into registers half a super-block ahead, and C groups of 16 activation rows.
// 4096 x 4096 x 2048, quantization and packing included: Q4_K 374 -> 150 us, Q6_K 346 -> 146; 77 rows 89 -> 28 and 89 -> 35.  Vector and matrix cycles bound both and
// hardly overlap: per super-block of 16 rows x 8 groups 845 vector instructions (768 of them the terms) of 4 cycles beside 1536 matrix cycles (Q4_K), 440 beside 2560 (Q6_K).
// The outer products on the matrix units and the halves of a super-block in turn (no second copy of it in registers) against 16 and 8 vector instructions
// per tile and sub-block: 22016 x 4096 x 2048 Q4_K 767 -> 730 us, 4096 x 11008 x 2048 Q6_K 445 -> 394, 300 rows 197 -> 156.
typedef _Float16 xk_h8 __attribute__((ext_vector_type(8)));
typedef float xk_v4f __attribute__((ext_vector_type(4)));

__device__ __forceinline__ xk_v4f xk_mfma(const uint4 &a, const uint4 &b, const xk_v4f &c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(xk_h8, a), __builtin_bit_cast(xk_h8, b), c, 0, 0, 0);
}
__device__ __forceinline__ uint32_t xk_pk_mul(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(xt_h2, a) * __builtin_bit_cast(xt_h2, b));
}
__device__ __forceinline__ uint32_t xk_pk_fma(uint32_t a, uint32_t b, uint32_t c) {
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(__builtin_bit_cast(xt_h2, a), __builtin_bit_cast(xt_h2, b), __builtin_bit_cast(xt_h2, c)));
}
typedef uint32_t xk_u2 __attribute__((ext_vector_type(2), aligned(2)));
typedef uint32_t xk_u4 __attribute__((ext_vector_type(4), aligned(2)));

// the raw super-block of a lane's weight row: its quants and the row's scales
template <int WT> struct xk_raw;
template <> struct xk_raw<SPY_HIP_Q4_K> { uint2 qs[4]; uint4 head; };
template <> struct xk_raw<SPY_HIP_Q6_K> { uint2 ql[4], qh[2]; uint4 sc; uint32_t d; };

template <int WT>
__device__ __forceinline__ xk_raw<WT> xk_load(const uint8_t *row, int sb, int q) {
    xk_raw<WT> t;
    if constexpr (WT == SPY_HIP_Q4_K) {
        const uint8_t *p = row + (int64_t)sb * 144;
        t.head = *(const uint4 *)p;
#pragma unroll
        for (int k = 0; k < 4; k++) t.qs[k] = *(const uint2 *)(p + 16 + 32 * k + 8 * q);
    } else {                                                         // super-blocks of 210 bytes: two-byte alignment
        const uint8_t *p = row + (int64_t)sb * 210;
#pragma unroll
        for (int k = 0; k < 4; k++) t.ql[k] = __builtin_bit_cast(uint2, *(const xk_u2 *)(p + 32 * k + 8 * q));
#pragma unroll
        for (int k = 0; k < 2; k++) t.qh[k] = __builtin_bit_cast(uint2, *(const xk_u2 *)(p + 128 + 32 * k + 8 * q));
        t.sc = __builtin_bit_cast(uint4, *(const xk_u4 *)(p + 192));
        t.d = *(const uint16_t *)(p + 208);
    }
    return t;
}
// half H of a super-block, what stage H of its two takes, and of the first half the scales
template <int H> __device__ __forceinline__ void xk_load_half(xk_raw<SPY_HIP_Q4_K> &t, const uint8_t *row, int sb, int q) {
    const uint8_t *p = row + (int64_t)sb * 144;
    if constexpr (H == 0) t.head = *(const uint4 *)p;
#pragma unroll
    for (int k = 2 * H; k < 2 * H + 2; k++) t.qs[k] = *(const uint2 *)(p + 16 + 32 * k + 8 * q);
}
template <int H> __device__ __forceinline__ void xk_load_half(xk_raw<SPY_HIP_Q6_K> &t, const uint8_t *row, int sb, int q) {
    const uint8_t *p = row + (int64_t)sb * 210;
#pragma unroll
    for (int k = 2 * H; k < 2 * H + 2; k++) t.ql[k] = __builtin_bit_cast(uint2, *(const xk_u2 *)(p + 32 * k + 8 * q));
    t.qh[H] = __builtin_bit_cast(uint2, *(const xk_u2 *)(p + 128 + 32 * H + 8 * q));
    const uint2 sc = __builtin_bit_cast(uint2, *(const xk_u2 *)(p + 192 + 8 * H));
    if constexpr (H == 0) { t.sc.x = sc.x; t.sc.y = sc.y; t.d = *(const uint16_t *)(p + 208); }
    else { t.sc.z = sc.x; t.sc.w = sc.y; }
}
// the compiler's wait for half H stands where this does
template <int H, int WT> __device__ __forceinline__ void xk_arrived(xk_raw<WT> &t) {
#if defined(__HIP_DEVICE_COMPILE__)
    if constexpr (WT == SPY_HIP_Q4_K) {
        asm volatile("" : "+v"(t.qs[2 * H].x), "+v"(t.qs[2 * H].y), "+v"(t.qs[2 * H + 1].x), "+v"(t.qs[2 * H + 1].y));
        if constexpr (H == 0) asm volatile("" : "+v"(t.head.x), "+v"(t.head.y), "+v"(t.head.z), "+v"(t.head.w));
    } else {
        asm volatile("" : "+v"(t.ql[2 * H].x), "+v"(t.ql[2 * H].y), "+v"(t.ql[2 * H + 1].x), "+v"(t.ql[2 * H + 1].y), "+v"(t.qh[H].x), "+v"(t.qh[H].y));
        if constexpr (H == 0) asm volatile("" : "+v"(t.sc.x), "+v"(t.sc.y), "+v"(t.d));
        else asm volatile("" : "+v"(t.sc.z), "+v"(t.sc.w));
    }
#endif
}
__device__ __forceinline__ float xk_half(uint32_t h) { return h == 0xFFFFu ? 0.0f : h2f((uint16_t)h); }      // conversion.h:39-41
// The scales of a super-block into the wave's table: lane (q, r) prepares those of row r, sub-blocks 2q and 2q + 1.
// Q4_K: [sub-block][d * sc | dmin * m][row]; Q6_K: [row] d
template <int WT>
__device__ __forceinline__ void xk_put_scales(const xk_raw<WT> &w, float *tab, int q, int r) {
    if constexpr (WT == SPY_HIP_Q4_K) {
        const float d = xk_half(w.head.x & 0xFFFFu), dmin = xk_half(w.head.x >> 16);
        const int s16 = 16 * (q & 1);
        const uint32_t t0 = w.head.y >> s16, t1 = w.head.z >> s16, t2 = w.head.w >> s16;      // bytes 2q, 2q + 1 (mod 4) of scales[0..3], [4..7], [8..11]
        const bool hi = q >= 2;                                                               // get_scale_min_k4 for sub-blocks 4 .. 7
        const uint32_t sc = hi ? (t2 & 0x0F0Fu) | ((t0 >> 2) & 0x3030u) : t0 & 0x3F3Fu, mm = hi ? ((t2 >> 4) & 0x0F0Fu) | ((t1 >> 2) & 0x3030u) : t1 & 0x3F3Fu;
        float *o = tab + 2 * q * 32 + r;
        o[0] = (d * 16777216.0f) * (float)(sc & 0xFFu);                 // low nibbles: n * 2^-24
        o[16] = dmin * (float)(mm & 0xFFu);
        o[32] = (d * 1048576.0f) * (float)((sc >> 8) & 0xFFu);          // high nibbles stay where they are: n * 2^-20
        o[48] = dmin * (float)((mm >> 8) & 0xFFu);
    } else if (q == 0) tab[r] = xk_half(w.d) * 16777216.0f;
    __builtin_amdgcn_wave_barrier();                                    // other lanes of the wave read them
    asm volatile("" ::: "memory");
}
// Q4_K in the own order: [sub-block][row] sc as a pair of fp16 (times 2^10 / 2^6: the product with a nibble is n * sc * 2^-14), [sub-block][row] m, [row] d * 2^14, [row] -dmin
__device__ __forceinline__ void xk_put_scales_own(const xk_raw<SPY_HIP_Q4_K> &w, float *tab, int q, int r) {
    const int s16 = 16 * (q & 1);
    const uint32_t t0 = w.head.y >> s16, t1 = w.head.z >> s16, t2 = w.head.w >> s16;
    const bool hi = q >= 2;
    const uint32_t sc = hi ? (t2 & 0x0F0Fu) | ((t0 >> 2) & 0x3030u) : t0 & 0x3F3Fu, mm = hi ? ((t2 >> 4) & 0x0F0Fu) | ((t1 >> 2) & 0x3030u) : t1 & 0x3F3Fu;
    const _Float16 s0 = (_Float16)(float)((sc & 0xFFu) << 10), s1 = (_Float16)(float)((sc >> 8 & 0xFFu) << 6);
    const xt_h2 p0 = {s0, s0}, p1 = {s1, s1};
    uint32_t *o = (uint32_t *)tab + 2 * q * 16 + r;
    o[0] = __builtin_bit_cast(uint32_t, p0);
    o[16] = __builtin_bit_cast(uint32_t, p1);
    tab[128 + 2 * q * 16 + r] = (float)(mm & 0xFFu);
    tab[128 + (2 * q + 1) * 16 + r] = (float)((mm >> 8) & 0xFFu);
    if (q == 0) tab[256 + r] = xk_half(w.head.x & 0xFFFFu) * 16384.0f;
    if (q == 1) tab[272 + r] = -xk_half(w.head.x >> 16);
    __builtin_amdgcn_wave_barrier();
    asm volatile("" ::: "memory");
}
// operand(s) of sub-block t of the super-block
template <int WT, int t>
__device__ __forceinline__ void xk_unpack(const xk_raw<WT> &w, int q, uint4 (&o)[WT == SPY_HIP_Q4_K ? 1 : 2]) {
    if constexpr (WT == SPY_HIP_Q4_K) {
        const uint2 v = w.qs[t >> 1];
        constexpr uint32_t m = t & 1 ? 0x00F000F0u : 0x000F000Fu;
        o[0] = make_uint4(v.x & m, (v.x >> 8) & m, v.y & m, (v.y >> 8) & m);
    } else {
        constexpr int n = t >> 2, grp = t & 3;
        const uint2 l = w.ql[2 * n + (grp & 1)], h = w.qh[n];
        const uint32_t scw = t < 2 ? w.sc.x : t < 4 ? w.sc.y : t < 6 ? w.sc.z : w.sc.w;
        const int sci = (int)(int8_t)(scw >> (16 * (t & 1) + 8 * (q >> 1)));                        // the scale of this lane's half of the sub-block
        const xt_h2 s2 = {(_Float16)(short)sci, (_Float16)(short)sci};
        constexpr uint32_t up[4] = {0x4C004C00u, 0x44004400u, 0x3C003C00u, 0x34003400u};            // 16 / 4^grp: the high pair of bits is taken where it stands
        const uint32_t s = __builtin_bit_cast(uint32_t, s2), sl = grp >> 1 ? xk_pk_mul(s, 0x2C002C00u) : s, sh = xk_pk_mul(s, up[grp]), sm = xk_pk_mul(s, 0x80208020u);
        constexpr uint32_t ml = grp >> 1 ? 0x00F000F0u : 0x000F000Fu, mh = 0x00030003u << (2 * grp);
        uint32_t lo[4], hh[4];
        const uint32_t w2[2] = {l.x, l.y}, h2[2] = {h.x, h.y};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            lo[i] = xk_pk_mul((w2[i >> 1] >> (8 * (i & 1))) & ml, sl);
            hh[i] = xk_pk_fma((h2[i >> 1] >> (8 * (i & 1))) & mh, sh, sm);
        }
        o[0] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
        o[1] = make_uint4(hh[0], hh[1], hh[2], hh[3]);
    }
}

// OWN: this backend's own order.  The terms of a super-block are added before its d and dmin are applied:
//   acc = acc + d * (sum d_x * (sc * isum)) - dmin * (sum m * (d_x * bsum))
// with sc on the weights' operand and the second sum, a contraction over sub-blocks, on v_mfma_f32_16x16x4_f32: 5 vector instructions per tile and
// sub-block instead of 17 (Q4_K) and 9 (Q6_K) before the outer products of the host's order went to the matrix units.  4096 x 4096 x 1000, packing included: Q4_K 105 -> 87 us, Q6_K 112 -> 97; 22016 x 4096 x 1000: 557 -> 355
// and 588 -> 449 (the 128 x 128 tiles of gemm.hip: 424 and 755).
// KS (own order): that many sets of RG waves, each with its share of the super-blocks and activation stages of its own; their sums meet at the end.
template <int WT, bool OWN, int RG, int C, int OCC, int KS = 1>
__global__ __launch_bounds__(64 * RG * KS, OCC) void xk_kernel(XT_PARAMS) {
    XT_HOT;
    constexpr bool K4 = WT == SPY_HIP_Q4_K;
    static_assert(KS == 1 || OWN, "the host's order is one chain over K");
    constexpr int NT = 64 * RG, ROWS = 16 * RG, NXI = C * 256 / NT, C2 = (C + 1) / 2;
    constexpr int XB = C * XT_XB + C2 * 1024;
    constexpr int NXS = 2;                         // stage s is worked on, stage s + 1 is on its way
    static_assert(NXI * NT == C * 256 && RG >= C2, "one request per thread and group, one wave per two groups' records");
    extern __shared__ __attribute__((aligned(16))) uint8_t smem_all[];
    const int tid = threadIdx.x, lane = tid & 63, wg_wave = __builtin_amdgcn_readfirstlane(tid >> 6), q = lane >> 4, r = lane & 15;
    const int ks = KS > 1 ? wg_wave / RG : 0, wave = KS > 1 ? wg_wave % RG : wg_wave;
    const int mat = hot.mat((int)blockIdx.x), m0 = ((int)blockIdx.x - mat * hot.tiles) * ROWS, cg0 = (int)blockIdx.y * C;
    const int ncg = a.ncg, M = a.M;
    // the set's super-blocks: sb0 .. sb0 + nsb - 1; every set takes part in as many steps as the longest
    const int all = hot.nst / 2, per = (all + KS - 1) / KS, sb0 = min(ks * per, all - 1), nsb = KS > 1 ? max(min(per, all - ks * per), 0) : all;
    const int nst = 2 * nsb, nstep = 2 * per;
    uint8_t *smem = smem_all + ks * (NXS * XB);
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)smem;
    // activation stages into the ring, as in xt_kernel; one request brings the records of two groups
    const uint8_t *bx[NXI], *bd;
#pragma unroll
    for (int i = 0; i < NXI; i++) bx[i] = hot.xq + ((int64_t)min(cg0 + (i * NT + wave * 64) / 256, ncg - 1) * hot.nst + 2 * sb0) * XT_XB + (i * NT + wave * 64) % 256 * 16;
    const int dc0 = min(cg0 + 2 * min(wave, C2 - 1), ncg - 1), dc1 = min(dc0 + 1, ncg - 1);
    bd = hot.xd + ((int64_t)dc0 * hot.nst + 2 * sb0) * XT_XD;
    const uint32_t l16 = lane * 16, ld = (lane & 31) * 16 + (lane >> 5) * (uint32_t)((dc1 - dc0) * hot.nst * XT_XD);
    const uint32_t ldsx = __builtin_amdgcn_readfirstlane(lds0 + wave * 1024), ldsd = __builtin_amdgcn_readfirstlane(lds0 + C * XT_XB + min(wave, C2 - 1) * 1024);
    int is = 0;
    auto issue_x = [&]() {
        const uint32_t o = (is & (NXS - 1)) * XB;
        const int adv = is + 1 < nst ? 1 : 0;
#pragma unroll
        for (int i = 0; i < NXI; i++) { xt_dma16(bx[i], l16, ldsx + o + i * NT * 16); bx[i] += adv * XT_XB; }
        xt_dma16(bd, ld, ldsd + o);
        bd += adv * XT_XD;
        is++;
    };
    const uint8_t *wr = hot.w(mat) + (int64_t)min(m0 + wave * 16 + r, M - 1) * hot.w_row;
    xk_raw<WT> cur;
    xk_load_half<0>(cur, wr, sb0, q);
    issue_x();
    uint32_t dd = 0;                               // Q6_K in the host's order: the row's d

    float acc[C][4];                               // rows 4q .. 4q + 3 of the wave's 16, activation row r of the group
#pragma unroll
    for (int c = 0; c < C; c++)
#pragma unroll
        for (int v = 0; v < 4; v++) acc[c][v] = 0.0f;
    float A[OWN ? C : 1][4];
    xk_v4f Bm[OWN && K4 ? C : 1];
    float *tab = (float *)(smem_all + KS * NXS * XB) + wg_wave * (K4 ? (OWN ? 288 : 256) : 16);      // the wave's scales: Q4_K [sub-block][d * sc, dmin * m][row], Q6_K [row] d
    const xk_v4f zero = {0.0f, 0.0f, 0.0f, 0.0f};
    auto compute_own = [&](int s, auto par_c) {
        constexpr int par = decltype(par_c)::value;
        const uint8_t *sx = smem + (s & (NXS - 1)) * XB + q * 256 + r * 16, *sd = smem + (s & (NXS - 1)) * XB + C * XT_XB + r * 4;
        // steps (sub-block, activation group): operands of step j + 2 read and the matrix instruction of step j + 1 issued before the vector work of step j
        constexpr int NJ = 4 * C;
        uint4 w[2][K4 ? 1 : 2], xv[3];
        uint32_t dx[3];
        xk_v4f p[2];
        auto rd = [&](int j) {
            const int b = j / C, c = j % C;
            xv[j % 3] = *(const uint4 *)(sx + c * XT_XB + b * 1024);
            dx[j % 3] = *(const uint32_t *)(sd + c * XT_XD + b * 64);
        };
        auto weights = [&](auto b_c) {
            constexpr int b = decltype(b_c)::value;
            xk_unpack<WT, 4 * par + b>(cur, q, w[b & 1]);
            if constexpr (K4) {
                const uint32_t sc = ((const uint32_t *)tab)[(4 * par + b) * 16 + r];
                uint4 &o = w[b & 1][0];
                o = make_uint4(xk_pk_mul(o.x, sc), xk_pk_mul(o.y, sc), xk_pk_mul(o.z, sc), xk_pk_mul(o.w, sc));
            }
        };
        auto mm = [&](int j) {
            const int b = j / C;
            p[j & 1] = xk_mfma(w[b & 1][0], xv[j % 3], zero);
            if constexpr (!K4) p[j & 1] = xk_mfma(w[b & 1][1], xv[j % 3], p[j & 1]);
        };
        rd(0);
        rd(1);
        weights(std::integral_constant<int, 0>{});
        mm(0);
        auto step = [&](auto j_c) {
            constexpr int j = decltype(j_c)::value, b = j / C, c = j % C;
            if constexpr (j + 2 < NJ) rd(j + 2);
            if constexpr (j + 1 < NJ) {
                if constexpr ((j + 1) % C == 0) weights(std::integral_constant<int, (j + 1) / C>{});
                mm(j + 1);
            }
            __builtin_amdgcn_sched_barrier(0);
            const float x = h2f((uint16_t)dx[j % 3]);
#pragma unroll
            for (int v = 0; v < 4; v++) A[c][v] = par == 0 && b == 0 ? x * p[j & 1][v] : fmaf(x, p[j & 1][v], A[c][v]);
            __builtin_amdgcn_sched_barrier(0);
        };
        [&]<int... J>(std::integer_sequence<int, J...>) { (step(std::integral_constant<int, J>{}), ...); }(std::make_integer_sequence<int, NJ>{});
        if constexpr (K4) {                        // lane (q, r): sub-block q of the stage, row r of either side
            const float m = tab[128 + (4 * par + q) * 16 + r];
            const uint8_t *sq = sd + q * 64;
#pragma unroll
            for (int c = 0; c < C; c++) {
                const float xb = h2f((uint16_t)*(const uint32_t *)(sq + c * XT_XD)) * *(const float *)(sq + c * XT_XD + 256);
                Bm[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(m, xb, par == 0 ? zero : Bm[c], 0, 0, 0);
            }
        }
        if constexpr (par == 1) {
            const xk_v4f d = *(const xk_v4f *)(tab + (K4 ? 256 : 0) + 4 * q);
            xk_v4f dmin = zero;
            if constexpr (K4) dmin = *(const xk_v4f *)(tab + 272 + 4 * q);
#pragma unroll
            for (int c = 0; c < C; c++)
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    acc[c][v] = fmaf(d[v], A[c][v], acc[c][v]);
                    if constexpr (K4) acc[c][v] = fmaf(dmin[v], Bm[c][v], acc[c][v]);
                }
        }
    };
    auto compute_host = [&](int s, auto par_c) {
        constexpr int par = decltype(par_c)::value;
        const uint8_t *sx = smem + (s & (NXS - 1)) * XB + q * 256 + r * 16, *sd = smem + (s & (NXS - 1)) * XB + C * XT_XB + r * 4;
        const uint8_t *so = sd + (q >> 1) * XT_XD + (q & 1) * 64;
        // steps of four: sub-blocks 2h and 2h + 1 by activation groups 2g and 2g + 1, whose outer products come from one instruction of four blocks
        constexpr int NJ = 4 * C;
        static_assert(OWN || C % 2 == 0, "groups in pairs");
        uint4 w[2][K4 ? 1 : 2], xv[3];
        uint32_t dx[3];
        xk_v4f p[2], dsc[2];
        xt_v16f D;
        auto rd = [&](int j) {
            const int b = j / (2 * C) * 2 + (j & 1), c = j % (2 * C) / 4 * 2 + (j >> 1 & 1);
            xv[j % 3] = *(const uint4 *)(sx + c * XT_XB + b * 1024);
            if constexpr (K4) dx[j % 3] = *(const uint32_t *)(sd + c * XT_XD + b * 64);
        };
        float dm = 0.0f, bs = 0.0f;
        uint32_t dxo = 0;
        auto rd_outer = [&](int j) {               // lane (q, r): sub-block 2h + q % 2, group 2g + q / 2
            const int h = j / (2 * C), g = j % (2 * C) / 4;
            if constexpr (K4) bs = *(const float *)(so + 256 + 2 * g * XT_XD + h * 128);
            else dxo = *(const uint32_t *)(so + 2 * g * XT_XD + h * 128);
        };
        auto outer = [&]() {
            if constexpr (K4) D = __builtin_amdgcn_mfma_f32_16x16x1f32(dm, bs, xt_v16f{}, 0, 0, 0);
            else D = xt_mfma(dd, 0u, dxo, 0u);
        };
        auto weights = [&](auto h_c) {
            constexpr int h = decltype(h_c)::value;
            xk_unpack<WT, 4 * par + 2 * h>(cur, q, w[0]);
            xk_unpack<WT, 4 * par + 2 * h + 1>(cur, q, w[1]);
            if constexpr (K4) {
                dsc[0] = *(const xk_v4f *)(tab + (4 * par + 2 * h) * 32 + 4 * q);
                dsc[1] = *(const xk_v4f *)(tab + (4 * par + 2 * h + 1) * 32 + 4 * q);
                dm = tab[(4 * par + 2 * h + (q & 1)) * 32 + 16 + r];
            }
        };
        auto mm = [&](int j) {
            p[j & 1] = xk_mfma(w[j & 1][0], xv[j % 3], zero);
            if constexpr (!K4) p[j & 1] = xk_mfma(w[j & 1][1], xv[j % 3], p[j & 1]);
        };
        rd(0);
        rd_outer(0);
        rd(1);
        weights(std::integral_constant<int, 0>{});
        mm(0);
        outer();
        auto step = [&](auto j_c) {
            constexpr int j = decltype(j_c)::value, c = j % (2 * C) / 4 * 2 + (j >> 1 & 1);
            const xk_v4f ds = dsc[j & 1];
            if constexpr (j + 2 < NJ) rd(j + 2);
            if constexpr ((j & 3) == 1 && j + 3 < NJ) rd_outer(j + 3);
            if constexpr (j + 1 < NJ) {
                if constexpr ((j + 1) % (2 * C) == 0) weights(std::integral_constant<int, (j + 1) / (2 * C)>{});
                mm(j + 1);
            }
            __builtin_amdgcn_sched_barrier(0);
            float x = 0.0f;
            if constexpr (K4) x = h2f((uint16_t)dx[j % 3]);
#pragma unroll
            for (int v = 0; v < 4; v++) {
                if constexpr (K4) acc[c][v] = fmaf(x, ds[v] * p[j & 1][v] - D[4 * (j & 3) + v], acc[c][v]);
                else acc[c][v] = fmaf(D[4 * (j & 3) + v], p[j & 1][v], acc[c][v]);
            }
            if constexpr ((j & 3) == 3 && j + 1 < NJ) outer();
            __builtin_amdgcn_sched_barrier(0);
        };
        [&]<int... J>(std::integer_sequence<int, J...>) { (step(std::integral_constant<int, J>{}), ...); }(std::make_integer_sequence<int, NJ>{});
    };
    auto compute = [&](int s, auto par_c) {
        if constexpr (OWN) compute_own(s, par_c);
        else compute_host(s, par_c);
    };
    auto ready = [&]() {
        xt_wait_vm<0>();
        __builtin_amdgcn_s_barrier();
    };
    for (int s = 0; s < nstep; s += 2) {
        const bool on = KS == 1 || s < nst;
        ready();
        xk_arrived<0>(cur);                        // where nothing is on its way
        if constexpr (OWN && K4) xk_put_scales_own(cur, tab, q, r);
        else if constexpr (OWN || K4) xk_put_scales<WT>(cur, tab, q, r);
        else dd = cur.d == 0xFFFFu ? 0u : cur.d;
        // the activations of the next stage ahead of the weights, which come from memory: requests are served in order, and the
        // own order's stages are shorter than what the weights take (11008 x 4096 x 128 Q4_K 51.5 -> 47.2 us, 16000 x 6144 x 200 142 -> 130).
        // A half of a super-block is requested a stage ahead, into the registers of the one that has been unpacked.
        issue_x();
        __builtin_amdgcn_sched_barrier(0);
        xk_load_half<1>(cur, wr, sb0 + max(min(s / 2, nsb - 1), 0), q);
        if (on) compute(s, std::integral_constant<int, 0>{});
        ready();
        xk_arrived<1>(cur);
        issue_x();
        __builtin_amdgcn_sched_barrier(0);
        xk_load_half<0>(cur, wr, sb0 + max(min(s / 2 + 1, nsb - 1), 0), q);
        if (on) compute(s + 1, std::integral_constant<int, 1>{});
    }
    xt_wait_vm<0>();
    if constexpr (KS > 1) {                         // the sets' sums, in order
        __builtin_amdgcn_s_barrier();
        float *ex = (float *)smem_all;
        if (ks > 0) {
#pragma unroll
            for (int c = 0; c < C; c++)
#pragma unroll
                for (int v = 0; v < 4; v++) ex[(((ks - 1) * RG + wave) * C * 4 + c * 4 + v) * 64 + lane] = acc[c][v];
        }
        __syncthreads();
        if (ks > 0) return;
#pragma unroll
        for (int k = 0; k < KS - 1; k++)
#pragma unroll
            for (int c = 0; c < C; c++)
#pragma unroll
                for (int v = 0; v < 4; v++) acc[c][v] += ex[((k * RG + wave) * C * 4 + c * 4 + v) * 64 + lane];
    }
    if constexpr (!OWN && !K4) {                    // their operands were small integers times 2^-24
#pragma unroll
        for (int c = 0; c < C; c++)
#pragma unroll
            for (int v = 0; v < 4; v++) acc[c][v] *= 16777216.0f;
    }
    const int row = m0 + wave * 16 + 4 * q;
    float *dst = a.dst[mat];
#pragma unroll
    for (int c = 0; c < C; c++) {
        const int t = (cg0 + c) * 16 + r;
        if (t < a.T && row + 3 < M) {
            const int64_t at = (int64_t)t * a.d_row + row;
            float4 o = make_float4(acc[c][0], acc[c][1], acc[c][2], acc[c][3]);
            if (a.resid) { const float4 z = *(const float4 *)(a.resid + at); o.x += z.x; o.y += z.y; o.z += z.z; o.w += z.w; }
            *(float4 *)(dst + at) = o;
        }
    }
}
// The same dots for few activation rows: a workgroup takes one 16 x 16 tile and its four waves take every fourth super-block.  What is serial is only
// the fma per sub-block; the terms are independent, so each round the waves leave the terms of four super-blocks in LDS and then every wave
// walks a quarter of the outputs through their 32 fmas.  (16 rows of a 4096 x 4096 Q4_K matrix: 20 us as a chain in one wave, 10 here.)
template <int WT>
__global__ __launch_bounds__(256, 3) void xks_kernel(xt_args a) {
    constexpr bool K4 = WT == SPY_HIP_Q4_K;
    __shared__ __align__(16) float s_t[32][4][64];                  // [sub-block of the round][row 4q + v][lane]
    __shared__ __align__(16) float s_tab[4][K4 ? 256 : 16];
    __shared__ float s_x[32][16], s_d[4][16];                       // d_x of the round's sub-blocks; Q6_K: d of its super-blocks
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), q = lane >> 4, r = lane & 15;
    const int mat = (int)blockIdx.x / a.tiles, m0 = ((int)blockIdx.x - mat * a.tiles) * 16, cg = (int)blockIdx.y, nsb = a.nst / 2;
    const uint8_t *wr = a.w[mat] + (int64_t)min(m0 + r, a.M - 1) * a.w_row;
    const uint8_t *xq = a.xq + (int64_t)cg * a.nst * XT_XB + q * 256 + r * 16, *xd = a.xd + (int64_t)cg * a.nst * XT_XD;
    xk_raw<WT> cur = xk_load<WT>(wr, min(wave, nsb - 1), q), nxt;
    uint4 xv[8], xn[8];
    uint32_t dx[2], dn[2];
    float bs[K4 ? 8 : 1], bn[K4 ? 8 : 1];
    auto fetch = [&](int sb, uint4 (&v)[8], uint32_t (&d)[2], float (&b)[K4 ? 8 : 1]) {
        const uint8_t *p = xq + (int64_t)sb * 2 * XT_XB, *e = xd + (int64_t)sb * 2 * XT_XD;
#pragma unroll
        for (int k = 0; k < 8; k++) v[k] = *(const uint4 *)(p + k * 1024);
#pragma unroll
        for (int k = 0; k < 2; k++) d[k] = *(const uint32_t *)(e + k * XT_XD + lane * 4);            // lane (q, r): block q of the stage, activation row r
        if constexpr (K4) {
#pragma unroll
            for (int k = 0; k < 8; k++) b[k] = *(const float *)(e + (k >> 2) * XT_XD + 256 + (k & 3) * 64 + r * 4);
        }
    };
    fetch(min(wave, nsb - 1), xv, dx, bs);
    float *tab = s_tab[wave];
    const int v_ = wave;                           // the row 4q + v_ of the tile whose outputs this wave walks
    float acc = 0.0f;
    const xk_v4f zero = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int s0 = 0; s0 < nsb; s0 += 4) {
        const int sb = s0 + wave;
        xk_put_scales<WT>(cur, tab, q, r);
        if (s0 + 4 < nsb) { nxt = xk_load<WT>(wr, min(sb + 4, nsb - 1), q); fetch(min(sb + 4, nsb - 1), xn, dn, bn); }
        if (s0) __syncthreads();                   // the terms of the round before have been walked
#pragma unroll
        for (int k = 0; k < 2; k++) s_x[wave * 8 + 4 * k + q][r] = h2f((uint16_t)dx[k]);
        if (!K4 && q == 0) s_d[wave][r] = tab[r];
        auto term = [&](auto t_c) {
            constexpr int t = decltype(t_c)::value;
            uint4 w[K4 ? 1 : 2];
            xk_unpack<WT, t>(cur, q, w);
            xk_v4f p = xk_mfma(w[0], xv[t], zero);
            if constexpr (!K4) p = xk_mfma(w[1], xv[t], p);
            if constexpr (K4) {
                const xk_v4f dsc = *(const xk_v4f *)(tab + t * 32 + 4 * q), dm = *(const xk_v4f *)(tab + t * 32 + 16 + 4 * q);
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const float pos = dsc[v] * p[v], neg = dm[v] * bs[t];
                    p[v] = pos - neg;
                }
            }
#pragma unroll
            for (int v = 0; v < 4; v++) s_t[wave * 8 + t][v][lane] = p[v];
        };
        [&]<int... J>(std::integer_sequence<int, J...>) { (term(std::integral_constant<int, J>{}), ...); }(std::make_integer_sequence<int, 8>{});
        __syncthreads();
        const int nb = min(4, nsb - s0) * 8;
#pragma unroll 8
        for (int b = 0; b < nb; b++) {
            float x = s_x[b][r];
            if constexpr (!K4) x = x * s_d[b >> 3][4 * q + v_];
            acc = fmaf(x, s_t[b][v_][lane], acc);
        }
        cur = nxt;
#pragma unroll
        for (int k = 0; k < 8; k++) xv[k] = xn[k];
        dx[0] = dn[0]; dx[1] = dn[1];
        if constexpr (K4) {
#pragma unroll
            for (int k = 0; k < 8; k++) bs[k] = bn[k];
        }
    }
    const int row = m0 + 4 * q + v_, t = cg * 16 + r;
    if (t < a.T && row < a.M) {
        const int64_t at = (int64_t)t * a.d_row + row;
        a.dst[mat][at] = a.resid ? acc + a.resid[at] : acc;
    }
}
// ---- Q4_0 in this backend's own order: ONE accumulator per output, acc = fma(d_w * d_x, float(block dot), acc) block after block -----
// (the arithmetic and the bits of gemm_q8act_kernel in gemm.hip).  The block dot of a 16 x 16 tile is one v_mfma_f32_16x16x32_f16, a float and exact,
// and the scale products of four blocks are one 16x16x4_4b as above: 24 matrix-core cycles and four fmas (16 cycles) per tile and block, where
// the int8 form takes a 35-cycle instruction, a 32-cycle one and two vector instructions per output of a 32 x 32 tile.
// Matrix and vector cycles of these instructions hardly overlap (counters of 16 x 16 tiles at 1000 rows: vector 36 %, matrix 38 %, at once 13 % of the time), which is
// why the cycles above are what counts; and the tiles fill the chip better than 128 x 128 ones.  Packing included, weights from memory, Q4_0, 4096 x 4096: 385 rows 90 -> 40 us,
// 512 rows 92 -> 41, 1000 rows 95 -> 68, 2048 rows 117 -> 109; 4096 x 11008: 1000 rows 232 -> 165; 22016 x 4096: 77 rows 90 -> 54, 1000 rows 312 -> 278.
// Two kernels of one arithmetic.  xo_kernel, for few workgroups: four waves of 16 rows by four activation groups, in tiles of 16 x 16.
// Weights: lane (q, r) reads blocks 2q and 2q + 1 of row r and chunk (contiguous over the four lanes of a row), brings words 2i and 2i + 1 of a block
// into one dword, and 4 x 4 exchanges between the lane blocks (v_permlane16_swap, v_permlane32_swap) leave words 2q and 2q + 1 of every block in lane block q:
// the sixteen neighbouring bytes that a lane's activation operand is in LDS.  (With words q and 4 + q, two 8-byte reads 16 bytes apart met in the same banks,
// half of the LDS cycles: 4096 x 11008 x 1000 182 -> 166 us, 22016 x 4096 x 1000 307 -> 297, 4096 x 4096 x 1000 74 -> 71.)
typedef float xo_v32f __attribute__((ext_vector_type(32)));
__device__ __forceinline__ xt_v16f xo_mfma(const uint4 &a, const uint4 &b, const xt_v16f &c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(xk_h8, a), __builtin_bit_cast(xk_h8, b), c, 0, 0, 0);
}
// eight quants of two words, low and high nibbles, as fp16 less 8: elements 0, 2, 1, 3 of either
__device__ __forceinline__ uint4 xo_unpack(uint32_t v) {
    const uint32_t u = v >> 8, c64 = 0x64006400u;
    return make_uint4(xt_sub(xt_and_or(v, 0x000F000Fu, c64), 0x64086408u), xt_sub(xt_and_or(u, 0x000F000Fu, c64), 0x64086408u),
                      xk_pk_fma(xt_and_or(v, 0x00F000F0u, c64), 0x2C002C00u, 0xD480D480u), xk_pk_fma(xt_and_or(u, 0x00F000F0u, c64), 0x2C002C00u, 0xD480D480u));        // (1024 + 16 n) / 16 - 72
}
// products of two blocks' scales, 32 x 32 each: lane (h, r) brings those of block h and row r
__device__ __forceinline__ xo_v32f xo_scales(uint32_t a, uint32_t b) {
    return __builtin_amdgcn_mfma_f32_32x32x4f16(__builtin_bit_cast(xt_h4, make_uint2(a, 0u)), __builtin_bit_cast(xt_h4, make_uint2(b, 0u)), xo_v32f{}, 0, 0, 0);
}
__device__ __forceinline__ void xo_transpose(uint32_t (&r)[4]) {
    auto s16 = [](uint32_t &a, uint32_t &b) { auto v = __builtin_amdgcn_permlane16_swap(a, b, false, false); a = v[0]; b = v[1]; };
    auto s32 = [](uint32_t &a, uint32_t &b) { auto v = __builtin_amdgcn_permlane32_swap(a, b, false, false); a = v[0]; b = v[1]; };
    s16(r[0], r[1]); s16(r[2], r[3]);
    s32(r[0], r[2]); s32(r[1], r[3]);
}
constexpr int XO_C = 4;
__global__ __launch_bounds__(256, 3) void xo_kernel(XT_PARAMS) {
    XT_HOT;
    constexpr int C = XO_C, NT = 256, ROWS = 64, C2 = C / 2, XB = C * XT_XB + C2 * 1024, NDW = 9, CB = xt_w<SPY_HIP_Q4_0>::CB;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), q = lane >> 4, r = lane & 15;
    const int mat = hot.mat((int)blockIdx.x), m0 = ((int)blockIdx.x - mat * hot.tiles) * ROWS, cg0 = (int)blockIdx.y * C;
    const int nst = hot.nst, ncg = a.ncg, M = a.M;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)smem;
    const uint8_t *bx[C], *bd;
#pragma unroll
    for (int i = 0; i < C; i++) bx[i] = hot.xq + (int64_t)min(cg0 + i, ncg - 1) * nst * XT_XB + wave * 1024;
    const int dc0 = min(cg0 + 2 * min(wave, C2 - 1), ncg - 1), dc1 = min(dc0 + 1, ncg - 1);
    bd = hot.xd + (int64_t)dc0 * nst * XT_XD;
    const uint32_t l16 = lane * 16, ld = (lane & 31) * 16 + (lane >> 5) * (uint32_t)((dc1 - dc0) * nst * XT_XD);
    const uint32_t ldsx = __builtin_amdgcn_readfirstlane(lds0 + wave * 1024), ldsd = __builtin_amdgcn_readfirstlane(lds0 + C * XT_XB + min(wave, C2 - 1) * 1024);
    int is = 0;
    auto issue_x = [&]() {
        const uint32_t o = (is & 1) * XB;
        const int adv = is + 1 < nst ? 1 : 0;
#pragma unroll
        for (int i = 0; i < C; i++) { xt_dma16(bx[i], l16, ldsx + o + i * NT * 16); bx[i] += adv * XT_XB; }
        xt_dma16(bd, ld, ldsd + o);
        bd += adv * XT_XD;
        is++;
    };
    const uint8_t *wr = hot.w(mat) + (int64_t)min(m0 + wave * 16 + r, M - 1) * hot.w_row + q * (NDW * 4);
    uint32_t cur[NDW];
    auto load_w = [&](int chunk) { __builtin_memcpy(cur, __builtin_assume_aligned(wr + (int64_t)chunk * CB, 4), NDW * 4); };
    load_w(0);
    issue_x();
    float acc[C][4];
#pragma unroll
    for (int c = 0; c < C; c++)
#pragma unroll
        for (int v = 0; v < 4; v++) acc[c][v] = 0.0f;
    uint32_t wd[2][4], dd;                         // [even, odd blocks][block of that kind]; the lane's two scales
    auto spread = [&]() {
        const uint32_t *v = cur;
        dd = (v[0] & 0xFFFFu) | (v[4] & 0xFFFF0000u);
        // dword i of a block: word 2i in the low nibbles, word 2i + 1 in the high ones (words 0..3 are the low nibbles of the block's four dwords, words 4..7 the high ones)
        auto pair = [](uint32_t (&o)[4], uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
            constexpr uint32_t lo = 0x0F0F0F0Fu;
            o[0] = (a & lo) | ((b << 4) & ~lo); o[1] = (c & lo) | ((d << 4) & ~lo);
            o[2] = ((a >> 4) & lo) | (b & ~lo); o[3] = ((c >> 4) & lo) | (d & ~lo);
        };
        pair(wd[0], __builtin_amdgcn_alignbit(v[1], v[0], 16), __builtin_amdgcn_alignbit(v[2], v[1], 16), __builtin_amdgcn_alignbit(v[3], v[2], 16), __builtin_amdgcn_alignbit(v[4], v[3], 16));
        pair(wd[1], v[5], v[6], v[7], v[8]);
        xo_transpose(wd[0]);
        xo_transpose(wd[1]);
    };
    const xk_v4f zero = {0.0f, 0.0f, 0.0f, 0.0f};
    auto compute = [&](int s, auto par_c) {
        constexpr int par = decltype(par_c)::value;
        const uint8_t *sx = smem + (s & 1) * XB + q * 256 + r * 16, *sd = smem + (s & 1) * XB + C * XT_XB + lane * 4;
        uint4 w[4];                                // operands of the stage's four blocks: words 2q and 2q + 1, elements 0, 2, 1, 3 each
        // lane (kb, r): the scale of block 4 par + kb, which lane block 2 par + kb / 2 holds
        const uint32_t d2 = (uint32_t)__builtin_amdgcn_ds_bpermute(((2 * par + (q >> 1)) * 16 + r) * 4, (int)dd), dw = (q & 1) ? d2 >> 16 : d2 & 0xFFFFu;
#pragma unroll
        for (int b = 0; b < 4; b++) w[b] = xo_unpack(wd[b & 1][2 * par + (b >> 1)]);
        constexpr int NJ = 4 * C;                  // steps (activation group, block)
        uint4 xv[3];
        uint32_t dx[2];
        xk_v4f p[2];
        xt_v16f D;
        auto rd = [&](int j) {
            xv[j % 3] = *(const uint4 *)(sx + (j >> 2) * XT_XB + (j & 3) * 1024);
        };
        dx[0] = *(const uint32_t *)sd;
        rd(0);
        rd(1);
        p[0] = xk_mfma(w[0], xv[0], zero);
        D = xt_mfma(dw, 0u, dx[0], 0u);
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            const int c = j >> 2, b = j & 3;
            if (j + 2 < NJ) rd(j + 2);
            if (b == 1 && c + 1 < C) dx[(c + 1) & 1] = *(const uint32_t *)(sd + (c + 1) * XT_XD);
            // one matrix instruction, then the four fmas that run beside it
            if (j + 1 < NJ) p[(j + 1) & 1] = xk_mfma(w[(j + 1) & 3], xv[(j + 1) % 3], zero);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int v = 0; v < 4; v++) acc[c][v] = fmaf(D[4 * b + v], p[j & 1][v], acc[c][v]);
            if (b == 3 && c + 1 < C) D = xt_mfma(dw, 0u, dx[(c + 1) & 1], 0u);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    auto ready = [&]() {
        xt_wait_vm<0>();
        __builtin_amdgcn_s_barrier();
    };
    for (int s = 0; s < nst; s += 2) {
        ready();
        spread();                                  // the compiler's own wait for the chunk stands here, where nothing is on its way
        issue_x();
        load_w(min(s / 2 + 1, nst / 2 - 1));
        compute(s, std::integral_constant<int, 0>{});
        ready();
        issue_x();
        compute(s + 1, std::integral_constant<int, 1>{});
    }
    xt_wait_vm<0>();
    float *dst = a.dst[mat];
    const int row = m0 + wave * 16 + 4 * q;
#pragma unroll
    for (int c = 0; c < C; c++) {
        const int t = (cg0 + c) * 16 + r;
        if (t < a.T && row + 3 < M) {
            const int64_t at = (int64_t)t * a.d_row + row;
            float4 o = make_float4(acc[c][0], acc[c][1], acc[c][2], acc[c][3]);
            if (a.resid) { const float4 z = *(const float4 *)(a.resid + at); o.x += z.x; o.y += z.y; o.z += z.z; o.w += z.w; }
            *(float4 *)(dst + at) = o;
        }
    }
}
// The same for many activation rows: four waves of 32 rows by four pairs of activation groups, in tiles of 32 x 32.  An operand read from LDS serves twice the
// arithmetic of a 16 x 16 tile's, and the compiler may order the matrix and vector instructions of a tile, which with 16 x 16 it did worse than by hand.
// On registers alone this form takes 19.4 ns per 16 x 16 x 32 and SIMD (two waves; the clock falls under these instructions) and the other 23.2; here it is
// 23.8, for 100 instructions of unpacking beside 256 fmas and 1536 matrix cycles.  Packing included, weights from memory, against two row groups of 16 per wave
// (with the operand reads in one bank that xo_kernel had then): 22016 x 4096 x 1000 310 -> 278 us, 12288 x 4096 x 1000 168 -> 151, 4096 x 11008 x 1000 188 -> 165, 4096 x 4096 x 1000 78 -> 68.
// (Two pairs per wave: 340 us at 22016 x 4096 x 1000; three: 311.)
constexpr int XO_CP = 4;
__global__ __launch_bounds__(256, 2) void xo32_kernel(XT_PARAMS) {
    XT_HOT;
    constexpr int CP = XO_CP, NT = 256, ROWS = 128, C = 2 * CP, XB = C * XT_XB + CP * 1024, NDW = 18, CB = xt_w<SPY_HIP_Q4_0>::CB;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), h = lane >> 5, r = lane & 31;
    const int mat = hot.mat((int)blockIdx.x), m0 = ((int)blockIdx.x - mat * hot.tiles) * ROWS, cg0 = (int)blockIdx.y * C;
    const int nst = hot.nst, ncg = a.ncg, M = a.M;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)smem;
    const uint8_t *bx[C], *bd;
#pragma unroll
    for (int i = 0; i < C; i++) bx[i] = hot.xq + (int64_t)min(cg0 + i, ncg - 1) * nst * XT_XB + wave * 1024;
    const int dc0 = min(cg0 + 2 * min(wave, CP - 1), ncg - 1), dc1 = min(dc0 + 1, ncg - 1);
    bd = hot.xd + (int64_t)dc0 * nst * XT_XD;
    const uint32_t l16 = lane * 16, ld = r * 16 + h * (uint32_t)((dc1 - dc0) * nst * XT_XD);
    const uint32_t ldsx = __builtin_amdgcn_readfirstlane(lds0 + wave * 1024), ldsd = __builtin_amdgcn_readfirstlane(lds0 + C * XT_XB + min(wave, CP - 1) * 1024);
    int is = 0;
    auto issue_x = [&]() {
        const uint32_t o = (is & 1) * XB;
        const int adv = is + 1 < nst ? 1 : 0;
#pragma unroll
        for (int i = 0; i < C; i++) { xt_dma16(bx[i], l16, ldsx + o + i * NT * 16); bx[i] += adv * XT_XB; }
        xt_dma16(bd, ld, ldsd + o);
        bd += adv * XT_XD;
        is++;
    };
    // lane (h, r): blocks 4h .. 4h + 3 of row r and chunk
    const uint8_t *wr = hot.w(mat) + (int64_t)min(m0 + wave * 32 + r, M - 1) * hot.w_row + h * (NDW * 4);
    uint32_t cur[NDW];
    auto load_w = [&](int chunk) { __builtin_memcpy(cur, __builtin_assume_aligned(wr + (int64_t)chunk * CB, 4), NDW * 4); };
    load_w(0);
    issue_x();
    float acc[CP][16];
#pragma unroll
    for (int c = 0; c < CP; c++)
#pragma unroll
        for (int v = 0; v < 16; v++) acc[c][v] = 0.0f;
    uint32_t wd[2][4][2], dd[2][2];                // [stage of the chunk][block][words 4h, 4h + 1 | 4h + 2, 4h + 3]; [stage][block pair] scales
    auto swap = [](uint32_t &x, uint32_t &y) { auto v = __builtin_amdgcn_permlane32_swap(x, y, false, false); x = v[0]; y = v[1]; };
    auto spread = [&]() {
        constexpr uint32_t lo = 0x0F0F0F0Fu;
#pragma unroll
        for (int b = 0; b < 4; b++) {
            uint32_t v[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int k = b * 9 / 2 + i;                                    // the block's quants start at byte 18 b + 2
                v[i] = b & 1 ? cur[k + 1] : __builtin_amdgcn_alignbit(cur[k + 1], cur[k], 16);
            }
            // words 0 .. 3 are the low nibbles of the block's four dwords, 4 .. 7 the high ones: the lanes below keep the low ones of theirs and take those of the others
#pragma unroll
            for (int i = 0; i < 2; i++) {
                uint32_t l = (v[2 * i] & lo) | ((v[2 * i + 1] << 4) & ~lo), u = ((v[2 * i] >> 4) & lo) | (v[2 * i + 1] & ~lo);
                swap(l, u);
                wd[0][b][i] = l;
                wd[1][b][i] = u;
            }
        }
#pragma unroll
        for (int k = 0; k < 2; k++) {
            uint32_t x = (cur[9 * k] & 0xFFFFu) | (cur[9 * k + 4] & 0xFFFF0000u), y = x;
            swap(x, y);
            dd[0][k] = h ? x >> 16 : x & 0xFFFFu;
            dd[1][k] = h ? y >> 16 : y & 0xFFFFu;
        }
    };
    auto compute = [&](int s, auto par_c) {
        constexpr int par = decltype(par_c)::value;
        const uint8_t *sx = smem + (s & 1) * XB + (r >> 4) * XT_XB + h * 512 + (r & 15) * 16, *sd = smem + (s & 1) * XB + C * XT_XB + (r >> 4) * XT_XD + h * 64 + (r & 15) * 4;
        uint4 w[4][2];
#pragma unroll
        for (int b = 0; b < 4; b++)
#pragma unroll
            for (int i = 0; i < 2; i++) w[b][i] = xo_unpack(wd[par][b][i]);
        constexpr int NJ = 4 * CP;                 // steps (activation pair, block)
        uint4 xv[3][2];
        uint32_t dx[2];
        xt_v16f p[2];
        xo_v32f D;
        auto rd = [&](int j) {
            xv[j % 3][0] = *(const uint4 *)(sx + (j >> 2) * 2 * XT_XB + (j & 3) * 1024);
            xv[j % 3][1] = *(const uint4 *)(sx + (j >> 2) * 2 * XT_XB + (j & 3) * 1024 + 256);
        };
        auto rd_d = [&](int k) { dx[k & 1] = *(const uint32_t *)(sd + (k >> 1) * 2 * XT_XD + (k & 1) * 128); };        // k: (activation pair, block pair)
        auto mm = [&](int j) { p[j & 1] = xo_mfma(w[j & 3][1], xv[j % 3][1], xo_mfma(w[j & 3][0], xv[j % 3][0], xt_v16f{})); };
        rd_d(0);
        rd(0);
        rd_d(1);
        rd(1);
        mm(0);
        D = xo_scales(dd[par][0], dx[0]);
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            if (j + 2 < NJ) rd(j + 2);
            if ((j & 1) == 0 && j / 2 + 2 < NJ / 2) rd_d(j / 2 + 2);
            if (j + 1 < NJ) mm(j + 1);
#pragma unroll
            for (int v = 0; v < 16; v++) acc[j >> 2][v] = fmaf(D[16 * (j & 1) + v], p[j & 1][v], acc[j >> 2][v]);
            if ((j & 1) && j + 1 < NJ) D = xo_scales(dd[par][(j + 1) >> 1 & 1], dx[(j + 1) >> 1 & 1]);
        }
    };
    auto ready = [&]() {
        xt_wait_vm<0>();
        __builtin_amdgcn_s_barrier();
    };
    for (int s = 0; s < nst; s += 2) {
        ready();
        spread();                                  // the compiler's own wait for the chunk stands here, where nothing is on its way
        issue_x();
        load_w(min(s / 2 + 1, nst / 2 - 1));
        compute(s, std::integral_constant<int, 0>{});
        ready();
        issue_x();
        compute(s + 1, std::integral_constant<int, 1>{});
    }
    xt_wait_vm<0>();
    float *dst = a.dst[mat];
#pragma unroll
    for (int c = 0; c < CP; c++) {
        const int t = (cg0 + 2 * c) * 16 + r;
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const int row = m0 + wave * 32 + 8 * g + 4 * h;
            if (t < a.T && row + 3 < M) {
                const int64_t at = (int64_t)t * a.d_row + row;
                float4 o = make_float4(acc[c][4 * g], acc[c][4 * g + 1], acc[c][4 * g + 2], acc[c][4 * g + 3]);
                if (a.resid) { const float4 z = *(const float4 *)(a.resid + at); o.x += z.x; o.y += z.y; o.z += z.z; o.w += z.w; }
                *(float4 *)(dst + at) = o;
            }
        }
    }
}
int xo32_launch(hipStream_t st, xt_args a, int nmat) {
    constexpr size_t lds = 2 * (2 * XO_CP * XT_XB + XO_CP * 1024);
    const int rc = spy_raise_lds_limit((const void *)xo32_kernel, lds);
    if (rc) return rc;
    a.tiles = (a.M + 127) / 128;
    xo32_kernel<<<dim3((unsigned)(a.tiles * nmat), (unsigned)((a.ncg + 2 * XO_CP - 1) / (2 * XO_CP))), dim3(256), lds, st>>>(XT_ARGS(a));
    return SPY_LAUNCH_RC();
}
int xo_launch(hipStream_t st, xt_args a, int nmat) {
    constexpr size_t lds = 2 * (XO_C * XT_XB + XO_C / 2 * 1024);
    static_assert(lds <= 64 * 1024, "");
    a.tiles = (a.M + 63) / 64;
    xo_kernel<<<dim3((unsigned)(a.tiles * nmat), (unsigned)((a.ncg + XO_C - 1) / XO_C)), dim3(256), lds, st>>>(XT_ARGS(a));
    return SPY_LAUNCH_RC();
}
template <int WT, bool OWN, int RG, int C, int OCC, int KS = 1>
int xk_launch(hipStream_t st, xt_args a, int nmat) {
    constexpr size_t lds = KS * (2 * (C * XT_XB + (C + 1) / 2 * 1024) + RG * (OWN ? 1152 : 1024));
    static_assert(lds <= 160 * 1024 && lds >= (size_t)(KS - 1) * RG * C * 1024, "");
    if (lds > 64 * 1024) { const int rc = spy_raise_lds_limit((const void *)xk_kernel<WT, OWN, RG, C, OCC, KS>, lds); if (rc) return rc; }
    a.tiles = (a.M + 16 * RG - 1) / (16 * RG);
    xk_kernel<WT, OWN, RG, C, OCC, KS><<<dim3((unsigned)(a.tiles * nmat), (unsigned)((a.ncg + C - 1) / C)), dim3(64 * RG * KS), lds, st>>>(XT_ARGS(a));
    return SPY_LAUNCH_RC();
}
template <int WT>
int xks_launch(hipStream_t st, xt_args a, int nmat) {
    a.tiles = (a.M + 15) / 16;
    xks_kernel<WT><<<dim3((unsigned)(a.tiles * nmat), (unsigned)a.ncg), dim3(256), 0, st>>>(a);
    return SPY_LAUNCH_RC();
}

template <int WT>
int xt_dispatch(hipStream_t st, const xt_args &a, int nmat) {
    switch (xt_choose(WT == SPY_HIP_Q8_0, a.M, nmat, a.ncg, spy_num_cu())) {
    case XT_N4: return xn_launch<WT, 4>(st, a, nmat);
    case XT_N2: return xn_launch<WT, 2>(st, a, nmat);
    case XT_1: return xt_launch<WT, 1, 4, 2, 2>(st, a, nmat);
    case XT_2: return xt_launch<WT, 2, 4, 2, 2>(st, a, nmat);
    case XT_4: return xt_launch<WT, 4, 2, 1, 2>(st, a, nmat);
    case XT_MIXED + 1: return xt_launch_mixed<WT, 1>(st, a, nmat);
    case XT_MIXED + 2: return xt_launch_mixed<WT, 2>(st, a, nmat);
    default: return xt_launch_mixed<WT, 3>(st, a, nmat);
    }
}
template <int WT>
int xk_dispatch(hipStream_t st, const xt_args &a, int nmat) {
    switch (xk_choose(WT == SPY_HIP_Q4_K, a.M, nmat, a.ncg, spy_num_cu())) {
    case 0: return xks_launch<WT>(st, a, nmat);
    case 1: return xk_launch<WT, false, 2, 2, 4>(st, a, nmat);
    case 2: return xk_launch<WT, false, 4, 2, 4>(st, a, nmat);
    case 3: return xk_launch<WT, false, 4, 4, 4>(st, a, nmat);
    default: return xk_launch<WT, false, 8, 8, 4>(st, a, nmat);
    }
}

// the own order of the K-quants.  xks_kernel and the tiles that split K add the terms in other orders than the rest: the choice is that of the whole call, so
// that a call in pieces has its bits
template <int WT>
int xko_dispatch(hipStream_t st, const xt_args &a, int nmat) {
    switch (xko_choose(WT == SPY_HIP_Q4_K, a.M, nmat, a.ncg_all, spy_num_cu())) {
    case 0: return xks_launch<WT>(st, a, nmat);
    case 1: return xk_launch<WT, true, 2, 2, 4>(st, a, nmat);
    case 2: return xk_launch<WT, true, 4, 2, 4>(st, a, nmat);
    case 3: return xk_launch<WT, true, 2, 4, 3>(st, a, nmat);
    case 4: return xk_launch<WT, true, 4, 4, 4>(st, a, nmat);
    case 5: return xk_launch<WT, true, 4, 8, 2>(st, a, nmat);
    case 6: return xk_launch<WT, true, 2, 2, 2, 4>(st, a, nmat);
    case 7: return xk_launch<WT, true, 2, 4, 2, 4>(st, a, nmat);
    default: return xk_launch<WT, true, 4, 4, 2, 2>(st, a, nmat);
    }
}

int xo_dispatch(hipStream_t st, const xt_args &a, int nmat) {
    return xo_choose(a.M, nmat, a.ncg, spy_num_cu()) == 0 ? xo_launch(st, a, nmat) : xo32_launch(st, a, nmat);
}

}   // namespace

// ---- what exact_order.hip and the engine call -----------------------------------------------------------------------------------------
// bytes of packed activations of T rows of K elements (0: K is not a multiple of 256, or more groups of 16 rows than a grid's y takes)
size_t spy_xgemm_pack_bytes(int64_t T, int64_t K) {
    if (T <= 0 || T > 16 * 65535 || K <= 0 || K % 256) return 0;
    return (size_t)((T + 15) / 16 * (K / 128) * (XT_XB + XT_XD));
}
// shapes and alignments the kernels take: whole chunks, 16-byte-aligned weight rows, four outputs stored together
bool spy_xgemm_ok(int wtype, const void *w, const float *dst, int64_t M, int64_t K, int64_t T, int64_t d_row) {
    return (wtype == SPY_HIP_Q4_0 || wtype == SPY_HIP_Q8_0 || wtype == SPY_HIP_Q4_K || wtype == SPY_HIP_Q6_K) && T >= 1 && T <= 16 * 65535 && K > 0 && K % 256 == 0 && K <= (1 << 20) && M > 0 && M % 4 == 0 && M < (1 << 24) &&
           ((uintptr_t)w & 15) == 0 && ((uintptr_t)dst & 15) == 0 && d_row % 4 == 0;
}
int spy_xgemm_pack(hipStream_t st, const float *x, int64_t x_stride, int64_t T, int64_t K, void *pack) {
    if (((uintptr_t)x & 15) || x_stride % 16 || ((uintptr_t)pack & 15) || !spy_xgemm_pack_bytes(T, K)) return SPY_HIP_EINVAL;
    const int nst = (int)(K / 128), ncg = (int)((T + 15) / 16);
    uint8_t *xq = (uint8_t *)pack, *xd = xq + (int64_t)ncg * nst * XT_XB;
    xt_pack_kernel<<<dim3((unsigned)(K / 64), (unsigned)ncg), dim3(256), 0, st>>>((const uint8_t *)x, x_stride, (int)T, nst, xq, xd);
    return SPY_LAUNCH_RC();
}
// x [T][K] f32 -> NormRMS * w -> packed activations; own: sum of squares in this backend's own order
int spy_xgemm_norm_pack(hipStream_t st, bool own, const float *x, const float *w, float eps, int64_t T, int64_t K, void *pack) {
    if (((uintptr_t)x & 15) || ((uintptr_t)w & 15) || ((uintptr_t)pack & 15) || !spy_xgemm_pack_bytes(T, K) || K > 8192) return SPY_HIP_EINVAL;
    const int nst = (int)(K / 128), ncg = (int)((T + 15) / 16);
    uint8_t *xq = (uint8_t *)pack, *xd = xq + (int64_t)ncg * nst * XT_XB;
    const dim3 grid((unsigned)((ncg + 7) / 8 * 128));
    if (own && K <= 4096) xt_norm_pack_kernel<2, true><<<grid, dim3(256), 0, st>>>(x, w, eps, (int)K, (int)T, nst, xq, xd);
    else if (own) xt_norm_pack_kernel<4, true><<<grid, dim3(256), 0, st>>>(x, w, eps, (int)K, (int)T, nst, xq, xd);
    else if (K <= 4096) xt_norm_pack_kernel<2, false><<<grid, dim3(256), 0, st>>>(x, w, eps, (int)K, (int)T, nst, xq, xd);
    else xt_norm_pack_kernel<4, false><<<grid, dim3(256), 0, st>>>(x, w, eps, (int)K, (int)T, nst, xq, xd);
    return SPY_LAUNCH_RC();
}
// gate, up [T][F] f32 -> up * silu(gate) -> packed activations; lut: the host's tables (spy_exact_luts), or null
int spy_xgemm_silu_pack(hipStream_t st, const float *gate, const float *up, const float *lut, int64_t T, int64_t F, void *pack) {
    if (((uintptr_t)gate & 15) || ((uintptr_t)up & 15) || ((uintptr_t)pack & 15) || !spy_xgemm_pack_bytes(T, F)) return SPY_HIP_EINVAL;
    const int nst = (int)(F / 128), ncg = (int)((T + 15) / 16);
    uint8_t *xq = (uint8_t *)pack, *xd = xq + (int64_t)ncg * nst * XT_XB;
    const int64_t tiles = (int64_t)nst * ncg, cu = spy_num_cu();
    if (lut && tiles >= 3 * cu && tiles < INT32_MAX - 4 * cu) {
        constexpr size_t lds = 2 * SL_N * 4;
        const int rc = spy_raise_lds_limit((const void *)xt_silu_pack_many_kernel, lds);
        if (rc) return rc;
        xt_silu_pack_many_kernel<<<dim3((unsigned)cu), dim3(1024), lds, st>>>(gate, up, lut, (int)F, (int)T, nst, (int)tiles, xq, xd);
        return SPY_LAUNCH_RC();
    }
    xt_silu_pack_kernel<<<dim3((unsigned)nst, (unsigned)ncg), dim3(256), 0, st>>>(gate, up, lut, (int)F, (int)T, nst, xq, xd);
    return SPY_LAUNCH_RC();
}
static int xt_fill(xt_args &a, int wtype, int nmat, const void *const *w, float *const *dst, int64_t M, int64_t K, int64_t T, int64_t d_row, const float *resid, const void *pack) {
    if (nmat < 1 || nmat > 3 || (resid && nmat != 1) || ((uintptr_t)resid & 15) || ((uintptr_t)pack & 15)) return SPY_HIP_EINVAL;
    a = {};
    for (int i = 0; i < nmat; i++) {
        if (!spy_xgemm_ok(wtype, w[i], dst[i], M, K, T, d_row)) return SPY_HIP_EINVAL;
        a.w[i] = (const uint8_t *)w[i];
        a.dst[i] = dst[i];
    }
    a.resid = resid; a.w_row = spy_row_size(wtype, K); a.d_row = d_row;
    a.M = (int)M; a.nst = (int)(K / 128); a.ncg = a.ncg_all = (int)((T + 15) / 16); a.T = (int)T;
    a.xq = (const uint8_t *)pack; a.xd = a.xq + (int64_t)a.ncg * a.nst * XT_XB;
    return 0;
}
// nmat (1 .. 3) matrices of the same type and shape times the packed activations; resid (one matrix only): added to the result
int spy_xgemm(hipStream_t st, int wtype, int nmat, const void *const *w, float *const *dst, int64_t M, int64_t K, int64_t T, int64_t d_row, const float *resid, const void *pack) {
    xt_args a;
    const int rc = xt_fill(a, wtype, nmat, w, dst, M, K, T, d_row, resid, pack);
    if (rc) return rc;
    switch (wtype) {
    case SPY_HIP_Q4_0: return xt_dispatch<SPY_HIP_Q4_0>(st, a, nmat);
    case SPY_HIP_Q8_0: return xt_dispatch<SPY_HIP_Q8_0>(st, a, nmat);
    case SPY_HIP_Q4_K: return xk_dispatch<SPY_HIP_Q4_K>(st, a, nmat);
    default: return xk_dispatch<SPY_HIP_Q6_K>(st, a, nmat);
    }
}
// the same in this backend's own order; T_all: rows of the whole call where it comes in pieces (0: this is all of it); Q4_0, Q4_K, Q6_K (Q8_0 unpacks more per block than Q4_0: 3 % slower than the tile kernel of gemm.hip at 22016 rows)
int spy_xgemm_own(hipStream_t st, int wtype, int nmat, const void *const *w, float *const *dst, int64_t M, int64_t K, int64_t T, int64_t d_row, const float *resid, const void *pack, int64_t T_all) {
    xt_args a;
    const int rc = xt_fill(a, wtype, nmat, w, dst, M, K, T, d_row, resid, pack);
    if (rc) return rc;
    if (T_all > T) a.ncg_all = (int)((T_all + 15) / 16);
    return wtype == SPY_HIP_Q4_0 ? xo_dispatch(st, a, nmat) : wtype == SPY_HIP_Q4_K ? xko_dispatch<SPY_HIP_Q4_K>(st, a, nmat) : wtype == SPY_HIP_Q6_K ? xko_dispatch<SPY_HIP_Q6_K>(st, a, nmat) : SPY_HIP_EINVAL;
}
