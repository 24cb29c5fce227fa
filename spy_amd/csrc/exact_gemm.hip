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
//     of 16 activation rows.  The accumulators of an output are split over AS waves (words 0..3 | 4..7, or pairs of words), which meet
//     in hsum_float_8 at the end: few activation rows still give AS * rows / 16 waves, and a wave's chain is AS times shorter.
//   * Weights (in chunks of eight blocks) and activations (in stages of four) go from memory straight into rings of LDS slots
//     (global_load_lds), P stages ahead of their use, one workgroup barrier per stage.
// Measured against what these kernels replaced (operands packed as fp16 once per call, 64 x 64 tiles), packing included:
// 4096 x 4096 Q4_0: 16 rows 80 -> 15 us, 77 rows 104 -> 28, 512 rows 137 -> 88, 2048 rows 400 -> 313; 8 rows (one launch per row) 36 -> 15.
#include "common.cuh"

#include <type_traits>

namespace {

typedef _Float16 xt_h2 __attribute__((ext_vector_type(2)));
typedef _Float16 xt_h4 __attribute__((ext_vector_type(4)));
typedef float xt_v16f __attribute__((ext_vector_type(16)));

// Layout of packed activations, per group of 16 rows and stage of four Q8_0 blocks: XT_XB bytes of quants
//   [block][word pair g][row][word of the pair][4 x fp16: elements 0, 2, 1, 3 of the word]
// and one record of scales [block][row], XT_XD bytes: fp16 in the lower half of a dword
#define XT_XB 4096
#define XT_XD 256

// 16 (4) bytes per lane from base + off to LDS bytes lds .. in lane order; base and lds are uniform over the wave.  Written as
// instructions so that the compiler does not wait for them at the next LDS read; xt_wait_vm says when they have to be there.
__device__ __forceinline__ void xt_dma16(const void *base, uint32_t off, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" :: "s"(lds), "v"(off), "s"(base) : "memory");
}
__device__ __forceinline__ void xt_dma4(const void *base, uint32_t off, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" :: "s"(lds), "v"(off), "s"(base) : "memory");
}
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
    const uint8_t *xq, *xd;
};

// AS: waves that share the accumulators of a tile (2 or 4); RG: groups of 16 weight rows per workgroup; C: groups of 16 activation rows per
// wave; NXS, NWC: LDS slots for stages and chunks (powers of two); P: stages requested ahead
template <int WT, int AS, int RG, int C, int NXS, int P, int NWC, int OCC>
__global__ __launch_bounds__(64 * AS * RG, OCC) void xt_kernel(xt_args a) {
    constexpr int NT = 64 * AS * RG, ROWS = 16 * RG;
    constexpr int CU = xt_w<WT>::CU, UW = ROWS * CU, NI = (UW + NT - 1) / NT, NXI = C * 256 / NT;
    constexpr int XB = C * (XT_XB + XT_XD), WB = (UW + 63) / 64 * 1024;
    static_assert(NXI * NT == C * 256 && AS * RG >= C && NXS > P && NWC * 2 > P, "one request per thread and group, one wave per group's scales, slots for what is on its way");
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = wave % AS, rg = wave / AS, q = lane >> 4, r = lane & 15;
    const int mat = (int)blockIdx.x / a.tiles, m0 = ((int)blockIdx.x - mat * a.tiles) * ROWS, cg0 = (int)blockIdx.y * C;
    const int nst = a.nst, ncg = a.ncg, M = a.M;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)smem;

    // what a wave requests: uniform bases that advance, per-lane offsets that stay.  Row groups and activation groups past the end
    // repeat the last one.
    const uint8_t *bx[NXI], *bd, *bw = a.w[mat] + (int64_t)m0 * a.w_row;
    uint32_t ow[NI];
#pragma unroll
    for (int i = 0; i < NXI; i++) bx[i] = a.xq + (int64_t)min(cg0 + (i * NT + wave * 64) / 256, ncg - 1) * nst * XT_XB + (i * NT + wave * 64) % 256 * 16;
    bd = a.xd + (int64_t)min(cg0 + min(wave, C - 1), ncg - 1) * nst * XT_XD;
#pragma unroll
    for (int i = 0; i < NI; i++) {
        const int u = min(tid + i * NT, UW - 1);
        ow[i] = (uint32_t)(min(m0 + u / CU, M - 1) - m0) * (uint32_t)a.w_row + (u % CU) * 16;
    }
    // (the last request of a chunk covers it with the first waves only: the others put what they repeat into the spare kilobyte after the rings)
    const bool spare = wave * 64 + (NI - 1) * NT >= UW;
    const uint32_t lds_spare = __builtin_amdgcn_readfirstlane(lds0 + NXS * XB + NWC * WB);
    const uint32_t l16 = lane * 16, l4 = lane * 4;
    const uint32_t ldsx = __builtin_amdgcn_readfirstlane(lds0 + wave * 1024), ldsd = __builtin_amdgcn_readfirstlane(lds0 + C * XT_XB + min(wave, C - 1) * XT_XD),
                   ldsw = __builtin_amdgcn_readfirstlane(lds0 + NXS * XB + wave * 1024);
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
        const uint32_t o = ldsw + ((is >> 1) & (NWC - 1)) * WB;
#pragma unroll
        for (int i = 0; i < NI; i++) xt_dma16(bw, ow[i], i == NI - 1 && spare ? lds_spare : o + i * NT * 16);
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

    // Where a lane finds its operands.  AS == 2: word 4g + q of one block per matrix instruction.  AS == 4: lane block q holds word 2g + (q & 1)
    // of block 2i + (q >> 1), so one instruction takes two blocks.  A Q4_0 block holds words 0..3 in the low nibbles and 4..7 in the
    // high nibbles of its four quant dwords (which start at byte 2: blocks at odd dword halves are read as two dwords).
    constexpr bool Q4 = WT == SPY_HIP_Q4_0;
    constexpr int PD = xt_w<WT>::PD, OD = Q4 ? 5 : 9, BB = xt_w<WT>::BB;
    const int kbpar = q >> 1;
    const uint32_t wbase = (rg * 16 + r) * xt_w<WT>::CB +
                           4 * (AS == 2 ? q + (Q4 ? 0 : 4 * g) : kbpar * OD + (q & 1) + (Q4 ? 2 * (g & 1) : 2 * g));
    const uint32_t al = AS == 4 && kbpar ? 0 : 16;
    const int sh = Q4 ? 4 * (AS == 2 ? g : g >> 1) : 0;
    const uint32_t dbase = (rg * 16 + r) * xt_w<WT>::CB + q * BB;
    const uint32_t xbase = AS == 2 ? (2 * g + (q >> 1)) * 256 + r * 16 + (q & 1) * 8 : kbpar * 1024 + g * 256 + r * 16 + (q & 1) * 8;
    const uint32_t c64 = 0x64006400u;

    auto compute = [&](int s, auto par_c) {
        constexpr int par = decltype(par_c)::value;                 // which half of the chunk
        const uint8_t *sx = smem + (s & (NXS - 1)) * XB, *sw = smem + NXS * XB + ((s >> 1) & (NWC - 1)) * WB;
        constexpr int NW = AS == 2 ? 4 : 2;                         // weight operands of the stage
        uint32_t wa[NW], wb[NW];
        {
            const uint32_t *b = (const uint32_t *)(sw + wbase);
            uint32_t v[NW];
#pragma unroll
            for (int i = 0; i < 2; i++) {
                if constexpr (AS == 2) {
                    v[2 * i] = __builtin_amdgcn_alignbit(b[PD * (2 * par + i) + 1], b[PD * (2 * par + i)], 16);
                    v[2 * i + 1] = b[PD * (2 * par + i) + OD];
                } else v[i] = __builtin_amdgcn_alignbit(b[PD * (2 * par + i) + 1], b[PD * (2 * par + i)], al);
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
        auto rd = [&](int j) -> uint2 { return *(const uint2 *)(sx + (j / NW) * XT_XB + (j % NW) * (AS == 2 ? 1024 : 2048) + xbase); };
        uint2 xv[3];
        xt_v16f p[2], D[2];
        uint32_t dx = *(const uint32_t *)sd, dxn = 0;
        xv[0] = rd(0);
        xv[1] = rd(1);
        if (C > 1) dxn = *(const uint32_t *)(sd + XT_XD);
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
                    if (c1 + 1 < C) dxn = *(const uint32_t *)(sd + (c1 + 1) * XT_XD);
                }
                p[(j + 1) & 1] = xt_mfma(wa[i1], wb[i1], xv[(j + 1) % 3].x, xv[(j + 1) % 3].y);
            }
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (AS == 2) {
#pragma unroll
                for (int n = 0; n < 16; n++) acc[c][n] = fmaf(D[c & 1][4 * i + (n & 3)], p[j & 1][n], acc[c][n]);
            } else {
#pragma unroll
                for (int b = 0; b < 2; b++)
#pragma unroll
                    for (int n = 0; n < 8; n++) acc[c][n] = fmaf(D[c & 1][4 * (2 * i + b) + (n & 3)], p[j & 1][8 * b + n], acc[c][n]);
            }
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
            if constexpr (AS == 2) {
#pragma unroll
                for (int k = 0; k < 4; k++) rr[k] = ex[(c * NACC + 4 * k + v) * 64 + lane] + acc[c][4 * k + v];
            } else {
#pragma unroll
                for (int k = 0; k < 2; k++) {
                    rr[k] = ex[((C + c) * NACC + 4 * k + v) * 64 + lane] + acc[c][4 * k + v];
                    rr[2 + k] = ex[((2 * C + c) * NACC + 4 * k + v) * 64 + lane] + ex[(c * NACC + 4 * k + v) * 64 + lane];
                }
            }
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

// f32 rows -> packed activations: Quantizator<FP32,Q8_0>::transform (vec_convert.h:178-261), as quantize_q8_0_kernel, the quants as fp16.
// Rows past T become zeros.  8 lanes per block; a workgroup takes 16 rows and two blocks.
__global__ __launch_bounds__(256) void xt_pack_kernel(const uint8_t *__restrict__ x, int64_t x_stride, int T, int nst, uint8_t *__restrict__ xq, uint8_t *__restrict__ xd) {
    const int tid = threadIdx.x, e = tid & 7, c = (tid >> 3) & 15, b = (int)blockIdx.x * 2 + (tid >> 7), cg = blockIdx.y;
    const int t = cg * 16 + c;
    float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (t < T) v = *(const float4 *)(x + (int64_t)t * x_stride + (b * 32 + e * 4) * 4);
    float amax = fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w)));
    amax = fmaxf(amax, __shfl_xor(amax, 1, SPY_WAVE));
    amax = fmaxf(amax, __shfl_xor(amax, 2, SPY_WAVE));
    amax = fmaxf(amax, __shfl_xor(amax, 4, SPY_WAVE));
    const float d = amax / 127.0f, id = (amax != 0.0f) ? 127.0f / amax : 0.0f;
    int qv[4] = {(int)rintf(v.x * id), (int)rintf(v.y * id), (int)rintf(v.z * id), (int)rintf(v.w * id)};
    uint32_t h[4];
#pragma unroll
    for (int i = 0; i < 4; i++) { qv[i] = qv[i] < -128 ? -128 : (qv[i] > 127 ? 127 : qv[i]); h[i] = __builtin_bit_cast(uint16_t, (_Float16)(float)qv[i]); }
    uint8_t *o = xq + ((int64_t)cg * nst + (b >> 2)) * XT_XB + (b & 3) * 1024 + (e >> 1) * 256 + c * 16 + (e & 1) * 8;
    *(uint2 *)o = make_uint2(h[0] | (h[2] << 16), h[1] | (h[3] << 16));
    if (e == 0) *(uint32_t *)(xd + ((int64_t)cg * nst + (b >> 2)) * XT_XD + (b & 3) * 64 + c * 4) = f2h(d);
}

template <int WT, int AS, int RG, int C, int NXS, int P, int NWC, int OCC>
int xt_launch(hipStream_t st, xt_args a, int nmat) {
    constexpr size_t ring = NXS * C * (XT_XB + XT_XD) + NWC * ((16 * RG * xt_w<WT>::CU + 63) / 64) * 1024 + 1024, ex = (size_t)RG * (AS - 1) * C * (32 / AS) * 256, lds = ring > ex ? ring : ex;
    static_assert(lds <= 64 * 1024, "no raised LDS limit");
    a.tiles = (a.M + 16 * RG - 1) / (16 * RG);
    xt_kernel<WT, AS, RG, C, NXS, P, NWC, OCC><<<dim3((unsigned)(a.tiles * nmat), (unsigned)((a.ncg + C - 1) / C)), dim3(64 * AS * RG), lds, st>>>(a);
    return SPY_LAUNCH_RC();
}

int xt_num_cu() {
    static int n = 0;                              // the same value whoever writes it
    if (!n) {
        int dev = 0, v = 0;
        n = hipGetDevice(&dev) == hipSuccess && hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && v > 0 ? v : 256;
    }
    return n;
}

// Which tile: a workgroup of four waves puts one wave on each SIMD, and n workgroups per compute unit take about lat + (n - 1) * inc (in
// tenths of a microsecond for K = 4096, measured for n = 1 .. 16): small tiles have the shorter chain, large ones unpack a weight for
// more activation rows.
template <int WT>
int xt_dispatch(hipStream_t st, const xt_args &a, int nmat) {
    const int64_t cu = xt_num_cu(), r16 = (int64_t)((a.M + 15) / 16) * nmat, r32 = (int64_t)((a.M + 31) / 32) * nmat;
    auto cost = [&](int64_t wgs, int64_t lat, int64_t inc) { return lat + (wgs <= 6 * cu ? (wgs + cu - 1) / cu - 1 : (10 * wgs / cu - 10) / 10) * inc; };
    const int64_t k0 = cost(r16 * a.ncg, 86, 43), k1 = cost(r32 * a.ncg, 103, 56), k2 = cost(r32 * ((a.ncg + 1) / 2), 173, 96), k4 = cost(r32 * ((a.ncg + 3) / 4), 288, 165);
    if (k4 <= k0 && k4 <= k1 && k4 <= k2) return xt_launch<WT, 2, 2, 4, 2, 1, 2, 3>(st, a, nmat);
    if (k2 <= k0 && k2 <= k1) return xt_launch<WT, 2, 2, 2, 4, 2, 2, 3>(st, a, nmat);
    if (k1 <= k0) return xt_launch<WT, 2, 2, 1, 4, 2, 2, 3>(st, a, nmat);
    return xt_launch<WT, 4, 1, 1, 8, 6, 4, 2>(st, a, nmat);
}

}   // namespace

// ---- what exact_order.hip and the engine call -----------------------------------------------------------------------------------------
// bytes of packed activations of T rows of K elements (0: K is not a multiple of 256)
size_t spy_xgemm_pack_bytes(int64_t T, int64_t K) {
    if (T <= 0 || K <= 0 || K % 256) return 0;
    return (size_t)((T + 15) / 16 * (K / 128) * (XT_XB + XT_XD));
}
// shapes and alignments the kernels take: whole chunks, 16-byte-aligned weight rows, four outputs stored together
bool spy_xgemm_ok(int wtype, const void *w, const float *dst, int64_t M, int64_t K, int64_t T, int64_t d_row) {
    return (wtype == SPY_HIP_Q4_0 || wtype == SPY_HIP_Q8_0) && T >= 2 && T < (1 << 20) && K > 0 && K % 256 == 0 && K <= (1 << 20) && M > 0 && M % 4 == 0 && M < (1 << 24) &&
           ((uintptr_t)w & 15) == 0 && ((uintptr_t)dst & 15) == 0 && d_row % 4 == 0;
}
int spy_xgemm_pack(hipStream_t st, const float *x, int64_t x_stride, int64_t T, int64_t K, void *pack) {
    if (((uintptr_t)x & 15) || x_stride % 16 || ((uintptr_t)pack & 15) || !spy_xgemm_pack_bytes(T, K) || (T + 15) / 16 > 65535) return SPY_HIP_EINVAL;
    const int nst = (int)(K / 128), ncg = (int)((T + 15) / 16);
    uint8_t *xq = (uint8_t *)pack, *xd = xq + (int64_t)ncg * nst * XT_XB;
    xt_pack_kernel<<<dim3((unsigned)(K / 64), (unsigned)ncg), dim3(256), 0, st>>>((const uint8_t *)x, x_stride, (int)T, nst, xq, xd);
    return SPY_LAUNCH_RC();
}
// nmat (1 .. 3) matrices of the same type and shape times the packed activations; resid (one matrix only): added to the result
int spy_xgemm(hipStream_t st, int wtype, int nmat, const void *const *w, float *const *dst, int64_t M, int64_t K, int64_t T, int64_t d_row, const float *resid, const void *pack) {
    if (nmat < 1 || nmat > 3 || (resid && nmat != 1) || ((uintptr_t)resid & 15) || ((uintptr_t)pack & 15)) return SPY_HIP_EINVAL;
    xt_args a = {};
    for (int i = 0; i < nmat; i++) {
        if (!spy_xgemm_ok(wtype, w[i], dst[i], M, K, T, d_row)) return SPY_HIP_EINVAL;
        a.w[i] = (const uint8_t *)w[i];
        a.dst[i] = dst[i];
    }
    a.resid = resid; a.w_row = spy_row_size(wtype, K); a.d_row = d_row;
    a.M = (int)M; a.nst = (int)(K / 128); a.ncg = (int)((T + 15) / 16); a.T = (int)T;
    a.xq = (const uint8_t *)pack; a.xd = a.xq + (int64_t)a.ncg * a.nst * XT_XB;
    return wtype == SPY_HIP_Q4_0 ? xt_dispatch<SPY_HIP_Q4_0>(st, a, nmat) : xt_dispatch<SPY_HIP_Q8_0>(st, a, nmat);
}
