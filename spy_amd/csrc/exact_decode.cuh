// Kernels of the fused single-token pass in the HOST BACKEND'S SUMMATION ORDER: the same launches as
// decode_kernels.cuh (weights streamed once, activations quantized in LDS, epilogues fused), but every fp32 sum is
// added in the order of Spy's CPU loops, so that each output equals the CPU backend's bit for bit:
//   * quantized dots (vec_dot.h:42-115): eight accumulators per output element, lane l takes four products of every
//     block, acc[l] = fma(d_w * d_x, float(part[l]), acc[l]) block after block, then hsum_float_8 (vec_util.h:75-81);
//     K-quant rows: the project's order, one accumulator, one term per 32-element block;
//   * fp16 dots (vec_dot.h:117-146): 4 x 8 accumulators over chunks of 32 while i + 32 < n, the reduction tree, then
//     the scalar tail;
//   * NormRMS and Softmax sums (non-linear.cpp:129-223): libstdc++'s groups of four added to ONE running sum;
//   * exp and silu as the two fp16-indexed tables filled by the host's libm have them (exp in the attention worked out: exact_exp.cuh), the RoPE angles from a host table.
//
// How a serial sum is made fast.  The integer block dots stay where they are (64 lanes x v_dot4, one block pair per
// lane, weights read once, coalesced).  What changes is what follows them: instead of scaling and adding its blocks in
// lane order, a lane writes the eight partial sums of each of its blocks (as floats) and the block's scale product into
// LDS, transposed, and after a workgroup barrier ONE lane per accumulator walks its row of LDS block after block:
// 8 lanes per output element, 64 lanes = 8 output elements per wave, fed by 128-bit LDS reads.  The walk is a chain of
// dependent fmas (about 4 ns each on this part, whatever else the compute unit does), so a 4096-wide row costs about
// 0.6 us of latency per batch of rows; batches are as large as LDS allows (32 rows of 128 blocks; of K-quants all rows).
#pragma once

#include "decode_kernels.cuh"
#include "attn_reach.h"
#include "exact_exp.cuh"
#include "exact_sum.cuh"

#define XG_THREADS 1024
#define XG_WAVES 16
#define XG_NBS 128                         // blocks per K slab (= 64 lanes x one block pair)

template <int WT> struct xg_traits { static constexpr int NCH = (WT == SPY_HIP_Q4_0 || WT == SPY_HIP_Q8_0) ? 8 : 1; };
// floats of LDS per row slot: NCH rows of partials (+4: bank skew between the rows) and the row of scale products (+4: skew between slots)
static __host__ __device__ constexpr int xg_slot_floats(int nch) { return nch * (XG_NBS + 4) + XG_NBS + 4; }
// K-quant rows of several slabs: slots of their own for every slab, so that the waves that do not walk go on to the next one (11008 columns Q6_K 11.17 -> 10.48 us in a pass);
// two slots of eight accumulators per wave do not fit next to 11008 staged elements
static __host__ __device__ constexpr bool xg_slabs(int nch, int nitk) { return nch == 1 && nitk > 1; }

#define XG_LDS_PAD 64                       // what xg_chain reads past the last row

struct xg_args {
    const uint8_t *W0, *W1, *W2;
    int M, K;                              // output elements (RESID / STORE: rows of W0; GATEUP: rows of W0 = rows of W1; QKV: n_embd), contraction length
    const float *x_in, *normw; float eps;
    const float *resid; float *out;
    const dev_state *st; const float *rope_tab; uint16_t *q16, *kc, *vc;   // rope_tab: [n_ctx][hd] cos, sin per pair, from the host's libm
    const float *lut;                      // exp table [65536], then silu table [65536] (lookup_table_impl/non-linear.h:39-47,131-139)
    int n_ctx, d, hd;
    uint8_t *q8_dump;                      // tests: workgroup 0 writes its staged activations here as native Q8_0 blocks
    int pos_imm, rope_row0;                // st == nullptr: the position as a number; first position of rope_tab
    long long *dbg;                        // measurement builds (-DXDBG_STAMPS): wall-clock stamps of workgroup 0
};
// what the first requests of a launch need goes ahead of the rest: the first 14 dwords of a kernel's arguments come in registers (Makefile)
#define XG_ARGS(a) (a).x_in, (a).normw, (a).W0, (a).W1, (a).W2, (a).st, (a).K, (a).M, (a)
#ifdef XDBG_STAMPS
#define XSTAMP(dbg, i) do { if ((dbg) && blockIdx.x == 0 && threadIdx.x == 0) (dbg)[i] = wall_clock64(); } while (0)
#else
#define XSTAMP(dbg, i) do { } while (0)
#endif

// libstdc++'s std::reduce over the n values at s (LDS, 16-byte aligned; up to 40 floats beyond n may be read, never added): ONE
// running sum, value after value.  Every lane of the calling wave walks the same chain (same addresses: LDS broadcasts them), so
// the result is wave-uniform.  The additions are a chain of dependent operations (about 4 ns each); the 128-bit LDS reads of the
// next sixteen values are requested before the current sixteen additions (two register sets), so their latency hides behind the chain.
static __device__ __forceinline__ float xg_serial_sum(const float *s, int n, float init) {
    float4 a[2], b[2], c[2];
    auto ld = [&](float4 (&r)[2], int i) {
#pragma unroll
        for (int u = 0; u < 2; u++) r[u] = *(const float4 *)(s + i + 4 * u);
    };
    auto run = [&](const float4 (&r)[2]) {
#pragma unroll
        for (int u = 0; u < 2; u++) { init = init + r[u].x; init = init + r[u].y; init = init + r[u].z; init = init + r[u].w; }
    };
    // groups of 8 values, each requested two groups (sixteen dependent additions) ahead of its use: three register sets in rotation
    const int n24 = n - n % 24;
    int i = 0;
    if (n24) {
        ld(a, 0);
        ld(b, 8);
        for (; i < n24; i += 24) {
            ld(c, i + 16);
            __builtin_amdgcn_sched_barrier(0);
            run(a);
            __builtin_amdgcn_sched_barrier(0);
            ld(a, i + 24);                               // up to 28 floats beyond n: read, never added
            __builtin_amdgcn_sched_barrier(0);
            run(b);
            __builtin_amdgcn_sched_barrier(0);
            ld(b, i + 32);
            __builtin_amdgcn_sched_barrier(0);
            run(c);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    for (; i < n; i++) init = init + s[i];
    return init;
}

// ---- activations: f32 vector -> (RMSNorm * weight ->) Q8_0 in LDS, sums in the host order --------------------------
// NormRMS (non-linear.cpp:194-223): sum = std::transform_reduce(x, x) = groups of four ((x0^2 + x1^2) + (x2^2 + x3^2))
// added to one running sum in order; scale = 1 / sqrt(sum / n + eps); y = x * scale; then the Mul node: y * w.
// The 1024 threads form the group sums (one float4 each per 4096 elements), wave 0 adds them (xg_segment_sum).
template <int NITK, bool NORM, class Issue>
static __device__ __forceinline__ void xg_stage(const float4 (&xv)[NITK], const float4 (&wv)[NORM ? NITK : 1], int K, float eps,
                                                int8_t *s_q, int2 *s_meta, float *s_grp, float *s_scale, Issue issue_rows) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    float scale = 1.0f;
    if constexpr (NORM) {
#pragma unroll
        for (int j = 0; j < NITK; j++) {
            const int i = tid + j * XG_THREADS;
            if (i < K / 4) {
                const float4 v = xv[j];
                const float a0 = v.x * v.x, a1 = v.y * v.y, a2 = v.z * v.z, a3 = v.w * v.w;
                const float v1 = a0 + a1, v2 = a2 + a3;
                s_grp[xg_seg_at(i)] = v1 + v2;
            } else if (i < (K / 4 + 16 * NITK - 1) / (16 * NITK) * (16 * NITK)) s_grp[xg_seg_at(i)] = 0.0f;
        }
        // The weight rows are requested only after the group sums: a wave that asks for several rows sits in the issue stage until the memory
        // queue has room, and a request made earlier would hold up the barriers for every wave.  Wave 0 walks the sum first.
        __syncthreads();
        if (wave == 0) {
            const float mean = xg_segment_sum<NITK>(s_grp, K / 4) / (float)K, sc = 1.0f / sqrtf(mean + eps);
            if (lane == 0) *s_scale = sc;
        }
        issue_rows();
        __syncthreads();
        scale = *s_scale;
    } else issue_rows();
#pragma unroll
    for (int j = 0; j < NITK; j++) {
        const int i = tid + j * XG_THREADS;
        if (i < K / 4) {
            float4 v = xv[j];
            if constexpr (NORM) {
                const float4 w = wv[j];
                v.x = (v.x * scale) * w.x; v.y = (v.y * scale) * w.y; v.z = (v.z * scale) * w.z; v.w = (v.w * scale) * w.w;
            }
            int2 meta;
            const uint32_t q = quantize_oct(v, meta);
            ((uint32_t *)s_q)[act_dw(i, K >> 6)] = q;
            if ((tid & 7) == 0) s_meta[i >> 3] = meta;
        }
    }
    __syncthreads();
}

// the staged activations of a workgroup as native Q8_0 blocks (tests compare them with Quantizator<FP32,Q8_0>)
static __device__ __forceinline__ void xg_dump_q8(const int8_t *s_q, const int2 *s_meta, int K, uint8_t *out) {
    for (int b = threadIdx.x; b < K / 32; b += XG_THREADS) {
        uint16_t *dst = (uint16_t *)(out + (size_t)b * 34);
        dst[0] = f2h(__int_as_float(s_meta[b].x));
        for (int i = 0; i < 8; i++) {
            const uint32_t q = ((const uint32_t *)s_q)[act_dw(b * 8 + i, K >> 6)];
            dst[1 + 2 * i] = (uint16_t)(q & 0xFFFFu); dst[2 + 2 * i] = (uint16_t)(q >> 16);
        }
    }
}

// ---- phase 1: a lane's block pair of one weight row -> partial sums and scale products in LDS -------------------------
// x[0..3]: the 64 int8 activations of the pair (16 bytes each), mm / mm2: their {scale bits, sum q} (see load_act_frag),
// n8[i] = -8 * (sum of the four bytes of activation dword i): folds the -8 of the low Q4_0 nibbles into the accumulator
// input of v_dot4, so that each partial sum is sum (n - 8) * q exactly as sub_epi8 / maddubs / madd form it.  High nibbles stay where they are: with their sign bit turned
// they are 16 (n - 8) as signed bytes, one instruction instead of two, and accumulators 0..3 are walked times 16, which moves no rounding (every term is a
// multiple of 2^-48 below 2^56 or not finite).  down 9.22 -> 8.50 us, qkv 10.73 -> 10.50, gate|up 14.8 -> 14.6.
// slot: this row's LDS record; pl: the pair's index within the slab (= lane).
template <int WT>
static __device__ __forceinline__ void xg_phase1(const uint32_t *w, const act_frag<1> &f, const int (&n8)[16], int p, int pl, float *slot) {
    constexpr int NCH = xg_traits<WT>::NCH;
    float *P = slot, *D = slot + NCH * (XG_NBS + 4);
    const int4 x0 = f.x[0][0], x1 = f.x[0][1], x2 = f.x[0][2], x3 = f.x[0][3], mm = f.mm[0], mm2 = f.mm2[0];
    if constexpr (WT == SPY_HIP_Q4_0 || WT == SPY_HIP_Q8_0) {
        int pa[8], pb[8];
        float sA, sB;
        if constexpr (WT == SPY_HIP_Q4_0) {
            sA = h2f((uint16_t)(w[0] & 0xFFFFu)) * __int_as_float(mm.x); sB = h2f((uint16_t)(w[4] >> 16)) * __int_as_float(mm.z);
            const uint32_t a[4] = {__builtin_amdgcn_alignbit(w[1], w[0], 16), __builtin_amdgcn_alignbit(w[2], w[1], 16),
                                   __builtin_amdgcn_alignbit(w[3], w[2], 16), __builtin_amdgcn_alignbit(w[4], w[3], 16)};
            const int xa[4] = {x0.x, x0.y, x0.z, x0.w}, xb[4] = {x1.x, x1.y, x1.z, x1.w}, xc[4] = {x2.x, x2.y, x2.z, x2.w}, xd[4] = {x3.x, x3.y, x3.z, x3.w};
#pragma unroll
            for (int k = 0; k < 4; k++) {
                // accumulators 4..7: low nibbles against elements 0..15; 0..3: high nibbles against 16..31 (vec_dot.h:62-78)
                pa[4 + k] = __builtin_amdgcn_sdot4((int)(a[k] & 0x0F0F0F0Fu), xa[k], n8[k], true);
                pa[k]     = __builtin_amdgcn_sdot4((int)((a[k] & 0xF0F0F0F0u) ^ 0x80808080u), xb[k], 0, true);
                pb[4 + k] = __builtin_amdgcn_sdot4((int)(w[5 + k] & 0x0F0F0F0Fu), xc[k], n8[8 + k], true);
                pb[k]     = __builtin_amdgcn_sdot4((int)((w[5 + k] & 0xF0F0F0F0u) ^ 0x80808080u), xd[k], 0, true);
            }
        } else {
            sA = h2f((uint16_t)(w[0] & 0xFFFFu)) * __int_as_float(mm.x); sB = h2f((uint16_t)(w[8] >> 16)) * __int_as_float(mm.z);
            const int xa[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w}, xb[8] = {x2.x, x2.y, x2.z, x2.w, x3.x, x3.y, x3.z, x3.w};
#pragma unroll
            for (int l = 0; l < 8; l++) {               // accumulator l: elements 4l..4l+3 (vec_util.h:126-132)
                pa[l] = __builtin_amdgcn_sdot4((int)__builtin_amdgcn_alignbit(w[l + 1], w[l], 16), xa[l], 0, true);
                pb[l] = __builtin_amdgcn_sdot4((int)w[9 + l], xb[l], 0, true);
            }
        }
#pragma unroll
        for (int l = 0; l < 8; l++) *(float2 *)(P + l * (XG_NBS + 4) + 2 * pl) = make_float2((float)pa[l], (float)pb[l]);
        *(float2 *)(D + 2 * pl) = make_float2(sA, sB);
    } else if constexpr (WT == SPY_HIP_Q4_K) {
        // the two sub-blocks of the lane: term = d * float(sc * isum) - dmin * float(m * sum q), scale = d_x (one accumulator per row)
        const int j = p & 3, a = 2 * j;
        const float d = h2f((uint16_t)(w[0] & 0xFFFFu)), dmin = h2f((uint16_t)(w[0] >> 16));
        int scA, mA, scB, mB;
        if (j < 2) {
            scA = byte_of3(w[1], w[2], w[3], a) & 63;     mA = byte_of3(w[1], w[2], w[3], a + 4) & 63;
            scB = byte_of3(w[1], w[2], w[3], a + 1) & 63; mB = byte_of3(w[1], w[2], w[3], a + 5) & 63;
        } else {
            const uint32_t hA = byte_of3(w[1], w[2], w[3], a + 4), hB = byte_of3(w[1], w[2], w[3], a + 5);
            scA = (hA & 0x0F) | ((byte_of3(w[1], w[2], w[3], a - 4) >> 6) << 4); mA = (hA >> 4) | ((byte_of3(w[1], w[2], w[3], a) >> 6) << 4);
            scB = (hB & 0x0F) | ((byte_of3(w[1], w[2], w[3], a - 3) >> 6) << 4); mB = (hB >> 4) | ((byte_of3(w[1], w[2], w[3], a + 1) >> 6) << 4);
        }
        int iA = 0, iB = 0;
        const int xa[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w}, xb[8] = {x2.x, x2.y, x2.z, x2.w, x3.x, x3.y, x3.z, x3.w};
#pragma unroll
        for (int i = 0; i < 8; i++) {
            iA = __builtin_amdgcn_sdot4((int)(w[4 + i] & 0x0F0F0F0Fu), xa[i], iA, false);
            iB = __builtin_amdgcn_sdot4((int)((w[4 + i] >> 4) & 0x0F0F0F0Fu), xb[i], iB, false);
        }
        const float posA = d * (float)__mul24(scA, iA), negA = dmin * (float)__mul24(mA, mm.y);
        const float posB = d * (float)__mul24(scB, iB), negB = dmin * (float)__mul24(mB, mm.w);
        *(float2 *)(P + 2 * pl) = make_float2(posA - negA, posB - negB);
        *(float2 *)(D + 2 * pl) = make_float2(__int_as_float(mm.x), __int_as_float(mm.z));
    } else {
        // Q6_K: lane (n, e) holds the 16-element halves e of the four Q8_0 blocks 4n .. 4n+3 of its super-block; the other
        // halves are in the neighbouring lane.  term of block t = float(sc[2t] * isum(t, 0) + sc[2t+1] * isum(t, 1)), scale = d_x * d
        const uint32_t *qa = w, *qb = w + 4, *qh = w + 8;
        const uint32_t s0 = w[12], s1 = w[13];
        const int e = p & 1;
        const float d = h2f((uint16_t)(w[14] & 0xFFFFu));
        int isum[4] = {0, 0, 0, 0};
        const int xm[4][4] = {{x0.x, x0.y, x0.z, x0.w}, {x1.x, x1.y, x1.z, x1.w}, {x2.x, x2.y, x2.z, x2.w}, {x3.x, x3.y, x3.z, x3.w}};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t h = qh[i];
            isum[0] = __builtin_amdgcn_sdot4((int)q6_m32((qa[i] & 0x0F0F0F0Fu) | ((h & 0x03030303u) << 4)), xm[0][i], isum[0], false);
            isum[1] = __builtin_amdgcn_sdot4((int)q6_m32((qb[i] & 0x0F0F0F0Fu) | ((h & 0x0C0C0C0Cu) << 2)), xm[1][i], isum[1], false);
            isum[2] = __builtin_amdgcn_sdot4((int)q6_m32(((qa[i] >> 4) & 0x0F0F0F0Fu) | (h & 0x30303030u)), xm[2][i], isum[2], false);
            isum[3] = __builtin_amdgcn_sdot4((int)q6_m32(((qb[i] >> 4) & 0x0F0F0F0Fu) | ((h >> 2) & 0x30303030u)), xm[3][i], isum[3], false);
        }
        int sv[4];
#pragma unroll
        for (int m = 0; m < 4; m++) {
            const int k = e + 2 * m;
            const int sc = (int)(int8_t)(((k < 4 ? s0 : s1) >> (8 * (k & 3))) & 0xFFu);
            const int v = __mul24(sc, isum[m]);
            sv[m] = v + __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xF, 0xF, true);          // + the neighbour lane's half (quad_perm [1,0,3,2]); integer, order-free
        }
        const float dx[4] = {__int_as_float(mm.x), __int_as_float(mm.z), __int_as_float(mm2.x), __int_as_float(mm2.z)};
        // lane e writes blocks m = 2e, 2e+1 of the four: global block 2p, 2p+1
        const float t0 = (float)(e ? sv[2] : sv[0]), t1 = (float)(e ? sv[3] : sv[1]);
        const float c0 = (e ? dx[2] : dx[0]) * d, c1 = (e ? dx[3] : dx[1]) * d;
        *(float2 *)(P + 2 * pl) = make_float2(t0, t1);
        *(float2 *)(D + 2 * pl) = make_float2(c0, c1);
    }
}

// ---- phase 2: one lane walks one accumulator over the blocks of a slab ------------------------------------------------
static __device__ __forceinline__ float xg_chain(const float *P, const float *D, int nblk, float acc) {
    // Eight blocks per group (an odd four at the end of a row has zeros behind it, which leave a sum that started at +0 as it is).  The 128-bit reads of a group are
    // requested two groups (sixteen dependent fmas, about the latency of an LDS read under load) before its fmas: three register sets in rotation, no copies.  Reads
    // beyond the last group are not used.
    // (Taking the scale products, which the eight lanes of a row share, from one lane per quad through DPP broadcasts cut the LDS
    // traffic but measured slower: 1.25 instead of 0.8 us per 128 blocks.)
    const int ng = (nblk + 7) >> 3;
    float4 p0[2], p1[2], p2[2], d0[2], d1[2], d2[2];
    auto ld = [&](float4 (&p)[2], float4 (&d)[2], int g) {
#pragma unroll
        for (int u = 0; u < 2; u++) { p[u] = *(const float4 *)(P + 8 * g + 4 * u); d[u] = *(const float4 *)(D + 8 * g + 4 * u); }
    };
    auto run = [&](const float4 (&p)[2], const float4 (&d)[2]) {
#pragma unroll
        for (int u = 0; u < 2; u++) { acc = fmaf(d[u].x, p[u].x, acc); acc = fmaf(d[u].y, p[u].y, acc); acc = fmaf(d[u].z, p[u].z, acc); acc = fmaf(d[u].w, p[u].w, acc); }
    };
    ld(p0, d0, 0);
    ld(p1, d1, 1);
    int g = 0;
#pragma unroll 1
    for (; g + 3 <= ng; g += 3) {
        ld(p2, d2, g + 2);
        __builtin_amdgcn_sched_barrier(0);
        run(p0, d0);
        __builtin_amdgcn_sched_barrier(0);
        ld(p0, d0, g + 3);
        __builtin_amdgcn_sched_barrier(0);
        run(p1, d1);
        __builtin_amdgcn_sched_barrier(0);
        ld(p1, d1, g + 4);
        __builtin_amdgcn_sched_barrier(0);
        run(p2, d2);
        __builtin_amdgcn_sched_barrier(0);
    }
    if (g < ng) run(p0, d0);
    if (g + 1 < ng) run(p1, d1);
    return acc;
}

// hsum_float_8 over the eight lanes of an output element: (a0+a4)+(a2+a6) + (a1+a5)+(a3+a7); the operands of each
// addition commute, so the three exchanges leave the same bits in all eight lanes (vec_util.h:75-81)
static __device__ __forceinline__ float xg_hsum8(float acc) {
    acc += __shfl_xor(acc, 4, SPY_WAVE);
    acc += __shfl_xor(acc, 2, SPY_WAVE);
    acc += __shfl_xor(acc, 1, SPY_WAVE);
    return acc;
}

// ---- the kernel --------------------------------------------------------------------------------------------------------
// 1024 threads; wave w of the grid (gw) owns, per step, RPS rows:
//   EPI_RESID / EPI_STORE : rows gw * RPS + j + k * NW * RPS                              (NSTEP steps)
//   EPI_GATEUP            : rows i = gw + k * NW of W0 (gate) and of W1 (up), RPS / 2 pairs a step      (NSTEP steps)
//   EPI_QKV               : step 0: rows 2 gw, 2 gw + 1 of [W0; W1] (a RoPE pair), step 1 (K-quants: step 0): row gw of W2
// A step's rows of all 16 waves form one batch: phase 1 (all waves) -> barrier -> phase 2 (the first lanes, one per
// accumulator) -> barrier (none where every slab has slots of its own), per slab of 4096 elements of K; the accumulators stay in their lanes from slab to slab.
template <int WT, int NITK, int RPS, int NSTEP, int EPI, int WTV = WT>
__global__ __launch_bounds__(XG_THREADS) void xgemv_kernel(const float *x_in, const float *normw, const uint8_t *W0, const uint8_t *W1, const uint8_t *W2, const dev_state *st, int K_, int M,
                                                           xg_args a) {
    a.x_in = x_in; a.normw = normw; a.W0 = W0; a.W1 = W1; a.W2 = W2; a.st = st; a.K = K_; a.M = M;
    if constexpr (EPI == EPI_QKV) a.d = M;
    constexpr bool NORM = (EPI != EPI_RESID);
    constexpr int NCH = xg_traits<WT>::NCH, NCHV = xg_traits<WTV>::NCH;
    constexpr int NROW = EPI == EPI_QKV ? 3 : RPS * NSTEP;                  // rows per wave
    constexpr int SLOTF = xg_slot_floats(NCH > NCHV ? NCH : NCHV);
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    __shared__ float s_scale;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int NW = (int)gridDim.x * XG_WAVES, gw = (int)blockIdx.x * XG_WAVES + wave;
    const int K = a.K, npair = K / 64;
    const size_t RB = (size_t)spy_row_size(WT, K);

    // row index (within its matrix) and base of the wave's row r (0 .. NROW-1); rows beyond the matrix re-read the last one and are dropped in the epilogue
    auto row_of = [&](int r, bool &valid) -> int {
        if constexpr (EPI == EPI_QKV) { valid = gw < a.d; const int j = min(gw, a.d - 1); return r == 2 ? j : 2 * j - (2 * j < a.d ? 0 : a.d) + r; }
        else if constexpr (EPI == EPI_GATEUP) { const int u = gw + (r >> 1) * NW; valid = u < a.M; return min(u, a.M - 1); }
        else { const int u = (gw + (r / RPS) * NW) * RPS + (r % RPS); valid = u < a.M; return min(u, a.M - 1); }
    };
    auto row_ptr = [&](int r) -> const uint8_t * {
        bool v; int i = row_of(r, v);
#ifdef XDBG_SMALLROWS
        i &= 255;                                   // measurement build: every workgroup re-reads the same cached rows
#endif
        if constexpr (EPI == EPI_QKV) {
            if (r == 2) return a.W2 + (size_t)i * spy_row_size(WTV, K);
            return (2 * gw < a.d ? a.W0 : a.W1) + (size_t)i * RB;
        } else if constexpr (EPI == EPI_GATEUP) return ((r & 1) ? a.W1 : a.W0) + (size_t)i * RB;
        else return a.W0 + (size_t)i * RB;
    };

    // 1. the activation vector, 2. the first rows (issue_first): all unconditional, in this order (the compute unit serves its requests in order)
    float4 xv[NITK], wv[NORM ? NITK : 1];
#pragma unroll
    for (int j = 0; j < NITK; j++) {
        const int i = min(tid + j * XG_THREADS, K / 4 - 1);
        xv[j] = ((const float4 *)a.x_in)[i];
        if constexpr (NORM) wv[j] = ((const float4 *)a.normw)[i];
    }
    // Rows requested ahead of their use.  A wave waits in the issue stage while the memory queue is full, i.e. while the stream runs, and the barriers
    // of the norm wait for every wave: 2 rows of each of 16 waves (73 KB of Q4_0, 3.3 us of the stream) about cover the norm's sum.  qkv with 2 of 3
    // rows 10.4 us (all 3: 11.0; 1: 11.8), gate|up Q4_0 with 3 of 6 14.5 us (2: 15.1; 4: 15.3), Q4_K 11.8 (12.6; 12.35), Q8_0, whose rows are twice as long, with 2 19.8 us (3: 20.9;
    // 1: 22.3).  gate|up asks for its first row (37 KB, which the queue takes at once) right behind the activations (Q4_0 14.9 us without, Q8_0 20.4; two rows ahead of it: Q4_K 13.05); with less to
    // stream after the norm the other kernels lose by it (two rows ahead of it: 20 us and more).
    constexpr int DEPTH = EPI == EPI_GATEUP ? (WT == SPY_HIP_Q8_0 ? 2 : 3) : NROW < 2 ? NROW : 2, PRE = EPI == EPI_GATEUP ? 1 : 0;
    constexpr int RING = NROW < DEPTH + 1 ? NROW : DEPTH + 1;
    wtile<WT, NITK> t[RING];
    wtile<WTV, NITK> tv;
    auto issue = [&](int r) {
        if (EPI == EPI_QKV && r == 2) load_tile<WTV, 64, NITK>(tv, row_ptr(r), npair, lane);
        else load_tile<WT, 64, NITK>(t[r % RING], row_ptr(r), npair, lane);
    };
    // What the epilogue needs from memory is requested ahead where that pays: the residual of rows of several slabs with the activations (11008 columns Q4_0 9.7 -> 9.5 us,
    // Q6_K 11.85 -> 11.78; rows of one slab: 5.1 both ways, Q8_0 6.1 -> 6.3), the rotation of a pair ahead of the rows (qkv 10.82 -> 10.75; behind them 10.95).
    constexpr bool RS_AHEAD = EPI == EPI_RESID && NITK > 1;
    float rs = 0.0f;
    if constexpr (RS_AHEAD) { if (a.resid) rs = a.resid[min((int)blockIdx.x * XG_WAVES + tid / NCH % XG_WAVES, a.M - 1)]; }
    const int pos = EPI != EPI_QKV ? 0 : a.st ? a.st->pos : a.pos_imm;
    float2 cs = make_float2(0.0f, 0.0f);
    auto issue_first = [&]() {
        if constexpr (EPI == EPI_QKV)
            cs = *(const float2 *)(a.rope_tab + (size_t)(pos - a.rope_row0) * a.hd + ((2 * ((int)blockIdx.x * XG_WAVES + tid / ((NCH == 1 && NCHV == 1 ? 3 : 2) * NCH) % XG_WAVES)) & (a.hd - 1)));      // heads are 128 wide
        if constexpr (!NORM) __builtin_amdgcn_s_barrier();      // x of every wave ahead of every wave's rows in the compute unit's memory queue
#pragma unroll
        for (int r = 0; r < NROW; r++) if (r < DEPTH && r >= PRE) {
            // a row of several slabs: the first one ahead of the quantization, whose barrier waits for the issue, the next ones a slab ahead of their use
            // (11008 columns: Q4_0 11.8 -> 10.2 us, Q6_K 14.0 -> 11.9; two slabs ahead 10.9 and 13.0; with slots per slab Q6_K 10.48, two ahead 12.1, all 13.1)
            if constexpr (NITK > 1) load_slab<WT, 64, NITK>(t[0], row_ptr(0), npair, lane, 0);
            else issue(r);
        }
    };
    if constexpr (PRE > 0) {
        __builtin_amdgcn_s_barrier();
        issue(0);
    }

    // 3. stage the activations (the first rows are requested inside: after the group sums of the norm, or at once)
    int8_t *s_q = (int8_t *)smem;
    int2 *s_meta = (int2 *)(smem + staged_q_bytes(K));
    float *s_part = (float *)(smem + ((staged_bytes(K) + 15) & ~(size_t)15));      // row slots; the group sums of the norm use the same bytes before
    XSTAMP(a.dbg, 16);
    xg_stage<NITK, NORM>(xv, wv, K, a.eps, s_q, s_meta, s_part, &s_scale, issue_first);
    XSTAMP(a.dbg, 17);
    if (a.q8_dump && blockIdx.x == 0) xg_dump_q8(s_q, s_meta, K, a.q8_dump);
    staged_act act; act.q = s_q; act.meta = s_meta;

    // K-quant rows have one accumulator and small slots: all rows of a wave lie in LDS side by side and are walked together, once, instead of one walk (0.5 us) and two
    // barriers per step.  In a pass gate|up Q4_K 12.99 -> 11.76 us, qkv Q4_K with Q6_K 11.07 -> 10.22; the head (8 rows) is the same either way and keeps its two steps.
    constexpr bool ONE = EPI == EPI_QKV && NCH == 1 && NCHV == 1;
    constexpr int NSTEPS = EPI == EPI_QKV ? (ONE ? 1 : 2) : NSTEP;
    constexpr bool SLABS = xg_slabs(NCH, NITK);
    static_assert(NITK == 1 || NROW == 1, "rows longer than one slab are walked one row per wave");
    static_assert(WT == WTV || (NCH == 1 && NCHV == 1), "n8 and the factor 16 of Q4_0's high nibbles follow WT in every step");
    act_frag<1> af, av;
    int n8[16];
    // gate|up: the SiLU table's answers are awaited after the last step only (Q4_0 15.38 -> 15.08 us, Q4_K 14.26 -> 13.86; Q8_0 has no registers left for it: 21.3 -> 21.5)
    constexpr bool LATE = EPI == EPI_GATEUP && WT != SPY_HIP_Q8_0;
    float up[LATE ? NSTEP : 1], sl[LATE ? NSTEP : 1];
#pragma unroll
    for (int step = 0; step < NSTEPS; step++) {
        const int r0 = EPI == EPI_QKV ? 2 * step : step * RPS;                  // first row of the step
        const int rows = EPI == EPI_QKV ? (ONE ? 3 : 2 - step) : RPS;
        const int nch = EPI == EPI_QKV && step == 1 ? NCHV : NCH;
        const int chains = XG_WAVES * rows * nch;
        float acc = 0.0f;
#pragma unroll
        for (int it = 0; it < NITK; it++) {
            const int nblk = min(XG_NBS, K / 32 - it * XG_NBS);                // blocks of this slab
            if (nblk > 0) {
                const int p = it * 64 + lane;
                // this lane's activations of the slab (the same for every row) and the -8 * sum q per dword: read once where the
                // rows are one slab long (every step uses the same ones), per slab otherwise
                if (NITK > 1 || step == 0) {
                    if (p < npair) {
                        load_act_frag<WT, 1>(af, act, npair, p);
                        if constexpr (WT == SPY_HIP_Q4_0) {
                            const int xs[16] = {af.x[0][0].x, af.x[0][0].y, af.x[0][0].z, af.x[0][0].w, af.x[0][1].x, af.x[0][1].y, af.x[0][1].z, af.x[0][1].w,
                                                af.x[0][2].x, af.x[0][2].y, af.x[0][2].z, af.x[0][2].w, af.x[0][3].x, af.x[0][3].y, af.x[0][3].z, af.x[0][3].w};
#pragma unroll
                            for (int i = 0; i < 16; i++) n8[i] = -8 * __builtin_amdgcn_sdot4(xs[i], 0x01010101, 0, false);
                        }
                    }
                }
                if (it + 1 < NITK) load_slab<WT, 64, NITK>(t[0], row_ptr(0), npair, lane, it + 1);
                if constexpr (WTV != WT) { if ((ONE || step == 1) && p < npair) load_act_frag<WTV, 1>(av, act, npair, p); }
#pragma unroll
                for (int j = 0; j < rows; j++) {
                    const int r = r0 + j;
                    if (it == 0 && r + DEPTH < NROW) issue(r + DEPTH);            // its ring slot held row r - 1, multiplied in the previous step
                    float *slot = s_part + (size_t)((SLABS ? it * XG_WAVES : 0) + wave * rows + j) * SLOTF;
                    if (p < npair) {
                        if (EPI == EPI_QKV && r == 2) { if constexpr (WTV != WT) xg_phase1<WTV>(tv.w[it], av, n8, p, lane, slot); else xg_phase1<WTV>(tv.w[it], af, n8, p, lane, slot); }
                        else xg_phase1<WT>(t[r % RING].w[it], af, n8, p, lane, slot);
                    } else if (p < ((npair + 3) & ~3)) {                      // xg_chain's odd four blocks
                        for (int l = 0; l <= nch; l++) *(float2 *)(slot + l * (XG_NBS + 4) + 2 * lane) = make_float2(0.0f, 0.0f);
                    }
                }
                XSTAMP(a.dbg, 18 + 3 * (step * NITK + it));
                __syncthreads();
                XSTAMP(a.dbg, 19 + 3 * (step * NITK + it));
                if (tid < chains) {
                    const int slot_i = tid / nch, l = tid % nch;
                    const float *slot = s_part + (size_t)((SLABS ? it * XG_WAVES : 0) + slot_i) * SLOTF;
                    acc = xg_chain(slot + l * (XG_NBS + 4), slot + nch * (XG_NBS + 4), nblk, acc);
                }
                XSTAMP(a.dbg, 20 + 3 * (step * NITK + it));
                if (step + 1 < NSTEPS || (!SLABS && it + 1 < NITK)) __syncthreads();       // nothing is written behind the last walk
            }
        }
        // epilogue of the step: the lanes that walked accumulator 0 of a row hold its total after the tree
        if (nch == 8) {
            if constexpr (WT == SPY_HIP_Q4_0) acc *= tid & 4 ? 1.0f : 0.0625f;    // accumulators 0..3 were walked times 16 (xg_phase1)
            acc = xg_hsum8(acc);
        }
        const bool owner = tid < chains && (tid % nch) == 0;
        const int slot_i = tid / nch;                                         // = wave_of_row * rows + j
        const int ow = slot_i / rows, oj = slot_i % rows;                      // the wave that owned the row and its index in the step
        const int ogw = (int)blockIdx.x * XG_WAVES + ow;
        if constexpr (EPI == EPI_RESID || EPI == EPI_STORE) {
            const int u = (ogw + step * NW) * RPS + oj;
            if (owner && u < a.M) a.out[u] = (EPI == EPI_RESID && a.resid) ? acc + (RS_AHEAD ? rs : a.resid[u]) : acc;       // Add(KQV_linear, x) / Add(ffn_out, ffn_input); no resid: the MatMul alone
        } else if constexpr (EPI == EPI_GATEUP) {
            const float u = __shfl_xor(acc, nch, SPY_WAVE);                    // the row after (up_i) sits nch lanes further
            const int i = ogw + (step * (RPS / 2) + (oj >> 1)) * NW;
            if constexpr (LATE) {
                up[step] = u;
                if (owner && (oj & 1) == 0 && i < a.M) sl[step] = a.lut[65536 + f2h(acc)];
            } else if (owner && (oj & 1) == 0 && i < a.M) a.out[i] = u * a.lut[65536 + f2h(acc)];       // Mul(ffn_up, Silu(ffn_gate)) (ffn.cpp:24-35, non-linear.cpp:11-14)
        } else {
            if (step == 0) {
                const float x1 = ONE ? __shfl_down(acc, 1, SPY_WAVE) : __shfl_xor(acc, nch, SPY_WAVE);      // (ONE: 48 lanes of one wave)
                if (owner && oj == 0 && ogw < a.d) {
                    const float c = cs.x, sn = cs.y;
                    // (x0, x1) -> (x0*c - x1*s, x0*s + x1*c), every product rounded (non-linear.cpp:349-364)
                    const float pa_ = acc * c, pb_ = x1 * sn, pc_ = acc * sn, pd_ = x1 * c;
                    const uint32_t pr = (uint32_t)f2h(pa_ - pb_) | ((uint32_t)f2h(pc_ + pd_) << 16);
                    if (2 * ogw < a.d) ((uint32_t *)a.q16)[ogw] = pr;                                  // attn_score rounds Q to fp16 (mat.cpp:37)
                    else ((uint32_t *)(a.kc + (size_t)pos * a.d))[ogw - a.d / 2] = pr;                 // KCache_cpy: [token][head][hd]
                }
            }
            if (ONE ? oj == 2 : step == 1) {
                if (owner && ogw < a.d) a.vc[(size_t)ogw * a.n_ctx + pos] = f2h(acc);                 // VCache_cpy: [d][C] column pos
            }
        }
    }
    if constexpr (LATE) {
        const bool owner = tid < XG_WAVES * RPS * NCH && tid % (2 * NCH) == 0;
#pragma unroll
        for (int step = 0; step < NSTEP; step++) {
            const int i = (int)blockIdx.x * XG_WAVES + tid / (RPS * NCH) + (step * (RPS / 2) + tid / (2 * NCH) % (RPS / 2)) * NW;
            if (owner && i < a.M) a.out[i] = up[step] * sl[step];
        }
    }
}

// ---- attention scores in the order of Dot<FP16,FP16> -------------------------------------------------------------------
// result = tail + simd as vec_dot.h:124-145 has it for n = 128: accumulators sum[j][l] over the chunks i = 0, 32, 64 (i + 32 < n), the reduction tree of
// FP16::block_reduce, then the scalar tail over elements 96..127.  Stored: t = dot * scale (mask 0, then * scale: non-linear.cpp:141-150).
typedef uint32_t xp_u4 __attribute__((ext_vector_type(4)));
// ---- what the attention kernels of one token (the two below, attn_short.hip) share: the order of Dot<FP16,FP16> lies here and nowhere else.  A product of two fp16
// values is exact in fp32, so `sum + a * b` is the fma it is written as.
// eight elements of a key or query, packed in four words, onto the eight accumulators l of one (chunk, j)
static __device__ __forceinline__ void xa_fma8(float (&sum)[8], const uint4 kv, const uint4 qv) {
    const uint32_t kw[4] = {kv.x, kv.y, kv.z, kv.w}, qw[4] = {qv.x, qv.y, qv.z, qv.w};
#pragma unroll
    for (int e = 0; e < 4; e++) {
        sum[2 * e] = fmaf(h2f((uint16_t)(kw[e] & 0xFFFFu)), h2f((uint16_t)(qw[e] & 0xFFFFu)), sum[2 * e]);
        sum[2 * e + 1] = fmaf(h2f((uint16_t)(kw[e] >> 16)), h2f((uint16_t)(qw[e] >> 16)), sum[2 * e + 1]);
    }
}
// eight elements of the scalar tail, one after the other
static __device__ __forceinline__ float xa_tail8(float tail, const uint4 kv, const uint4 qv) {
    const uint32_t kw[4] = {kv.x, kv.y, kv.z, kv.w}, qw[4] = {qv.x, qv.y, qv.z, qv.w};
#pragma unroll
    for (int e = 0; e < 4; e++) {
        tail = fmaf(h2f((uint16_t)(kw[e] & 0xFFFFu)), h2f((uint16_t)(qw[e] & 0xFFFFu)), tail);
        tail = fmaf(h2f((uint16_t)(kw[e] >> 16)), h2f((uint16_t)(qw[e] >> 16)), tail);
    }
    return tail;
}
// first two steps of FP16::block_reduce where four adjacent lanes hold j = 0 .. 3: sum[0] += sum[2], sum[1] += sum[3]; sum[0] += sum[1]
static __device__ __forceinline__ void xa_quad(float (&sum)[8]) {
#pragma unroll
    for (int l = 0; l < 8; l++) {
        sum[l] += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(sum[l]), 0x4E, 0xF, 0xF, true));        // quad_perm [2, 3, 0, 1]
        sum[l] += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(sum[l]), 0xB1, 0xF, 0xF, true));        // quad_perm [1, 0, 3, 2]
    }
}
// its last three
static __device__ __forceinline__ float xa_tree8(const float (&sum)[8]) {
    const float u0 = sum[0] + sum[4], u1 = sum[1] + sum[5], u2 = sum[2] + sum[6], u3 = sum[3] + sum[7];
    const float v0 = u0 + u1, v1 = u2 + u3;
    return v0 + v1;
}
// Dot<FP16,FP16> of a key and its query by four adjacent lanes: lane `part` has elements 32 i + 8 part .. + 7 of either in piece i; the tail goes down the four lanes, eight
// elements each, so that the result is in the lane of part 3
static __device__ __forceinline__ float xa_dot4(const uint4 (&kv)[4], const uint4 (&q)[4]) {
    float sum[8];
#pragma unroll
    for (int l = 0; l < 8; l++) sum[l] = 0.0f;
#pragma unroll
    for (int i = 0; i < 3; i++) xa_fma8(sum, kv[i], q[i]);
    xa_quad(sum);
    const float simd = xa_tree8(sum);
    float tail = 0.0f;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        if (j) tail = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(tail), 0x90, 0xF, 0xF, true));      // quad_perm [0, 0, 1, 2]
        tail = xa_tail8(tail, kv[3], q[3]);
    }
    return tail + simd;
}
// a group of four of std::reduce's running sum
static __device__ __forceinline__ float xa_group(const float4 v) {
    const float v1 = v.x + v.y, v2 = v.z + v.w;
    return v1 + v2;
}
// block_reduce of 32 accumulators 8 j + l that 32 lanes hold: sum[0] += sum[2], sum[1] += sum[3] (lane ^ 16); sum[0] += sum[1] (^ 8); t_l = sum[0][l] + sum[0][l + 4] (^ 4);
// t_0 + t_1, t_2 + t_3 (^ 1); (t_0 + t_1) + (t_2 + t_3) (^ 2); inside a row of 16 as rotations where the values are periodic already
static __device__ __forceinline__ float xa_tree32(float acc) {
    const auto sw = __builtin_amdgcn_permlane16_swap(__float_as_uint(acc), __float_as_uint(acc), false, false);
    acc = __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
#define XP_ADD(CTRL) acc += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(acc), CTRL, 0xF, 0xF, true));
    XP_ADD(0x128) XP_ADD(0x124) XP_ADD(0xB1) XP_ADD(0x4E)
#undef XP_ADD
    return acc;
}
// the scalar tail of P.V^T: the first ntail of 32 elements tv . tq onto tail, one after the other.  A macro because the steps stay branches that way: in a function the
// compiler makes them selections, which doubles the chain.
#define XA_TAIL32(tail, tv, tq, ntail) \
    _Pragma("unroll") for (int e = 0; e < 32; e++) { \
        const uint32_t wv = tv[e >> 3][(e >> 1) & 3], wq = tq[e >> 3][(e >> 1) & 3]; \
        if (e < ntail) tail = fmaf(h2f((uint16_t)(e & 1 ? wv >> 16 : wv & 0xFFFFu)), h2f((uint16_t)(e & 1 ? wq >> 16 : wq & 0xFFFFu)), tail); \
    }
#define XA_MAX_CTX 4736                                 // longest cache, most heads of the attention kernels of one token
#define XA_MAX_HEAD 32
#define XS_THREADS 1024
#define XS_NU 3                                         // units of a wave in flight (2 and 4: the same)
// A unit is 16 keys, four adjacent lanes per key: lane `part` has the 16 bytes of accumulators (part, l) of every chunk, straight from memory, and its head's part of q
// in registers.  The tail goes down the four lanes, eight elements each.  The heads are dealt out over eight groups (heads g, g + 8, ...), a unit has one, two or four
// of its group's and tokens to match (attn_reach.h); workgroup b takes group b modulo 8, so that a head's keys are read and its scores written by one XCD, the one that reads
// them next where the cache is long (in a pass 4100 tokens 8.58 -> 8.26 us against units of 16 heads of one token, 2060 5.62 -> 5.17, 1000 and 600 the same).  A place without a head
// repeats the group's first and a group without heads has no work (with the last head in such places: 24 heads, scores and product of 4100 tokens 16.1 us, now 15.1, 2060 11.9 and
// 11.3).  A group's tokens are
// dealt out evenly over its workgroups, a workgroup's over its waves.
// What bounds it: the keys at 5.5 TB/s behind launch, position and first wait (4100 tokens: 33.6 MB in 8.05 us).  Through LDS, one thread per key, the dots began when the last
// key of a round was there and then took 1.6 us: 4100 tokens 9.9, 2060 6.7, 1000 and 600 4.83 us (now 4.75); here a wave's
// dots follow its own keys, and what is left after the last ones is one chain of 32 fmas.
// kc is not a restrict pointer on purpose: the loads must stay where they are written, ahead of the dots of the units before.
template <int DUMMY>
__global__ __launch_bounds__(XS_THREADS) void xattn_scores_kernel(const dev_state *st, int pos_imm, const uint16_t *__restrict__ q16, const uint16_t *kc,
                                                                  float *__restrict__ scores, int n_head, int n_ctx, float scale) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), part = lane & 3;
    const int nb = (int)gridDim.x >> 3, tb = (int)blockIdx.x >> 3, hg = (int)blockIdx.x & 7;
    if (hg >= n_head) return;
    const int hs = xs_log2(n_head), nt = 16 >> hs;
    const int n_kv = (st ? st->pos : pos_imm) + 1;
    const int tpw = xs_share(n_kv, nb, nt), t_end = min(n_kv, (tb + 1) * tpw);
    int t = tb * tpw + wave * nt;
    if (tb >= nb || t >= t_end) return;
    const int slot = (lane >> 2) & ((1 << hs) - 1), h = xs_head(n_head, hg, slot), dt = lane >> (2 + hs);
    const size_t d = (size_t)n_head * 128;
    const uint16_t *qp = q16 + h * 128 + part * 8, *kp = kc + h * 128 + part * 8;
    uint4 q[4];
    xp_u4 k[XS_NU][4];
#pragma unroll
    for (int i = 0; i < 4; i++) q[i] = *(const uint4 *)(qp + 32 * i);
    auto request = [&](int u, int tt) {
        if (tt >= t_end) return;
#pragma unroll
        for (int i = 0; i < 4; i++) k[u][i] = *(const xp_u4 *)(kp + (size_t)min(tt + dt, t_end - 1) * d + 32 * i);
    };
#pragma unroll
    for (int u = 0; u < XS_NU; u++) request(u, t + 16 * nt * u);
    for (; t < t_end; t += 16 * nt * XS_NU) {
#pragma unroll
        for (int u = 0; u < XS_NU; u++) {
            const int tt = t + 16 * nt * u;
            if (tt >= t_end) break;
            uint4 kv[4];
#pragma unroll
            for (int i = 0; i < 4; i++) kv[i] = make_uint4(k[u][i].x, k[u][i].y, k[u][i].z, k[u][i].w);
            const float dot = xa_dot4(kv, q);
            if (part == 3 && hg + 8 * slot < n_head && tt + dt < t_end) scores[(size_t)h * n_ctx + tt + dt] = dot * scale;
            request(u, tt + 16 * nt * XS_NU);
        }
    }
}

// ---- softmax + P.V^T in the host order ---------------------------------------------------------------------------------
// One 1024-thread workgroup per (head, 16 rows of V^T), the head first in the grid, so that the eight of a head are on one XCD, the one that wrote its scores
// (4100 tokens 10.04 -> 9.81 us in a pass, 2060 8.46 -> 8.11, 1000 and 600 the same).  Waves 0..7 do the softmax and then the product, waves 8..15 bring two rows of V^T each into LDS meanwhile.
// Softmax (non-linear.cpp:129-180): m = max t; e = exp_table[fp16(t - m)] (exact_exp.cuh); sum = std::reduce(e) = groups of four added to
// one running sum, then the last n % 4 elements; p = e * (1 / sum), rounded to fp16 for the product (mat.cpp:37).
// P.V^T (vec_dot.h:124-145 with n = n_kv): output row r has 4 x 8 accumulators, accumulator (j, l) adds elements
// 32 i + 8 j + l for every chunk with 32 i + 32 < n_kv.  32 lanes hold the accumulators of one row (two rows per wave); tree; scalar tail (the
// last 1..32 elements, by the lane of accumulator 0).
// Rows and probabilities lie in LDS by accumulator, not by token, so that a lane reads the elements of eight of its steps at once: a wave's 128-bit read costs the
// compute unit 4 clocks, a 16-bit one 2.7 (measured), and the walk took 2 us of them, 0.6 now.  The rows are turned on the way: a lane
// asks for the same octet of eight chunks, which 32 byte permutes turn into eight octets of one accumulator each.
// What bounds it: from 3500 tokens or so on the rows (16 per compute unit at 24 B/ns, then 0.6 us to write them to LDS and 0.6 to walk them), below the softmax's
// chain of latencies.  The waves of the softmax meet on counters in LDS: at a workgroup barrier they would wait until the other eight have
// asked for all their rows, which takes as long as the rows take to come.  All 16 waves taking part in both, with the table's gathers in the same memory
// queue as the rows: in a pass 4100 tokens 13.6 us, 2060 11.1, 1000 9.5, 600 8.1; now 9.8, 8.1, 7.0, 6.6.  One launch after the other (scores and list in the L2), before
// arguments came in registers: 4100 tokens 12.7 us, 3000 11.5, 2060 9.4, 600 7.5; this 10.2, 8.8, 8.2, 6.7; this layout and list but all waves in both: 11.5, 9.3, 8.5, 6.8; scores asked
// for before the position is known: 10.7, 9.2, 8.3, 6.8.
#define XP_THREADS 1024
#define XP_NP 10                           // 16-byte pieces per lane of a V^T row
#define XP_NG 3                            // groups of four scores per thread of the softmax
// Where an element lies in LDS: chunk c, accumulator a at [c & 1][4 (a & 7) + (a >> 3)][c >> 1], the last index
// xattn_pv_sa long, an odd number of 16-byte pieces (32 lanes, 16 at a time, on banks of their own); up to XP_LAY tokens, those behind them as they come.
#define XP_LAY 4608
static __host__ __device__ inline int xattn_pv_sa(int n_ctx) { return (((n_ctx < XP_LAY ? n_ctx : XP_LAY) + 511) / 512 * 8) | 8; }
static __host__ __device__ inline int xattn_pv_row(int n_ctx) { return 64 * xattn_pv_sa(n_ctx) + (n_ctx > XP_LAY ? XA_MAX_CTX - XP_LAY : 0) + 32; }       // halfs of a row: laid out, behind XP_LAY, its last chunk
// what the softmax works in: group sums, the list of exact_exp.cuh; behind the rows, or over the last of them where LDS is full
#define XP_LDS (160 * 1024 - 256)
static __host__ __device__ inline int xattn_pv_soft(int n_ctx) { return (n_ctx / 4 + 31) / 32 * 160 + XE_WORDS * 4; }
static __host__ __device__ inline int xattn_pv_soft_at(int n_ctx) {
    const int end = 17 * xattn_pv_row(n_ctx) * 2, at = XP_LDS - xattn_pv_soft(n_ctx);
    return end < at ? end : at & ~15;
}
static inline size_t xattn_pv_lds(int n_ctx) {
    const int end = 17 * xattn_pv_row(n_ctx) * 2, soft = xattn_pv_soft_at(n_ctx) + xattn_pv_soft(n_ctx);
    return end > soft ? end : soft;
}
// Arrival and wait of waves of one workgroup on a counter in LDS (all of them resident, and none waits before it has arrived).  Every lane's stores lie before the count, so every lane
// has the release; the count itself, by one of them, needs none of its own.
static __device__ __forceinline__ void xp_arrive(uint32_t *c) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_wave_barrier();
    if ((threadIdx.x & 63) == 0) __hip_atomic_fetch_add(c, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
static __device__ __forceinline__ void xp_await(uint32_t *c, uint32_t n) { while (__hip_atomic_load(c, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP) < n) __builtin_amdgcn_s_sleep(1); }
template <int DUMMY>
__global__ __launch_bounds__(XP_THREADS) void xattn_pv_kernel(const dev_state *st, int pos_imm, const float *__restrict__ scores, const uint16_t *vc,
                                                              float *attn_out, const float *__restrict__ lut, int n_ctx, long long *dbg) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    __shared__ float s_red[8], s_rem[4];
    __shared__ float s_sum;
    __shared__ uint32_t s_cnt[3];
    XSTAMP(dbg, 0);
    const int n_kv = (st ? st->pos : pos_imm) + 1;
    const int hd_ = blockIdx.x, dgrp = blockIdx.y;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int SA = xattn_pv_sa(n_ctx), RS = xattn_pv_row(n_ctx), REST = RS - 64 * SA - 32;
    uint16_t *s_p = (uint16_t *)smem, *s_v = s_p + RS;                // the probabilities as fp16, 16 rows of V^T
    float *s_grp = (float *)(smem + xattn_pv_soft_at(n_ctx));
    uint32_t *s_code = (uint32_t *)(s_grp + (n_ctx / 4 + 31) / 32 * 40);
    const int last_piece = (n_kv - 1) >> 3, nfull = (n_kv - 1) / 32;  // chunks with 32 i + 32 < n_kv
    const int ngrp = n_kv / 4, nall = (n_kv + 3) / 4;
    if (tid < 3) s_cnt[tid] = 0;
    typedef float f4 __attribute__((ext_vector_type(4), aligned(4)));
    f4 v[XP_NG];
    xp_u4 cd = {0, 0, 0, 0};
    if (wave < 8) {
        const float *srow = scores + (size_t)hd_ * n_ctx;
#pragma unroll
        for (int u = 0; u < XP_NG; u++) {
            const int g = min(tid + 512 * u, nall - 1);
            if (512 * u < nall) {
                if (4 * g + 3 < n_ctx) v[u] = *(const f4 *)(srow + 4 * g);
                else v[u] = f4{srow[4 * g], srow[min(4 * g + 1, n_ctx - 1)], srow[min(4 * g + 2, n_ctx - 1)], 0.0f};
            }
        }
        if (tid < XE_WORDS / 4) cd = ((const xp_u4 *)(lut + XE_AT))[tid];
    }
    __syncthreads();
    if (wave < 8) {
        // ---- softmax ----
        if (tid < XE_WORDS / 4) ((xp_u4 *)s_code)[tid] = cd;
        float mx = -INFINITY;
#pragma unroll
        for (int u = 0; u < XP_NG; u++)
            if (512 * u < nall) {
                const int left = n_kv - 4 * min(tid + 512 * u, nall - 1);          // behind the last token: -inf, which leaves 0
#pragma unroll
                for (int i = 1; i < 4; i++) v[u][i] = i < left ? v[u][i] : -INFINITY;
                mx = fmaxf(fmaxf(fmaxf(mx, v[u][0]), fmaxf(v[u][1], v[u][2])), v[u][3]);
            }
        mx = wave_max(mx);
        if (lane == 0) s_red[wave] = mx;
        xp_arrive(s_cnt);
        xp_await(s_cnt, 8);
        mx = s_red[0];
#pragma unroll
        for (int w = 1; w < 8; w++) mx = fmaxf(mx, s_red[w]);
        XSTAMP(dbg, 1);
#pragma unroll
        for (int u = 0; u < XP_NG; u++) {
            const int g = tid + 512 * u;
            if (512 * u + 64 * wave < nall) {
                float e[4];
                bool any = false;
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    bool ask;
                    e[i] = xe_exp(f2h(mx - v[u][i]), s_code, ask);
                    any |= ask;
                }
                if (__any(any)) {
#pragma unroll
                    for (int i = 0; i < 4; i++) e[i] = lut[f2h(v[u][i] - mx)];
                }
                v[u] = f4{e[0], e[1], e[2], e[3]};
                if (g < ngrp) s_grp[xg_seg_at(g)] = xa_group(make_float4(e[0], e[1], e[2], e[3]));
                else if (g < ((ngrp + 31) & ~31)) s_grp[xg_seg_at(g)] = 0.0f;
                if (g == ngrp) { s_rem[0] = e[0]; s_rem[1] = e[1]; s_rem[2] = e[2]; }
            } else if (g >= ngrp && g < ((ngrp + 31) & ~31)) s_grp[xg_seg_at(g)] = 0.0f;
        }
        xp_arrive(s_cnt + 1);
        if (wave == 0) {
            xp_await(s_cnt + 1, 8);
            XSTAMP(dbg, 3);
            float sum = xg_segment_sum<1>(s_grp, min(ngrp, 1024));
            for (int g = 1024; g < ngrp; g += 4) {                   // zeros behind the last group leave the sum as it is
                const float4 t = *(const float4 *)(s_grp + xg_seg_at(g));
                sum = sum + t.x; sum = sum + t.y; sum = sum + t.z; sum = sum + t.w;
            }
            for (int j = ngrp * 4; j < n_kv; j++) sum = sum + s_rem[j & 3];
            if (lane == 0) s_sum = sum;
            xp_arrive(s_cnt + 2);
        }
        xp_await(s_cnt + 2, 1);
        XSTAMP(dbg, 4);
        const float inv = 1.0f / s_sum;
#pragma unroll
        for (int u = 0; u < XP_NG; u++) {
            const int g = tid + 512 * u;
            if (g < nall) {                                          // (of the last group also what lies behind the last token: not used)
                uint16_t p[4];
#pragma unroll
                for (int i = 0; i < 4; i++) p[i] = f2h(v[u][i] * inv);
                const uint2 pp = make_uint2(p[0] | ((uint32_t)p[1] << 16), p[2] | ((uint32_t)p[3] << 16));
                if (g < XP_LAY / 4) {
                    uint16_t *at = s_p + (((g >> 3) & 1) * 32 + ((g >> 1) & 3) + 16 * (g & 1)) * SA + (g >> 4);
#pragma unroll
                    for (int i = 0; i < 4; i++) at[4 * i * SA] = p[i];
                } else *(uint2 *)(s_p + 64 * SA + 4 * g - XP_LAY) = pp;
                if (g >= 8 * nfull) *(uint2 *)(s_p + 64 * SA + REST + 4 * (g - 8 * nfull)) = pp;
            }
        }
    } else {
        // ---- two rows of V^T from memory to their places; nothing beyond the last cached token is asked for ----
        // vc is not a restrict pointer on purpose: the loads must stay where they are written.
        const uint16_t *vrow = vc + (size_t)(hd_ * 128 + dgrp * 16 + 2 * (wave - 8)) * n_ctx;
        xp_u4 vb[2][XP_NP], vt[2];
        const int u = lane >> 3, par = (lane >> 2) & 1, o = lane & 3;
        const int walked = 4 * nfull;                                 // pieces of whole chunks; the last chunk, 1 .. 32 elements, goes apart
        const bool mine = 64 * u + 4 * par < walked;
#pragma unroll
        for (int r = 0; r < 2; r++) {
            vt[r] = *(const xp_u4 *)(vrow + (size_t)r * n_ctx + (size_t)min(4 * nfull + o, last_piece) * 8);
#pragma unroll
            for (int i = 8; i < XP_NP; i++) if (64 * i < walked) vb[r][i] = *(const xp_u4 *)(vrow + (size_t)r * n_ctx + (size_t)min(64 * i + lane, walked - 1) * 8);
        }
        if (mine) {
#pragma unroll
            for (int r = 0; r < 2; r++)
#pragma unroll
                for (int i = 0; i < 8; i++) vb[r][i] = *(const xp_u4 *)(vrow + (size_t)r * n_ctx + (size_t)min(64 * u + 8 * i + (lane & 7), walked - 1) * 8);
        }
        if (RS * 2 * (2 * (wave - 8) + 3) > xattn_pv_soft_at(n_ctx)) xp_await(s_cnt + 2, 1);       // the softmax works where these rows go
#pragma unroll
        for (int r = 0; r < 2; r++) {
            uint16_t *row = s_v + (size_t)(2 * (wave - 8) + r) * RS;
            if (mine) {
                uint16_t *dst = row + (par * 32 + o) * SA + 8 * u;
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    xp_u4 w;
#pragma unroll
                    for (int k = 0; k < 4; k++) w[k] = __builtin_amdgcn_perm(vb[r][2 * k + 1][e >> 1], vb[r][2 * k][e >> 1], e & 1 ? 0x07060302u : 0x05040100u);
                    *(xp_u4 *)(dst + 4 * e * SA) = w;
                }
            }
            if (512 + lane < walked) {
                const int c = 128 + (lane >> 2);
#pragma unroll
                for (int e = 0; e < 8; e++) row[((c & 1) * 32 + 4 * e + o) * SA + (c >> 1)] = (uint16_t)(vb[r][8][e >> 1] >> (16 * (e & 1)));
            }
            if (576 + lane < walked) *(xp_u4 *)(row + 64 * SA + lane * 8) = vb[r][9];
            if (lane < 4) *(xp_u4 *)(row + 64 * SA + REST + lane * 8) = vt[r];
        }
    }
    __syncthreads();
    XSTAMP(dbg, 5);
    // ---- P . V^T ----
    if (wave < 8) {
        const int r16 = wave * 2 + (lane >> 5), cl = lane & 31, acl = 8 * (cl & 3) + (cl >> 2);       // row of the 16, place and accumulator 8 j + l
        const uint16_t *vr = s_v + (size_t)r16 * RS;
        const uint16_t *v0 = vr + cl * SA, *v1 = v0 + 32 * SA, *p0 = s_p + cl * SA, *p1 = p0 + 32 * SA;
        float acc = 0.0f;
        const int ntail = n_kv - 32 * nfull;                          // 1 .. 32
        // operands of the scalar tail, requested ahead of the walk (the 32 lanes of a row read the same addresses)
        xp_u4 tv[4], tq[4];
#pragma unroll
        for (int u = 0; u < 4; u++) { tv[u] = *(const xp_u4 *)(vr + 64 * SA + REST + 8 * u); tq[u] = *(const xp_u4 *)(s_p + 64 * SA + REST + 8 * u); }
        struct chunks16 { xp_u4 v0, v1, p0, p1; };
        auto ld = [&](chunks16 &x, int g) { x.v0 = *(const xp_u4 *)(v0 + 8 * g); x.v1 = *(const xp_u4 *)(v1 + 8 * g); x.p0 = *(const xp_u4 *)(p0 + 8 * g); x.p1 = *(const xp_u4 *)(p1 + 8 * g); };
        auto run = [&](const chunks16 &x, int n) {
#pragma unroll
            for (int c = 0; c < 16; c++) {
                const xp_u4 &v = c & 1 ? x.v1 : x.v0, &p = c & 1 ? x.p1 : x.p0;
                const int k = c >> 1;
                const uint32_t vw = v[k >> 1], pw = p[k >> 1];
                if (c < n) acc = fmaf(h2f((uint16_t)(k & 1 ? vw >> 16 : vw & 0xFFFFu)), h2f((uint16_t)(k & 1 ? pw >> 16 : pw & 0xFFFFu)), acc);
            }
        };
        const int nlay = min(nfull, XP_LAY / 32), ng = nlay / 16, glast = SA / 8 - 1;
        chunks16 A, B;
        ld(A, 0);
        int g = 0;
        for (; g + 2 <= ng; g += 2) {
            ld(B, g + 1);
            __builtin_amdgcn_sched_barrier(0);
            run(A, 16);
            __builtin_amdgcn_sched_barrier(0);
            ld(A, min(g + 2, glast));
            __builtin_amdgcn_sched_barrier(0);
            run(B, 16);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (g < ng) { run(A, 16); g++; ld(A, min(g, glast)); }
        run(A, nlay - 16 * g);
        for (int c = nlay; c < nfull; c++) acc = fmaf(h2f(vr[64 * SA + 32 * c - XP_LAY + acl]), h2f(s_p[64 * SA + 32 * c - XP_LAY + acl]), acc);
        XSTAMP(dbg, 6);
        // block_reduce of the 32 accumulators (xa_tree32's sums) at these places: a ^ 16 and a ^ 8 are lanes ^ 2 and ^ 1, a ^ 4 lane ^ 16, a ^ 1 and a ^ 2 lanes ^ 4 and ^ 8,
        // which a mirror reaches where the four or eight lanes of a group agree
#define XP_ADD(CTRL) acc += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(acc), CTRL, 0xF, 0xF, true));
        XP_ADD(0x4E) XP_ADD(0xB1)
        const auto sw = __builtin_amdgcn_permlane16_swap(__float_as_uint(acc), __float_as_uint(acc), false, false);
        acc = __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
        XP_ADD(0x141) XP_ADD(0x140)
#undef XP_ADD
        float tail = 0.0f;
        XA_TAIL32(tail, tv, tq, ntail)                               // elements 32 nfull .. n_kv - 1
        if (cl == 0) attn_out[hd_ * 128 + dgrp * 16 + r16] = tail + acc;
        XSTAMP(dbg, 7);
    }
}
