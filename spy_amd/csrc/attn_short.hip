// Attention of one token in the host backend's summation order where the cache is short: scores, softmax and P.V^T in one launch.
// (In a source of its own: the kernels of a layer of the single-token pass about fill the instruction cache, and where they lie in it counts.)
#include "exact_decode.cuh"
#include "engine_types.cuh"
#include "attn_reach.h"

// ---- scores, softmax and P.V^T of a short cache in one launch ------------------------------------------------------------
// Up to XF_MAX cached tokens: the same 256 workgroups (head, 16 rows of V^T), each with all the scores of its head.  The eight
// workgroups of a head read its keys eight times over, from the L2 of the one XCD that they share (head = workgroup index modulo n_head, n_head a
// multiple of 8 in the models there are), and what that costs is less than the launch and the scores' way through memory that it saves.
// Keys go straight into registers, four adjacent lanes per key (xattn_scores_kernel's form).
// In a pass, us: 550 tokens 10.6 -> 8.9, 300 8.1 -> 6.8, 40 5.4 -> 5.1 against keys by way of LDS, gathers of the exponentials and a walk that read its operands step by step
// after the sum (two launches take 11.4 with 600 tokens).  n_ctx is a multiple of 8 (16-byte pieces of a V^T row).
// What bounds it: the chain launch, keys and V^T rows (one wait for both), dots, maximum, exponentials, running sum, walk.
#define XF_NU ((XF_MAX + 255) / 256)       // units of 16 keys per wave
static int xattn_short_vs(int n_ctx) { return ((n_ctx < XF_MAX ? n_ctx : XF_MAX) + 63) / 64 * 64 + 32; }      // halfs between rows of V^T in LDS
static size_t xattn_short_lds(int n_ctx) { return (size_t)16 * xattn_short_vs(n_ctx) * 2; }
// IN_STATE: the position is st->pos, else pos_imm (decided when the kernel is compiled: asked in the kernel it cost the engine's launches 0.1 of 5 us)
template <bool IN_STATE>
static __global__ __launch_bounds__(XP_THREADS) void xattn_short_kernel(const dev_state *st, const uint16_t *__restrict__ q16, const uint16_t *kc, const uint16_t *vc, const float *__restrict__ lut,
                                                                 int n_ctx, int pos_imm, float *attn_out, float *__restrict__ scores, float scale) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    __shared__ __attribute__((aligned(16))) float s_t[XF_MAX], s_e[XF_MAX + 64], s_grp[(XF_MAX / 4 + 63) / 64 * 64];
    __shared__ __attribute__((aligned(16))) uint32_t s_code[XE_WORDS];
    __shared__ __attribute__((aligned(16))) uint16_t s_tail[8][32];
    __shared__ float s_sum;
    const int cap = n_ctx < XF_MAX ? n_ctx : XF_MAX, VS = (cap + 63) / 64 * 64 + 32;
    const int n_head = (int)gridDim.x, hd_ = (int)blockIdx.x, dgrp = (int)blockIdx.y, d = n_head * 128;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, part = lane & 3;
    uint16_t *s_v = (uint16_t *)smem;
    const uint16_t *vrow = vc + (size_t)(hd_ * 128 + dgrp * 16 + wave) * n_ctx;
    // Keys first, then the rows of V^T.  Where the position is on its way itself, the first piece of either does not wait for it: 64 keys and 512 elements
    // of a row, as far as the cache goes; what lies behind the last token is not used.  Where it is a number, nothing behind the last token is asked for (attn_reach.h).
    uint4 q[4], k[XF_NU][4];
    xp_u4 vb, vb1, cd;
    auto key_piece = [&](int u, int n) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int c = xf_piece((16 * (wave + 16 * u) + (lane >> 2)) * 16 + 4 * i + part, n * 16);
            k[u][i] = *(const uint4 *)(kc + (size_t)(c >> 4) * d + hd_ * 128 + (c & 15) * 8);
        }
    };
    const int keys0 = xf_keys_before(IN_STATE, pos_imm, cap);
#pragma unroll
    for (int i = 0; i < 4; i++) q[i] = *(const uint4 *)(q16 + hd_ * 128 + 32 * i + 8 * part);
    if (wave < 4) key_piece(0, keys0);
    if (tid < XE_WORDS / 4) cd = ((const xp_u4 *)(lut + XE_AT))[tid];
    const int n_kv = IN_STATE ? min(st->pos + 1, cap) : keys0, last_piece = (n_kv - 1) >> 3;
#pragma unroll
    for (int u = 0; u < XF_NU; u++) if ((u > 0 || wave >= 4) && 16 * (wave + 16 * u) < n_kv) key_piece(u, n_kv);
    vb = *(const xp_u4 *)(vrow + (size_t)xf_piece(lane, xf_row_pieces_before(IN_STATE, pos_imm, n_ctx)) * 8);
    if (last_piece >= 64) vb1 = *(const xp_u4 *)(vrow + (size_t)xf_piece(64 + lane, last_piece + 1) * 8);
#pragma unroll
    for (int u = 0; u < XF_NU; u++) {
        const int t = 16 * (wave + 16 * u) + (lane >> 2);
        if (16 * (wave + 16 * u) < n_kv) {
            const float x = xa_dot4(k[u], q) * scale;
            if (part == 3 && t < n_kv) {
                s_t[t] = x;
                if (dgrp == 0) scores[(size_t)hd_ * n_ctx + t] = x;             // as the launch of its own leaves them
            }
        }
    }
    if (tid < XE_WORDS / 4) ((xp_u4 *)s_code)[tid] = cd;
    if (lane <= last_piece) *(xp_u4 *)(s_v + (size_t)wave * VS + lane * 8) = vb;
    if (64 + lane <= last_piece) *(xp_u4 *)(s_v + (size_t)wave * VS + 512 + lane * 8) = vb1;
    __syncthreads();
    // the maximum, by every wave for itself; the exponentials
    if (wave * 64 < n_kv) {
        float mx = -INFINITY;
        for (int j = lane; j < n_kv; j += 64) mx = fmaxf(mx, s_t[j]);
        mx = wave_max(mx);
        const float t = s_t[min(tid, n_kv - 1)];
        bool ask;
        float e = xe_exp(f2h(mx - t), s_code, ask);
        if (__any(ask)) e = lut[f2h(t - mx)];
        s_e[tid] = tid < n_kv ? e : 0.0f;
    }
    __syncthreads();
    const int nfull = (n_kv - 1) / 32, ntail = n_kv - 32 * nfull, r16 = (wave & 7) * 2 + (lane >> 5), cl = lane & 31;
    const uint16_t *vr = s_v + (size_t)r16 * VS;
    constexpr int NS = (XF_MAX - 1) / 32;                             // steps of the walk
    uint16_t v[NS];
    float e[NS], et = 0.0f;
    xp_u4 tv[4];
    if (wave >= 8) {
        // the operands of the walk, while wave 0 walks the sum
#pragma unroll
        for (int i = 0; i < NS; i++) { const int at = 32 * min(i, nfull) + cl; v[i] = vr[at]; e[i] = s_e[at]; }
        et = s_e[32 * nfull + cl];
#pragma unroll
        for (int u = 0; u < 4; u++) tv[u] = *(const xp_u4 *)(vr + 32 * nfull + 8 * u);
    } else if (wave == 0) {
        // std::reduce: groups of four added to one running sum (at most 144 of them: a plain chain, the next sixteen read ahead; zeros behind the last one leave it as it is),
        // then the last n % 4 elements
        const int ngrp = n_kv / 4;
#pragma unroll
        for (int u = 0; u < (XF_MAX / 4 + 63) / 64; u++) {
            const int g = lane + 64 * u;
            s_grp[g] = xa_group(g < ngrp ? *(const float4 *)(s_e + 4 * g) : make_float4(0.0f, 0.0f, 0.0f, 0.0f));
        }
        __builtin_amdgcn_wave_barrier();
        float sum = 0.0f;
        float4 a[4], b[4];
        auto ld = [&](float4 (&x)[4], int g) {
#pragma unroll
            for (int u = 0; u < 4; u++) x[u] = *(const float4 *)(s_grp + g + 4 * u);
        };
        auto run = [&](const float4 (&x)[4]) {
#pragma unroll
            for (int u = 0; u < 4; u++) { sum = sum + x[u].x; sum = sum + x[u].y; sum = sum + x[u].z; sum = sum + x[u].w; }
        };
        ld(a, 0);
        for (int g = 0; g < ngrp; g += 32) {
            ld(b, g + 16);
            run(a);
            ld(a, g + 32);
            run(b);
        }
        for (int j = ngrp * 4; j < n_kv; j++) sum = sum + s_e[j];
        if (lane == 0) s_sum = sum;
    }
    __syncthreads();
    if (wave < 8) return;
    // P.V^T in the order of xattn_pv_kernel, the probabilities formed where they are used
    const float inv = 1.0f / s_sum;
    if (lane < 32) s_tail[wave - 8][lane] = f2h(et * inv);
    float acc = 0.0f;
#pragma unroll
    for (int i = 0; i < NS; i++) if (i < nfull) acc = fmaf(h2f(v[i]), h2f(f2h(e[i] * inv)), acc);
    acc = xa_tree32(acc);
    __builtin_amdgcn_wave_barrier();
    float tail = 0.0f;
    xp_u4 tq[4];
#pragma unroll
    for (int u = 0; u < 4; u++) tq[u] = *(const xp_u4 *)&s_tail[wave - 8][8 * u];
    XA_TAIL32(tail, tv, tq, ntail)
    if (cl == 0) attn_out[hd_ * 128 + dgrp * 16 + r16] = tail + acc;
}

int spy_attn_short_prepare(int n_ctx) {
    const int rc = spy_raise_lds_limit((const void *)xattn_short_kernel<true>, xattn_short_lds(n_ctx));
    return rc ? rc : spy_raise_lds_limit((const void *)xattn_short_kernel<false>, xattn_short_lds(n_ctx));
}
// scores: [n_head][n_ctx], as the launch of xattn_scores_kernel leaves them
int spy_attn_short(hipStream_t st, const dev_state *state, int pos_imm, const uint16_t *q16, const uint16_t *kc, const uint16_t *vc, float *scores, float *out,
                   const float *lut, int n_head, int n_ctx, float scale) {
    const dim3 grid((unsigned)n_head, 8), block(XP_THREADS);
    if (state) xattn_short_kernel<true><<<grid, block, xattn_short_lds(n_ctx), st>>>(state, q16, kc, vc, lut, n_ctx, pos_imm, out, scores, scale);
    else xattn_short_kernel<false><<<grid, block, xattn_short_lds(n_ctx), st>>>(state, q16, kc, vc, lut, n_ctx, pos_imm, out, scores, scale);
    return SPY_LAUNCH_RC();
}
