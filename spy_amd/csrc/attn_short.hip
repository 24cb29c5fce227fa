// Attention of one token in the host backend's summation order where the cache is short: scores, softmax and P.V^T in one launch.
// (In a source of its own: the kernels of a layer of the single-token pass about fill the instruction cache, and where they lie in it counts.)
#include "exact_decode.cuh"
#include "engine_types.cuh"
#include "attn_reach.h"

// ---- scores, softmax and P.V^T of a short cache in one launch ------------------------------------------------------------
// Up to XF_MAX cached tokens: the same 256 workgroups (head, 16 rows of V^T), each with all the scores of its head.  The eight
// workgroups of a head read its keys eight times over, from the L2 of the one XCD that they share (head = workgroup index modulo n_head, n_head a
// multiple of 8 in the models there are), and what that costs is less than the launch and the scores' way through memory that it saves:
// one layer's after the other, the two launches 8.4 -> 4.7 or 5.4 us (by process) with 40 tokens, 9.9 -> 7.0 with 300, 10.6 -> 9.2 with 512, 11.0 -> 10.4 with 576; kernel times
// in a pass 10.3 -> 4.9 with 8 .. 40 tokens, 12.0 -> 10.5 with 512 .. 535.  Up to XF_MAX tokens the keys of a head fit LDS.  n_ctx is a multiple of 8 (16-byte pieces of a V^T row).
// What bounds it: the chain launch, keys and V^T rows (one wait for both), dots, exponentials (a gather), running sum, walk.
#define XF_NP (XF_MAX * 16 / XP_THREADS)   // 16-byte pieces of keys per thread
static size_t xattn_short_lds(int n_ctx) { return (size_t)(n_ctx < XF_MAX ? n_ctx : XF_MAX) * 256 + 16 * 96 * 2; }      // the keys; later the rows of V^T (16 rows of cap + 32 .. 96 halfs)
// IN_STATE: the position is st->pos, else pos_imm (decided when the kernel is compiled: asked in the kernel it cost the engine's launches 0.1 of 5 us)
template <bool IN_STATE>
static __global__ __launch_bounds__(XP_THREADS) void xattn_short_kernel(const dev_state *st, int pos_imm, const uint16_t *__restrict__ q16, const uint16_t *kc, const uint16_t *vc,
                                                                 float *__restrict__ scores, float *attn_out, const float *__restrict__ lut, int n_ctx, float scale) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    __shared__ __attribute__((aligned(16))) uint4 s_qh[16];
    __shared__ __attribute__((aligned(16))) float s_t[XF_MAX], s_e[XF_MAX + 32], s_grp[(XF_MAX / 4 + 63) / 64 * 64];
    __shared__ __attribute__((aligned(16))) uint16_t s_tail[8][32];
    __shared__ float s_sum;
    const int cap = n_ctx < XF_MAX ? n_ctx : XF_MAX;
    const int n_head = (int)gridDim.x >> 3, hd_ = (int)blockIdx.x % n_head, dgrp = (int)blockIdx.x / n_head, d = n_head * 128;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int VS = (cap + 63) / 64 * 64 + 32;                         // as xattn_pv_vstride
    uint4 *s_k = (uint4 *)smem;                                       // [token][16 pieces], rotated by 4 pieces per token against bank conflicts
    uint16_t *s_v = (uint16_t *)smem;                                 // the rows of V^T, once the keys have been read
    const uint16_t *vrow = vc + (size_t)(hd_ * 128 + dgrp * 16 + wave) * n_ctx;
    // Keys first, then the rows of V^T.  Where the position is on its way itself, the first piece of either does not wait for it: 64 keys and 512 elements
    // of a row, as far as the cache goes; what lies behind the last token is not used.  Where it is a number, nothing behind the last token is asked for (attn_reach.h).
    xp_u4 kr[XF_NP], vb, vb1, qr;
    auto key_piece = [&](int u, int n) {
        const int c = xf_piece(tid + u * XP_THREADS, n * 16);
        kr[u] = *(const xp_u4 *)(kc + (size_t)(c >> 4) * d + hd_ * 128 + (c & 15) * 8);
    };
    const int keys0 = xf_keys_before(IN_STATE, pos_imm, cap);
    key_piece(0, keys0);
    if (tid < 16) qr = *(const xp_u4 *)(q16 + hd_ * 128 + tid * 8);
    const int n_kv = IN_STATE ? min(st->pos + 1, cap) : keys0, npiece = n_kv * 16, last_piece = (n_kv - 1) >> 3;
    vb = *(const xp_u4 *)(vrow + (size_t)xf_piece(lane, xf_row_pieces_before(IN_STATE, pos_imm, n_ctx)) * 8);
    if (last_piece >= 64) vb1 = *(const xp_u4 *)(vrow + (size_t)xf_piece(64 + lane, last_piece + 1) * 8);
#pragma unroll
    for (int u = 1; u < XF_NP; u++) if (u * XP_THREADS < npiece) key_piece(u, n_kv);
    if (tid < 16) *(xp_u4 *)&s_qh[tid] = qr;
#pragma unroll
    for (int u = 0; u < XF_NP; u++) {
        const int c = tid + u * XP_THREADS, t = c >> 4;
        if (c < npiece) *(xp_u4 *)&s_k[t * 16 + (((c & 15) + 4 * t) & 15)] = kr[u];
    }
    __syncthreads();
    // four adjacent threads per key, thread `part` with accumulators 8 part .. 8 part + 7 (xattn_scores_kernel's form for few keys)
    for (int base = 0; base < n_kv * 4; base += XP_THREADS) {
        const int key = (base + tid) >> 2, part = tid & 3;
        if (key >= n_kv) break;
        const uint4 *kp = s_k + key * 16;
        const int rot = 4 * key;
        float sum[8];
#pragma unroll
        for (int l = 0; l < 8; l++) sum[l] = 0.0f;
#pragma unroll
        for (int i = 0; i < 3; i++) xa_fma8(sum, kp[(4 * i + part + rot) & 15], s_qh[4 * i + part]);
        xa_quad(sum);
        const float simd = xa_tree8(sum);
        float tail = 0.0f;
#pragma unroll
        for (int j = 0; j < 4; j++) tail = xa_tail8(tail, kp[(12 + j + rot) & 15], s_qh[12 + j]);
        if (part == 0) {
            s_t[key] = (tail + simd) * scale;
            if (dgrp == 0) scores[(size_t)hd_ * n_ctx + key] = s_t[key];      // as the launch of its own leaves them
        }
    }
    __syncthreads();
    // the keys are dead: the rows of V^T take their place; the maximum, by every wave for itself; the exponentials
    if (lane <= last_piece) *(xp_u4 *)(s_v + (size_t)wave * VS + lane * 8) = vb;
    if (64 + lane <= last_piece) *(xp_u4 *)(s_v + (size_t)wave * VS + 512 + lane * 8) = vb1;
    if (wave * 64 < n_kv) {
        float mx = -INFINITY;
        for (int j = lane; j < n_kv; j += 64) mx = fmaxf(mx, s_t[j]);
        mx = wave_max(mx);
        const float e = lut[f2h(s_t[min(tid, n_kv - 1)] - mx)];
        s_e[tid] = tid < n_kv ? e : 0.0f;
    }
    __syncthreads();
    if (wave == 0) {
        // std::reduce: groups of four added to one running sum (at most 144 of them: a plain chain; zeros behind the last one leave it as it is), then the last n % 4 elements
        const int ngrp = n_kv / 4;
#pragma unroll
        for (int u = 0; u < (XF_MAX / 4 + 63) / 64; u++) {
            const int g = lane + 64 * u;
            s_grp[g] = xa_group(g < ngrp ? *(const float4 *)(s_e + 4 * g) : make_float4(0.0f, 0.0f, 0.0f, 0.0f));
        }
        __builtin_amdgcn_wave_barrier();
        float sum = 0.0f;
        for (int g = 0; g < ngrp; g += 16) {
            float4 v[4];
#pragma unroll
            for (int u = 0; u < 4; u++) v[u] = *(const float4 *)(s_grp + g + 4 * u);
#pragma unroll
            for (int u = 0; u < 4; u++) { sum = sum + v[u].x; sum = sum + v[u].y; sum = sum + v[u].z; sum = sum + v[u].w; }
        }
        for (int j = ngrp * 4; j < n_kv; j++) sum = sum + s_e[j];
        if (lane == 0) s_sum = sum;
    }
    __syncthreads();
    if (wave >= 8) return;
    // P.V^T as in xattn_pv_kernel, the probabilities formed where they are used
    const float inv = 1.0f / s_sum;
    const int nfull = (n_kv - 1) / 32, ntail = n_kv - 32 * nfull, r16 = wave * 2 + (lane >> 5), cl = lane & 31;
    const uint16_t *vr = s_v + (size_t)r16 * VS;
    if (lane < 32) s_tail[wave][lane] = f2h(s_e[32 * nfull + lane] * inv);
    float acc = 0.0f;
    for (int i = 0; i < nfull; i++) acc = fmaf(h2f(vr[32 * i + cl]), h2f(f2h(s_e[32 * i + cl] * inv)), acc);
    acc = xa_tree32(acc);
    __builtin_amdgcn_wave_barrier();
    float tail = 0.0f;
    xp_u4 tv[4], tq[4];
#pragma unroll
    for (int u = 0; u < 4; u++) { tv[u] = *(const xp_u4 *)(vr + 32 * nfull + 8 * u); tq[u] = *(const xp_u4 *)&s_tail[wave][8 * u]; }
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
    const dim3 grid((unsigned)(n_head * 8)), block(XP_THREADS);
    if (state) xattn_short_kernel<true><<<grid, block, xattn_short_lds(n_ctx), st>>>(state, pos_imm, q16, kc, vc, scores, out, lut, n_ctx, scale);
    else xattn_short_kernel<false><<<grid, block, xattn_short_lds(n_ctx), st>>>(state, pos_imm, q16, kc, vc, scores, out, lut, n_ctx, scale);
    return SPY_LAUNCH_RC();
}
