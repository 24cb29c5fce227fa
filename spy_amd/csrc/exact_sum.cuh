#pragma once

#include "common.cuh"

// libstdc++'s running sum (one value after the other added to ONE sum) of up to 1024 M NON-NEGATIVE terms by one wave, mostly in parallel and
// still bit for bit.
// While the running sum s stays inside one binade [2^e, 2^(e+1)) it is an integer multiple S of ulp = 2^(e-23), and adding a term
// g >= 0 with round-to-nearest-even is integer arithmetic: with f = g / ulp,
//     RNE(S + f) = S + floor(f) + r,   r = 1 if frac(f) > 1/2, 0 if < 1/2, and for frac(f) = 1/2 the parity of S + floor(f).
// So a run of terms is a map from the parity of the incoming S to an increment, (inc_even, inc_odd), and maps compose associatively
// (C[p] = A[p] + B[(p + A[p]) & 1]).  The sum is non-decreasing: if its first and last value lie in binade e, every value between does.
// Lane c has the 16 M terms from 16 M c on.
// Padded layout of the terms: 16 floats every 20 (80 bytes: the lanes' 128-bit reads spread over the banks); zeros up to the next multiple of 16 M.
static __device__ __forceinline__ int xg_seg_at(int i) { return i + (i >> 4) * 4; }
// Every lane adds its terms to two candidate values of the running sum, neighbours (even and odd) near an approximate prefix sum: by the rule above
// the differences are the increments for ANY incoming sum of that binade, as long as it stays there.  Runs of segments in one binade are composed by a
// segmented scan, and the walk takes a run in one addition; what remains are the segments in which the sum crosses a power of two (about one per
// doubling), added term by term.  Where the prefix sum named the wrong binade (the exact sum has another exponent before or after the run), the
// run is added term by term as well: nothing that is kept is approximate.  1024 terms: 2 us (chain of single additions: 4.4).
template <int M>
static __device__ __forceinline__ float xg_segment_sum(const float *s_g, int n) {
    if (n <= 0) return 0.0f;
    const int lane = threadIdx.x & 63, nseg = (n + 16 * M - 1) / (16 * M);
    float4 v[4 * M];
    auto term4 = [&](int c, int u) { return *(const float4 *)(s_g + c * (20 * M) + (u >> 2) * 20 + 4 * (u & 3)); };
#pragma unroll
    for (int u = 0; u < 4 * M; u++) v[u] = term4(min(lane, nseg - 1), u);
    float cs = 0.0f;
#pragma unroll
    for (int u = 0; u < 4 * M; u++) cs += (v[u].x + v[u].y) + (v[u].z + v[u].w);
    float incl = cs;                                     // inclusive prefix over the lanes (an approximation: its rounding does not matter)
#define XG_DPP_F(x, CTRL, ROWS) __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, ROWS, 0xF, true))
    incl += XG_DPP_F(incl, 0x111, 0xF); incl += XG_DPP_F(incl, 0x112, 0xF); incl += XG_DPP_F(incl, 0x114, 0xF); incl += XG_DPP_F(incl, 0x118, 0xF);
    incl += XG_DPP_F(incl, 0x142, 0xA); incl += XG_DPP_F(incl, 0x143, 0xC);
#undef XG_DPP_F
    // (bound_ctrl: lanes outside the row mask and before the row's start get 0)
    const int before = __float_as_int(__int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(incl), 0x138, 0xF, 0xF, true)));       // wave_shr:1
    const int be = before & ~1, bo = before | 1, eb = be >> 23;
    float se = __int_as_float(be), so = __int_as_float(bo);
#pragma unroll
    for (int u = 0; u < 4 * M; u++) {
        se += v[u].x; so += v[u].x; se += v[u].y; so += v[u].y; se += v[u].z; so += v[u].z; se += v[u].w; so += v[u].w;
    }
    const int ee = __float_as_int(se), eo = __float_as_int(so);
    const bool ok = eb >= 1 && eb < 254 && (ee >> 23) == eb && (eo >> 23) == eb;
    int t0 = ee - be, t1 = eo - bo;
    const int pe = __builtin_amdgcn_update_dpp(-1, ok ? eb : -1, 0x138, 0xF, 0xF, false);      // binade of the segment before, -1: none
    const bool head = !ok || pe != eb;
    int f = head ? 1 : 0;
#define XG_STEP(CTRL, ROWS) { const int p0 = __builtin_amdgcn_update_dpp(0, t0, CTRL, ROWS, 0xF, false), p1 = __builtin_amdgcn_update_dpp(0, t1, CTRL, ROWS, 0xF, false), \
                                        pf = __builtin_amdgcn_update_dpp(1, f, CTRL, ROWS, 0xF, false), has = __builtin_amdgcn_update_dpp(0, 1, CTRL, ROWS, 0xF, false); \
                              const int c0 = p0 + ((p0 & 1) ? t1 : t0), c1 = p1 + ((p1 & 1) ? t0 : t1); \
                              if (has && !f) { t0 = c0; t1 = c1; f = pf; } }
    XG_STEP(0x111, 0xF) XG_STEP(0x112, 0xF) XG_STEP(0x114, 0xF) XG_STEP(0x118, 0xF) XG_STEP(0x142, 0xA) XG_STEP(0x143, 0xC)
#undef XG_STEP
    const unsigned long long in = nseg >= 64 ? ~0ull : (1ull << nseg) - 1, heads = __ballot(head) & in, slow = __ballot(!ok) & in;
    auto next = [&](unsigned long long m, int from) -> int { const unsigned long long x = from < 64 ? m >> from << from : 0ull; return x ? __builtin_ctzll(x) : nseg; };
    float4 w[4 * M];
    auto request = [&](int c) {
#pragma unroll
        for (int u = 0; u < 4 * M; u++) w[u] = term4(c, u);
    };
    int have = next(slow, 0);                            // the next segment to be added term by term is requested ahead
    if (have < nseg) request(have);
    int bits = 0, c = 0;
    while (c < nseg) {
        int to = c + 1;
        if (!((slow >> c) & 1)) {
            const int x = next(heads, c + 1), e = __builtin_amdgcn_readlane(eb, c);
            const int nb = bits + ((bits & 1) ? __builtin_amdgcn_readlane(t1, x - 1) : __builtin_amdgcn_readlane(t0, x - 1));
            if ((bits >> 23) == e && (nb >> 23) == e) { bits = nb; c = x; continue; }
            to = x;                                      // the prefix sum named the wrong binade: the whole run term by term
        }
        float s = __int_as_float(bits);
        for (; c < to; c++) {
            if (c != have) request(c);
#pragma unroll
            for (int u = 0; u < 4 * M; u++) { s = s + w[u].x; s = s + w[u].y; s = s + w[u].z; s = s + w[u].w; }
            have = next(slow, c + 1);
            if (have < nseg) request(have);
        }
        bits = __builtin_amdgcn_readfirstlane(__float_as_int(s));
    }
    return __int_as_float(bits);
}
