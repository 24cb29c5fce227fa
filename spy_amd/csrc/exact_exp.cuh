#pragma once

#include "common.cuh"

// The host's expf of an argument that is a value of fp16 and not above 0 (a score minus its row maximum, rounded as Softmax rounds it), bit for bit.  The table of
// 65 536 results that the host's libm fills lies in device memory (exact_order.hip), and a gather of 64 of its entries takes about 64 cycles of the compute unit.
// Instead the value is worked out and put right by a code of two bits per argument: the distance in ulps from the table's entry, from a list of 5.5 KB that
// fits LDS beside anything.  e^x = 2^n 2^(f + x LL) as in prompt_attn.hip: with log2 e = LH + LL and 13 bits in LH the products x LH and its distance f from the
// nearest integer n are exact, so that what v_exp_f32 gets has one rounding; with glibc's expf 20 832 of the 22 145 arguments down to -104 need no change, 242 one
// ulp less, 1071 one more.  An argument where that is not enough (none there; another libm's) has code 3 and asks the table, as a NaN does.
// The list is made from the table by the device itself (xe_code_kernel), with the same function.
#define XE_MAX 0x5680                                    // fp16 104.0: exp(-104) and everything below is 0
#define XE_WORDS 1388                                    // dwords of the list: 16 arguments each, a whole number of 16-byte pieces
#define XE_AT (2 * 65536)                                // where it lies behind the tables, in dwords
static_assert(XE_WORDS * 16 > XE_MAX && XE_WORDS % 4 == 0, "");

// hx: bits of -x
static __device__ __forceinline__ float xe_near(uint32_t hx) {
    const float x = h2f((uint16_t)hx), LH = -5909.0f / 4096.0f, LL = -6.80877639634e-05f;
    const float ph = x * LH, n = rintf(ph), g = fmaf(x, LL, ph - n);
    return ldexpf(__builtin_amdgcn_exp2f(g), (int)n);
}
// e^-hx; `ask` where only the table can tell.  codes: the list (LDS)
static __device__ __forceinline__ float xe_exp(uint32_t hx, const uint32_t *codes, bool &ask) {
    const uint32_t hc = min(hx, (uint32_t)XE_MAX), code = (codes[hc >> 4] >> (2 * (hc & 15))) & 3;
    ask = code == 3 || hx > 0x7C00u;
    return __uint_as_float(__float_as_uint(xe_near(hc)) + code - 1);
}
