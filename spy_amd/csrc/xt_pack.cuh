#pragma once

#include "common.cuh"

// Layout of packed activations (exact_gemm.hip), per group of 16 rows and stage of four Q8_0 blocks: XT_XB bytes of quants
//   [block][word pair g][row][word of the pair][4 x fp16: elements 0, 2, 1, 3 of the word]
// and one record of XT_XD bytes: scales [block][row], fp16 in the lower half of a dword, then the sums of the quants [block][row], fp32
#define XT_XB 4096
#define XT_XD 512

// Quantizator<FP32,Q8_0>::transform (vec_convert.h:178-261), as quantize_q8_0_kernel, the quants as fp16: elements 4 e .. 4 e + 3 (in lane e of eight adjacent ones) of
// block b of row c of group cg
__device__ __forceinline__ void xt_store4(const float4 v, int cg, int nst, int b, int c, int e, uint8_t *xq, uint8_t *xd) {
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
    int sum = (qv[0] + qv[1]) + (qv[2] + qv[3]);
    sum += __shfl_xor(sum, 1, SPY_WAVE);
    sum += __shfl_xor(sum, 2, SPY_WAVE);
    sum += __shfl_xor(sum, 4, SPY_WAVE);
    if (e == 0) {
        uint32_t *rec = (uint32_t *)(xd + ((int64_t)cg * nst + (b >> 2)) * XT_XD + (b & 3) * 64 + c * 4);
        rec[0] = f2h(d);
        rec[64] = __float_as_uint((float)sum);
    }
}
