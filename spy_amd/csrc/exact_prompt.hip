// Attention of a prompt pass in the host backend's summation order: the three operators
//   KQ = MatMul(K cache, Q)   Dot<FP16,FP16> over the 128 elements of a head   (vec_dot.h:117-146)
//   P  = Softmax(KQ, mask)    table exp, sum in groups of four                  (non-linear.cpp:86-180)
//   O  = MatMul(V^T cache, P) Dot<FP16,FP16> over the cached positions
// as three kernels that leave out what the causal mask removes and keep every float operation that is left in
// the host's order, so the outputs equal those of the operator-by-operator exact path (exact_order.hip) bit for bit:
//   * a masked score is never read, a masked probability is +0: an fma with a +0 factor leaves a finite accumulator
//     unchanged, and (a + 0) in the softmax sum is a;
//   * what still depends on the length n of the whole row is passed in (n_total, the cached positions after the whole
//     call): the host's fp16 dot runs its 32 accumulators over whole chunks of 32 elements while i + 32 < n and adds
//     the last 1..32 elements one by one, and the softmax sum adds the last n % 4 terms one by one.  A call may therefore
//     be cut into chunks of query rows without moving a rounding.
// An infinite or NaN V element is added in by every row that sees its token.  The host also multiplies it with the masked zeros of the rows before it in the same
// pass, which makes their sums NaN; here they keep their finite sums, but for those that share its tile of 32 rows.
// Values that cannot occur are not looked after: the fp16 caches are written by this library's float -> half
// conversion, which never produces the pattern 0xFFFF that the host's conversion table maps to 0 (conversion.h:39-41).
#include "common.cuh"
#include "exact_exp.cuh"
#include "exact_sum.cuh"
#include "xt_pack.cuh"

#include <type_traits>

namespace {

// ---------------------------------------------------------------- fma on the matrix cores
// v_mfma_f32_16x16x1_4b_f32 is D_b[i][j] = fma(A_b[i], B_b[j], C_b[i][j]) for four blocks b of 16 x 16 outputs, one rounding, subnormals kept: the bits of
// fmaf on 24-step chains of every kind of operand.  Where a term of the host's order is an outer product -- accumulator a of all (row, column)
// pairs of a tile takes the product of their elements 32 c + a -- the four blocks are four of the 32 accumulators, and the chains of fmas run at twice
// the rate of the vector units (74 against 39 Tfma/s measured).
// Lane (g, j) = (lane / 16, lane % 16) supplies A_g[j] and B_g[j] and holds D_b[4 g + v][j] in register 4 b + v.
typedef uint32_t xp_v4u __attribute__((ext_vector_type(4)));
typedef float xp_v4f __attribute__((ext_vector_type(4)));
typedef float xp_v16f __attribute__((ext_vector_type(16)));
__device__ __forceinline__ xp_v16f xp_mfma(float a, float b, xp_v16f c) { return __builtin_amdgcn_mfma_f32_16x16x1f32(a, b, c, 0, 0, 0); }
__device__ __forceinline__ xp_v16f xp_zero() {
    const xp_v16f c = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    return c;
}
__device__ __forceinline__ void xp_widen(const uint4 w, float (&f)[8]) {
    const uint32_t u[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
    for (int i = 0; i < 4; i++) {
        f[2 * i] = h2f((uint16_t)(u[i] & 0xFFFFu));
        f[2 * i + 1] = h2f((uint16_t)(u[i] >> 16));
    }
}
// FP16::block_reduce (vec_util.h:61-71) of accumulators 8 b + l, block b in registers 4 b .. 4 b + 3: its first two steps for one l
__device__ __forceinline__ void xp_reduce8(const xp_v16f &s, float (&t)[4]) {
#pragma unroll
    for (int v = 0; v < 4; v++) t[v] = (s[v] + s[8 + v]) + (s[4 + v] + s[12 + v]);
}

// ---------------------------------------------------------------- scores
// One workgroup per (head, 64 query rows), a wave takes 16 of them: their q values as floats in registers, laid out as right operands.  A tile of
// 64 key rows is brought into LDS by the whole workgroup.  Per 16 key rows and l = 0 .. 7 one chain of three matrix instructions (chunks of 32
// elements while i + 32 < 128) gives accumulators l, 8 + l, 16 + l, 24 + l of the 16 x 16 scores; the vector units add them in the host's tree.  The
// last 32 elements, added one by one, are a chain of eight v_mfma_f32_16x16x4_f32, which do the fmas of their four elements one after the other, bit for bit: a lane's
// eight elements of q stay in registers.  (As 32 of the former, whose four blocks were the four groups of 16 keys, they were widened for every tile; 125 registers then, 113 now, four workgroups on a
// compute unit either way.  Both in one run, 32 heads: 2048 rows on 2048 positions 670 -> 632 us, 2048 rows 231 -> 220, 77 rows on 1000 positions 20.7 -> 19.4.)  What bounds
// it: matrix and vector instructions of this kind never run at once (counter SQ_VALU_MFMA_COEXEC_CYCLES: 0), so the 31 additions of the tree and the
// widening of the keys come on top of the fmas (348 us).  A last tile of few rows with its keys dealt out over the waves: nothing (77 rows on 1000 16.4 us).
#define XP_KSEG 512
template <bool F16Q>       // q: f32 [T][H * 128] as Rope leaves it, or already rounded to fp16 and laid out [H][T][128]
__global__ __launch_bounds__(256, 4) void xp_scores_kernel(const void *__restrict__ q, const uint16_t *__restrict__ kc, float *__restrict__ S,
                                                           int T, int H, int P, int64_t s_row, int kseg) {
    constexpr int QT = 64;
    __shared__ __align__(16) uint4 s_k[2][64][17];               // 64 key rows of 256 bytes, 16 bytes apart
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = lane >> 4, j = lane & 15;
    // The head is the fastest-running index of the grid: consecutive workgroups go to the eight XCDs in turn, and with the query tile
    // there an XCD would get tiles k and k + 8 of 16 only -- under the causal mask 24 to 10 units of work (68 % of the compute units
    // busy over the launch).  With the head there every XCD gets the same mix of tiles, and the key rows of its heads stay in its L2.
    const int t0 = ((int)gridDim.y - 1 - (int)blockIdx.y) * QT, h = blockIdx.x;      // the longest rows first
    const int64_t d = (int64_t)H * 128;
    // the cached positions are dealt out in segments of kseg (a multiple of 64) over blockIdx.z, so that the workgroups are of similar length
    // (one workgroup per query tile would make the longest rows the critical path of the launch)
    const int kv_end = min(P + min(t0 + QT - 1, T - 1) + 1, ((int)blockIdx.z + 1) * kseg);       // cached positions that some row of the tile may see, within this segment
    if ((int)blockIdx.z * kseg >= kv_end) return;
    const int tw = t0 + wave * 16, wave_end = tw < T ? P + min(tw + 15, T - 1) + 1 : 0;      // the wave's query rows, and the positions that some of them may see
    float qm[3][8], qt[8];                                       // elements 32 c + 8 g + l and 96 + 4 l + g of query row j
    const int t = min(tw + j, T - 1);
    if constexpr (F16Q) {
        const uint4 *qp = (const uint4 *)((const uint16_t *)q + ((int64_t)h * T + t) * 128);
#pragma unroll
        for (int c = 0; c < 3; c++) xp_widen(qp[4 * c + g], qm[c]);
#pragma unroll
        for (int l = 0; l < 8; l++) qt[l] = h2f(((const uint16_t *)qp)[96 + 4 * l + g]);
    } else {
        const float *qp = (const float *)q + (int64_t)t * d + (int64_t)h * 128;
        auto halves = [&](int at) -> uint4 {
            const float4 x = *(const float4 *)(qp + at), y = *(const float4 *)(qp + at + 4);
            auto pair = [](float a, float b) -> uint32_t { return (uint32_t)f2h(a) | ((uint32_t)f2h(b) << 16); };
            return make_uint4(pair(x.x, x.y), pair(x.z, x.w), pair(y.x, y.y), pair(y.z, y.w));
        };
#pragma unroll
        for (int c = 0; c < 3; c++) xp_widen(halves(32 * c + 8 * g), qm[c]);
#pragma unroll
        for (int l = 0; l < 8; l++) qt[l] = h2f(f2h(qp[96 + 4 * l + g]));
    }
    // staging: thread -> key row tid / 4 of the tile, 64 of its 256 bytes
    const int st_row = threadIdx.x >> 2, st_q = (threadIdx.x & 3) * 4;
    xp_v4u kst[4];
    auto fetch = [&](int kv_first) {
        const xp_v4u *src = (const xp_v4u *)(kc + (int64_t)min(kv_first + st_row, kv_end - 1) * d + (int64_t)h * 128) + st_q;
#pragma unroll
        for (int i = 0; i < 4; i++) kst[i] = src[i];
    };
    fetch((int)blockIdx.z * kseg);
    int buf = 0;
    for (int kv0 = (int)blockIdx.z * kseg; kv0 < kv_end; kv0 += 64, buf ^= 1) {
        // (two buffers: a wave that writes this one is past the barrier of the tile before, which every wave reaches after its reads of this one)
#pragma unroll
        for (int i = 0; i < 4; i++) *(xp_v4u *)&s_k[buf][st_row][st_q + i] = kst[i];
        __syncthreads();
        if (kv0 + 64 < kv_end) fetch(kv0 + 64);
        if (kv0 >= wave_end) continue;                            // the tile lies behind the mask of the wave's query rows
#pragma unroll 1
        for (int kt = 0; kt < 4; kt++) {
            if (kv0 + 16 * kt >= wave_end) break;
            xp_v4f tail = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int l = 0; l < 8; l++) tail = __builtin_amdgcn_mfma_f32_16x16x4f32(h2f(((const uint16_t *)s_k[buf][16 * kt + j])[96 + 4 * l + g]), qt[l], tail, 0, 0, 0);
            float a[3][8];
#pragma unroll
            for (int c = 0; c < 3; c++) xp_widen(s_k[buf][16 * kt + j][4 * c + g], a[c]);
            auto part = [&](int l, float (&r)[4]) {
                xp_v16f s = xp_mfma(a[0][l], qm[0][l], xp_zero());
                s = xp_mfma(a[1][l], qm[1][l], s);
                s = xp_mfma(a[2][l], qm[2][l], s);
                xp_reduce8(s, r);
            };
            float u[4][4], o[4];
#pragma unroll
            for (int l = 0; l < 4; l++) {
                float x[4], y[4];
                part(l, x);
                __builtin_amdgcn_sched_barrier(0);
                part(l + 4, y);
#pragma unroll
                for (int v = 0; v < 4; v++) {                    // added here and now: eight chains waiting for their tree are 210 registers, this is 130
                    u[l][v] = x[v] + y[v];
                    asm volatile("" : "+v"(u[l][v]));
                }
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const float x = u[0][v] + u[1][v], y = u[2][v] + u[3][v];
                o[v] = tail[v] + (x + y);
            }
            if (tw + j < T) *(float4 *)(S + ((int64_t)h * T + t) * s_row + kv0 + 16 * kt + 4 * g) = make_float4(o[0], o[1], o[2], o[3]);
        }
    }
}

// ---------------------------------------------------------------- softmax
// One wave per (head, query row), NW waves per resident workgroup, rows dealt out in turn (the longest first); L = the positions the row may see.  A
// lane keeps its share of the row in registers (groups of four consecutive elements, the unit of the host's sum), so the row is read once
// and written once.  The probabilities leave as fp16 (the first step of the KQV MatMul, mat.cpp:37), followed by zeros up to the end of the
// 32-row tile's last chunk, which the product kernel reads.
// The exponentials: a gather of 64 table entries from memory takes about 64 cycles of the compute unit, so for many rows the part of the table that is not zero lies in
// LDS: arguments are <= 0 (or NaN), and exp is 0 from -104 on.  The sum of a row goes through xg_segment_sum: 2 us instead of a chain of up to
// 1024 additions.  2048 rows of 2049 .. 4096 positions and 32 heads (1.2 GB): 462 -> 306 us; 2048 rows of 1 .. 2048: 193 -> 152.
// A row of a wave is a chain of latencies, so waves are what counts: with half the registers and group sums for rows of up to 2048 positions a workgroup has 16
// instead of 12 (2048 rows of 1 .. 2048 positions 155 -> 123 us, 1000 rows 66 -> 50, 512 rows 29 -> 21).  The next row's scores requested a row ahead: 160 instead of 123.
// LIST: few rows, where bringing 88 KB of table to every compute unit is most of the time: the exponentials are worked out (exact_exp.cuh), which is 5.5 KB and about twice the vector
// instructions (32 heads, table -> list: 8 rows 7.2 -> 5.0 us, 33 6.9 -> 5.0, 200 on 100 positions 11.9 -> 9.7, 512 22.6 -> 20.5, 1000 45.3 -> 46.1, 2048 118 -> 123; rows of up to 4096 positions:
// 2048 301 -> 303).
// (Five and three waves per SIMD of four-wave workgroups leave the list's form 2 and 5 registers short, 12 and 24 bytes of scratch a lane; the table's form of rows of up to 4096
// positions is as short.)
#define XP_LUT XE_MAX
#define XP_LIST_ROWS 24576
#define XP_SM_R 32         // groups per lane: rows of up to 8192 positions
template <int R, int NW, int OCC, bool LIST>
__global__ __launch_bounds__(64 * NW, OCC) void xp_softmax_kernel(const float *__restrict__ S, uint16_t *__restrict__ P16, const float *__restrict__ lut, int T, int H, int P,
                                                             int64_t s_row, int n_total, float scale) {
    constexpr int TAB = LIST ? XE_WORDS : XP_LUT + 4;
    extern __shared__ __align__(16) float s_mem[];               // table or list, then per wave 64 R padded group sums and 4 floats
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    float *s_grp = s_mem + TAB + wave * (80 * R + 4), *s_rem = s_grp + 80 * R;
    for (int i = threadIdx.x; i < TAB / 4; i += 64 * NW) ((float4 *)s_mem)[i] = ((const float4 *)(lut + (LIST ? XE_AT : 0x8000)))[i];
    __syncthreads();
    const int rows = T * H;
    for (int id = (int)blockIdx.x * NW + wave; id < rows; id += (int)gridDim.x * NW) {
        const int t = T - 1 - id / H, h = id % H;
        const float4 *s4 = (const float4 *)(S + ((int64_t)h * T + t) * s_row);
        const int L = P + t + 1, ng_row = (L + 3) / 4;           // groups that hold an element of the row
        float4 v[R];
        float mx = -INFINITY;
        // blocks of 64 groups: whole ones, and the one in which the row ends (elements past L: -inf, which leaves 0)
#pragma unroll
        for (int r = 0; r < R; r++) if (64 * r < ng_row) v[r] = s4[min(lane + 64 * r, ng_row - 1)];
#pragma unroll
        for (int r = 0; r < R; r++)
            if (64 * r < ng_row) {
                float e[4] = {v[r].x * scale, v[r].y * scale, v[r].z * scale, v[r].w * scale};      // (+ the mask value 0 of an allowed position: nothing but the sign of a zero)
                if (256 * (r + 1) > L) {
#pragma unroll
                    for (int k = 0; k < 4; k++) e[k] = 4 * (lane + 64 * r) + k < L ? e[k] : -INFINITY;
                }
                mx = fmaxf(fmaxf(fmaxf(mx, e[0]), fmaxf(e[1], e[2])), e[3]);
                v[r] = make_float4(e[0], e[1], e[2], e[3]);
            }
        mx = wave_max(mx);
        // std::reduce in libstdc++: groups of four as init + ((a0 + a1) + (a2 + a3)) over the first n_total / 4 * 4 elements, the rest one
        // by one; groups and elements past L are zeros and leave the sum as it is
        const int ng_sum = min(n_total / 4, ng_row);
        if ((ng_sum & 31) && lane < 32) s_grp[xg_seg_at((ng_sum & ~31) + lane)] = 0.0f;       // an open last segment
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int r = 0; r < R; r++)
            if (64 * r < ng_row) {
                float e[4] = {v[r].x, v[r].y, v[r].z, v[r].w};
                uint32_t hx[4];
                bool ask[4];
#pragma unroll
                for (int k = 0; k < 4; k++) hx[k] = f2h(mx - e[k]);          // the argument without its sign
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    if constexpr (LIST) e[k] = xe_exp(hx[k], (const uint32_t *)s_mem, ask[k]);
                    else { e[k] = s_mem[min(hx[k], (uint32_t)XP_LUT)]; ask[k] = hx[k] > 0x7C00u; }      // entry XP_LUT: 0, exp of everything below
                }
                if (__any(ask[0] || ask[1] || ask[2] || ask[3])) {           // a NaN somewhere
                    const float w[4] = {v[r].x, v[r].y, v[r].z, v[r].w};
#pragma unroll
                    for (int k = 0; k < 4; k++) if (ask[k] && 4 * (lane + 64 * r) + k < L) e[k] = lut[f2h(w[k] - mx)];
                }
                v[r] = make_float4(e[0], e[1], e[2], e[3]);
                const int g = lane + 64 * r;
                const float v1 = e[0] + e[1], v2 = e[2] + e[3];
                if (g < ng_sum) s_grp[xg_seg_at(g)] = v1 + v2;
                if (g == ng_sum) { s_rem[0] = e[0]; s_rem[1] = e[1]; s_rem[2] = e[2]; s_rem[3] = e[3]; }      // the group that n_total cuts short: its elements are added one by one
            }
        __builtin_amdgcn_wave_barrier();
        float sum = xg_segment_sum<(R + 15) / 16>(s_grp, ng_sum);
        for (int i = n_total / 4 * 4; i < min(n_total, L); i++) sum = sum + s_rem[i & 3];
        const float inv = 1.0f / sum;
        uint2 *p4 = (uint2 *)(P16 + ((int64_t)h * T + t) * s_row);
        const int zend = (int)min((int64_t)((P + (t | 31) + 1 + 31) & ~31), s_row);       // a multiple of 32
#pragma unroll
        for (int r = 0; r < R; r++)
            if (64 * r < ng_row) {
                const int g = lane + 64 * r;
                if (g < ng_row)                                  // elements past L are zeros
                    p4[g] = make_uint2((uint32_t)f2h(v[r].x * inv) | ((uint32_t)f2h(v[r].y * inv) << 16), (uint32_t)f2h(v[r].z * inv) | ((uint32_t)f2h(v[r].w * inv) << 16));
            }
        for (int g = ng_row + lane; g < zend / 4; g += 64) p4[g] = make_uint2(0, 0);
        __builtin_amdgcn_wave_barrier();
    }
}
template <int R, int NW, int OCC, bool LIST>
int xp_softmax_launch(hipStream_t st, const float *S, uint16_t *P16, const float *lut, int T, int H, int P, int64_t s_row, int n_total, float scale, int ncu) {
    constexpr size_t lds = ((LIST ? XE_WORDS : XP_LUT + 4) + NW * (80 * R + 4)) * 4;
    constexpr int WGS = OCC * 4 / NW;                            // workgroups on a compute unit
    static_assert(lds * WGS <= 160 * 1024, "");
    const int rc = spy_raise_lds_limit((const void *)xp_softmax_kernel<R, NW, OCC, LIST>, lds);
    if (rc) return rc;
    const int64_t need = ((int64_t)T * H + NW - 1) / NW, most = (int64_t)ncu * WGS;
    xp_softmax_kernel<R, NW, OCC, LIST><<<dim3((unsigned)(need < most ? need : most)), dim3(64 * NW), lds, st>>>(S, P16, lut, T, H, P, s_row, n_total, scale);
    return SPY_LAUNCH_RC();
}

// ---------------------------------------------------------------- product with V^T
// One workgroup per (head, 32 query rows, 32 of the 128 output elements), a wave per 16 x 16 outputs: eight matrix instructions per chunk of 32 cached
// positions, instruction l for accumulators l, 8 + l, 16 + l, 24 + l, so that lane (g, j) supplies positions 8 g .. 8 g + 7 of V^T row j and of the
// probabilities of query row j: 16 bytes each, and every lane ends with all 32 accumulators of its four outputs.  Stages of two chunks go through LDS
// (rows of 128 bytes, their 16-byte pieces exchanged by the row so that reads and writes meet no bank twice), requested one stage ahead.
// 2048 rows on 2048 positions, 32 heads: 947 -> 557 us (the fmas on the vector units, a lane per accumulator); 77 rows on 1000: 26.5 -> 15.7.
// What bounds it: 348 us of matrix instructions and, beside none of them, the two conversions each needs (about 90).  Straight from memory without LDS:
// 705 us (the L2); two waves per SIMD instead of three: 609.
typedef uint32_t xp_u4 __attribute__((ext_vector_type(4), aligned(2)));          // V^T rows of a caller's cache: no more alignment than an element's
// PACK: the outputs leave as the packed activations of the MatMul that follows (xt_pack.cuh) instead of as floats: the 32 outputs of a row that a workgroup forms
// are one Q8_0 block.  A launch less, and the outputs do not go through memory: 8 rows 3.5 + 2.6 -> 4.4 us, 33 4.7 + 4.7 -> 5.1,
// 77 on 1000 positions 16.6 + 4.9 -> 17.5, 512 19.2 + 5.4 -> 21.6, 2048 215 + 10.2 -> 224.
// (With packing three registers do not fit, 16 bytes of scratch a lane, written before the loop and read behind it: in those times.)
template <bool PACK>
__global__ __launch_bounds__(256, 3) void xp_pv_kernel(const uint16_t *__restrict__ P16, const uint16_t *__restrict__ vt, float *__restrict__ out,
                                                       int T, int H, int P, int64_t p_row, int64_t C, int n_total, uint8_t *__restrict__ pack) {
    __shared__ __align__(16) xp_v4u s_v[2][32][8], s_p[2][32][8];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = lane >> 4, j = lane & 15;
    const int h = blockIdx.x, tb = ((int)gridDim.z - 1 - (int)blockIdx.z) * 32;      // head fastest: see xp_scores_kernel
    const int t0 = tb + (wave >> 1) * 16, dd0 = (int)blockIdx.y * 32 + (wave & 1) * 16;
    const int Lmax = P + min(tb + 31, T - 1) + 1;
    const int tail_start = (n_total - 1) / 32 * 32;
    // whole chunks, and the one whose elements the host adds one by one (tail_start on, where a row of the tile reaches it)
    const int nchunk = min(tail_start, (Lmax + 31) & ~31) / 32, nall = nchunk + (Lmax > tail_start ? 1 : 0);
    // staging: thread -> row tid / 8 of either tile, 16 of the 128 bytes
    const int st_row = threadIdx.x >> 3, st_i = threadIdx.x & 7, st_slot = st_i ^ ((st_row >> 1) & 7), st_pos = 8 * st_i;
    const uint16_t *vsrc = vt + ((int64_t)h * 128 + blockIdx.y * 32 + st_row) * C, *psrc = P16 + ((int64_t)h * T + min(tb + st_row, T - 1)) * p_row;
    xp_v16f acc[8];
#pragma unroll
    for (int l = 0; l < 8; l++) acc[l] = xp_zero();
    vsrc += st_pos;
    psrc += st_pos;
    xp_v4u vn, pn;
    auto fetch = [&](int s) {                                       // the next stage, s; a second chunk that does not exist is the first one again
        if (2 * s >= nall) return;
        const int back = 2 * s + 2 > nall && st_pos >= 32 ? 32 : 0;
        vn = *(const xp_u4 *)(vsrc - back);
        pn = *(const xp_v4u *)(psrc - back);
        vsrc += 64;
        psrc += 64;
        __builtin_amdgcn_sched_barrier(0);                          // (or the loads sink to where their data go into LDS)
    };
    const int rd_v = (wave & 1) * 16 + j, rd_p = (wave >> 1) * 16 + j, sw = (j >> 1) & 7;
    // a stage in buffer b (a wave that writes it is past the barrier of the stage before, which every wave reaches after its reads of it)
    auto put = [&](int b) {
        s_v[b][st_row][st_slot] = vn;
        s_p[b][st_row][st_slot] = pn;
        __syncthreads();
    };
    auto chunk = [&](int b, int c) {
        const xp_v4u v = s_v[b][rd_v][(4 * c + g) ^ sw], p = s_p[b][rd_p][(4 * c + g) ^ sw];
        float x[8], y[8];
        xp_widen(make_uint4(v.x, v.y, v.z, v.w), x);
        xp_widen(make_uint4(p.x, p.y, p.z, p.w), y);
#pragma unroll
        for (int l = 0; l < 8; l++) acc[l] = xp_mfma(x[l], y[l], acc[l]);
    };
    xp_v4f tail = {0.0f, 0.0f, 0.0f, 0.0f};
    auto tail_chunk = [&](int b, int c) {                           // v_mfma_f32_16x16x4_f32: the fmas of its four elements one after the other, bit for bit
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int slot = (4 * c + (i >> 1)) ^ sw, e = 4 * (i & 1) + g;          // lane (g, j): element 4 i + g of the chunk
            tail = __builtin_amdgcn_mfma_f32_16x16x4f32(h2f(((const uint16_t *)&s_v[b][rd_v][slot])[e]), h2f(((const uint16_t *)&s_p[b][rd_p][slot])[e]), tail, 0, 0, 0);
        }
    };
    fetch(0);
    const int nwhole = min(Lmax / 64, nchunk / 2);                  // stages of two chunks without a position past Lmax
    int s = 0;
    for (; s + 2 <= nwhole; s += 2) {
#pragma unroll
        for (int b = 0; b < 2; b++) {
            put(b);
            fetch(s + b + 1);
            chunk(b, 0);
            chunk(b, 1);
        }
    }
    for (; 2 * s < nall; s++) {
        const int left = Lmax - (64 * s + st_pos), b = s & 1;       // past Lmax every probability is 0, but the cache may hold anything
#pragma unroll
        for (int i = 0; i < 4; i++) vn[i] = left >= 2 * i + 2 ? vn[i] : left == 2 * i + 1 ? vn[i] & 0xFFFFu : 0u;
        put(b);
        fetch(s + 1);
#pragma unroll 1
        for (int c = 0; c < 2; c++)
            if (2 * s + c < nchunk) chunk(b, c);
            else if (2 * s + c < nall) tail_chunk(b, c);
    }
    // FP16::block_reduce: t_l from the four accumulators of instruction l, t_l + t_(l + 4), (u0 + u1) + (u2 + u3)
    float u[4][4];
#pragma unroll
    for (int l = 0; l < 4; l++) {
        float x[4], y[4];
        xp_reduce8(acc[l], x);
        xp_reduce8(acc[l + 4], y);
#pragma unroll
        for (int v = 0; v < 4; v++) u[l][v] = x[v] + y[v];
    }
    const int t = t0 + j;
    if (!PACK && t >= T) return;
    float o[4];
#pragma unroll
    for (int v = 0; v < 4; v++) {
        const float x = u[0][v] + u[1][v], y = u[2][v] + u[3][v];
        o[v] = tail[v] + (x + y);
    }
    if constexpr (PACK) {
        // the 32 x 32 outputs through LDS (rows of 36 floats) to eight lanes per row; rows past T are zeros
        static_assert(32 * 36 * 4 <= sizeof(s_v), "");
        float *s_o = (float *)s_v;
        const float4 z = t < T ? make_float4(o[0], o[1], o[2], o[3]) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        __syncthreads();
        *(float4 *)(s_o + ((wave >> 1) * 16 + j) * 36 + (wave & 1) * 16 + 4 * g) = z;
        __syncthreads();
        const int c = threadIdx.x >> 3, e = threadIdx.x & 7, ncg = (T + 15) / 16, cg = tb / 16 + (c >> 4);
        if (cg < ncg) xt_store4(*(const float4 *)(s_o + c * 36 + 4 * e), cg, H, h * 4 + (int)blockIdx.y, c & 15, e, pack, pack + (int64_t)ncg * H * XT_XB);
    } else *(float4 *)(out + (int64_t)t * H * 128 + (int64_t)h * 128 + dd0 + 4 * g) = make_float4(o[0], o[1], o[2], o[3]);
}

}   // namespace

// q: after Rope, fp32 [T][H][128], or (q_f16) fp16 [H][T][128]; kc: fp16 [position][H][128]; vt: fp16 [H * 128][C]; out: fp32 [T][H][128], or pack: the outputs as packed activations;
// S: H * T * s_row floats and P16: H * T * s_row halves of scratch, s_row = spy_exact_prompt_attn_row(P + T)
int64_t spy_exact_prompt_attn_row(int64_t n_kv) { return (n_kv + 127) & ~(int64_t)127; }

static int prompt_attn(hipStream_t st, const void *q, bool q_f16, const uint16_t *kc, const uint16_t *vt, float *S, uint16_t *P16, float *out, const float *lut,
                          int T, int H, int P, int64_t C, int n_total, float scale, void *pack) {
    if (T <= 0 || H <= 0 || H > 65535 || P < 0 || (int64_t)P + T > C || n_total < P + T || n_total > C || C % 32) return SPY_HIP_EINVAL;
    if ((int64_t)P + T > 256 * XP_SM_R) return SPY_HIP_EUNSUPPORTED;      // the softmax kernel keeps a row in the registers of a wave
    if (((uintptr_t)q & 15) || ((uintptr_t)kc & 15) || ((uintptr_t)S & 15) || ((uintptr_t)P16 & 15) || ((uintptr_t)out & 15) || ((uintptr_t)pack & 15)) return SPY_HIP_EINVAL;
    const int64_t s_row = spy_exact_prompt_attn_row((int64_t)P + T);
    // segments of the cached positions: 512 long where that gives every compute unit its four workgroups three times over, down to one key tile for short passes (512 rows
    // with 1024 workgroups asked for 28.8 us, 2048 22.0, 3072 21.6, 4096 22.0; 1000 rows 75.8, 66.4, 62.0, 62.2; 77 rows on 1000 positions 16.4 with any)
    const int tiles = (T + 63) / 64;
    int kseg = XP_KSEG;
    while (kseg > 64 && (int64_t)H * tiles * ((P + T + kseg - 1) / kseg) < 3072) kseg >>= 1;
    const dim3 sgrid((unsigned)H, (unsigned)tiles, (unsigned)((P + T + kseg - 1) / kseg));
    if (q_f16) xp_scores_kernel<true><<<sgrid, dim3(256), 0, st>>>(q, kc, S, T, H, P, s_row, kseg);
    else xp_scores_kernel<false><<<sgrid, dim3(256), 0, st>>>(q, kc, S, T, H, P, s_row, kseg);
    if (hipGetLastError() != hipSuccess) return SPY_HIP_EINVAL;
    const int64_t n_kv = (int64_t)P + T;
    const int ncu = spy_num_cu();
    const bool few = (int64_t)T * H <= XP_LIST_ROWS;
#define XP_SOFTMAX(...) xp_softmax_launch<__VA_ARGS__>(st, S, P16, lut, T, H, P, s_row, n_total, scale, ncu)
    const int rc = n_kv <= 2048 ? (few ? XP_SOFTMAX(8, 4, 5, true) : XP_SOFTMAX(8, 16, 4, false)) : n_kv <= 4096 ? (few ? XP_SOFTMAX(16, 4, 3, true) : XP_SOFTMAX(16, 12, 3, false))
                 : n_kv <= 6144 ? XP_SOFTMAX(24, 8, 2, false) : XP_SOFTMAX(32, 4, 1, false);
#undef XP_SOFTMAX
    if (rc) return rc;
    const dim3 pgrid((unsigned)H, 4, (unsigned)((T + 31) / 32));
    if (pack) xp_pv_kernel<true><<<pgrid, dim3(256), 0, st>>>(P16, vt, nullptr, T, H, P, s_row, C, n_total, (uint8_t *)pack);
    else xp_pv_kernel<false><<<pgrid, dim3(256), 0, st>>>(P16, vt, out, T, H, P, s_row, C, n_total, nullptr);
    return SPY_LAUNCH_RC();
}

int spy_exact_prompt_attn(hipStream_t st, const void *q, bool q_f16, const uint16_t *kc, const uint16_t *vt, float *S, uint16_t *P16, float *out, const float *lut,
                          int T, int H, int P, int64_t C, int n_total, float scale) {
    return prompt_attn(st, q, q_f16, kc, vt, S, P16, out, lut, T, H, P, C, n_total, scale, nullptr);
}
// q: fp16 [H][T][128]; the outputs as packed activations: spy_xgemm_pack_bytes(T, 128 H) bytes
int spy_exact_prompt_attn_pack(hipStream_t st, const uint16_t *q16, const uint16_t *kc, const uint16_t *vt, float *S, uint16_t *P16, void *pack, const float *lut,
                               int T, int H, int P, int64_t C, int n_total, float scale) {
    if (!pack || H % 2) return SPY_HIP_EINVAL;
    return prompt_attn(st, q16, true, kc, vt, S, P16, nullptr, lut, T, H, P, C, n_total, scale, pack);
}

int spy_exact_luts(const float **lut);           // exact_order.hip

extern "C" size_t spy_hip_prompt_attention_exact_scratch_size(int32_t T, int32_t H, int32_t past) {
    if (T <= 0 || H <= 0 || past < 0) return 0;
    return (size_t)spy_exact_prompt_attn_row((int64_t)past + T) * (size_t)T * (size_t)H * 6;       // fp32 scores, then fp16 probabilities
}

extern "C" int spy_hip_prompt_attention_exact(void *stream, const float *q, const void *k_cache, const void *v_cache, float *out, int32_t T, int32_t H,
                                              int32_t hd, int32_t past, int64_t n_ctx, int32_t n_total, float scale, void *scratch, size_t scratch_bytes) {
    SPY_CHECK_ARG(q && k_cache && v_cache && out && scratch);
    if (hd != 128 || n_ctx % 32) return SPY_HIP_EUNSUPPORTED;
    const size_t need = spy_hip_prompt_attention_exact_scratch_size(T, H, past);
    if (!need) return SPY_HIP_EINVAL;
    if (scratch_bytes < need || ((uintptr_t)scratch & 255)) return SPY_HIP_ENOSPACE;
    const float *lut = nullptr;
    const int rc = spy_exact_luts(&lut);
    if (rc) return rc;
    float *S = (float *)scratch;
    uint16_t *P16 = (uint16_t *)((uint8_t *)scratch + need / 6 * 4);
    return spy_exact_prompt_attn((hipStream_t)stream, q, false, (const uint16_t *)k_cache, (const uint16_t *)v_cache, S, P16, out, lut, T, H, past, n_ctx, n_total, scale);
}

// xe_exp argument by argument (exact_exp.cuh), the list in LDS as the attention kernels have it
__global__ __launch_bounds__(256) void exp_f16_kernel(const uint16_t *__restrict__ x, int64_t n, int worked_out, const float *__restrict__ lut, float *__restrict__ out) {
    __shared__ __align__(16) uint32_t s_code[XE_WORDS];
    for (int i = threadIdx.x; i < XE_WORDS / 4; i += 256) ((uint4 *)s_code)[i] = ((const uint4 *)(lut + XE_AT))[i];
    __syncthreads();
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
        bool ask = true;
        float e = 0.0f;
        if (worked_out) e = xe_exp((uint32_t)x[i] ^ 0x8000u, s_code, ask);
        out[i] = ask ? lut[x[i]] : e;
    }
}
extern "C" int spy_hip_exp_f16(void *stream, const void *x, int64_t n, int32_t worked_out, float *out) {
    SPY_CHECK_ARG(x && out && n > 0 && (worked_out == 0 || worked_out == 1) && ((uintptr_t)x % 2) == 0 && ((uintptr_t)out % 4) == 0);
    const float *lut = nullptr;
    const int rc = spy_exact_luts(&lut);
    if (rc) return rc;
    const int64_t need = (n + 255) / 256;
    exp_f16_kernel<<<dim3((unsigned)(need < 1024 ? need : 1024)), dim3(256), 0, (hipStream_t)stream>>>((const uint16_t *)x, n, worked_out, lut, out);
    return SPY_LAUNCH_RC();
}
