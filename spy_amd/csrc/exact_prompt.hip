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
// Values that cannot occur are not looked after: the fp16 caches are written by this library's float -> half
// conversion, which never produces the pattern 0xFFFF that the host's conversion table maps to 0 (conversion.h:39-41).
#include "common.cuh"
#include "exact_sum.cuh"

namespace {

typedef _Float16 xp_half2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ xp_half2 xp_pack(float a, float b) {
    xp_half2 r;
    r.x = __builtin_bit_cast(_Float16, f2h(a));
    r.y = __builtin_bit_cast(_Float16, f2h(b));
    return r;
}

// ---------------------------------------------------------------- scores
// One workgroup per (head, 128 query rows); a lane takes query rows t0 + lane and t0 + 64 + lane, their 2 x 128 q values
// as packed fp16 pairs in registers.  A tile of 64 key rows is brought into LDS by the whole workgroup; every lane of a
// wave reads the same key row -- LDS delivers that as a broadcast, but
// at the cost of a full read, which is why a key row read serves two query rows per lane: with one, the kernel ran at the
// LDS read rate (16 ds_read_b128 per 160 vector instructions).  A wave takes 16 of the 64 cached positions of a tile; the
// scores go through LDS as well so that the rows of S are written in whole segments.
#define XP_QT 128
#define XP_KSEG 512
// fma(float(lower halves), c) and fma(float(upper halves), c) of two packed fp16 pairs, written out as instructions: left to
// itself the compiler folds only one fp16 source into v_fma_mix_f32 and converts the loop-invariant q values to fp32 (once, which
// doubles the registers they occupy, or inside the loop, which doubles the instructions)
__device__ __forceinline__ float xp_fma_lo(uint32_t a, uint32_t b, float c) {
    float r;
    asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel_hi:[1,1,0]" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
__device__ __forceinline__ float xp_fma_hi(uint32_t a, uint32_t b, float c) {
    float r;
    asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[1,1,0] op_sel_hi:[1,1,0]" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}

// One key row (in LDS, 16 x 16 bytes) against the two query rows of a lane; the row is taken in its four chunks of 32 elements
// so that only one chunk of it is in registers at a time.  A, B: the first / second query row takes part (else its score is not needed).
template <bool A, bool B, int NB>
__device__ __forceinline__ void xp_dot128_pair(const uint32_t (&qa)[64], const uint32_t (&qb)[NB], const uint4 *kr, float &sa, float &sb) {
    float sum_a[32], sum_b[32];
    // chunks of 32 elements while i + 32 < 128: accumulator l takes elements l, 32 + l, 64 + l
#pragma unroll
    for (int c = 0; c < 3; c++) {
        uint4 k4[4];
#pragma unroll
        for (int v = 0; v < 4; v++) k4[v] = kr[4 * c + v];
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const uint32_t kw[4] = {k4[v].x, k4[v].y, k4[v].z, k4[v].w};
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int l = 8 * v + 2 * i, qi = 16 * c + 4 * v + i;
                if (A) {
                    sum_a[l] = xp_fma_lo(kw[i], qa[qi], c == 0 ? 0.0f : sum_a[l]);
                    sum_a[l + 1] = xp_fma_hi(kw[i], qa[qi], c == 0 ? 0.0f : sum_a[l + 1]);
                }
                if (B) {
                    sum_b[l] = xp_fma_lo(kw[i], qb[qi], c == 0 ? 0.0f : sum_b[l]);
                    sum_b[l + 1] = xp_fma_hi(kw[i], qb[qi], c == 0 ? 0.0f : sum_b[l + 1]);
                }
            }
        }
    }
    // the last 32 elements one by one (their products are exact in fp32, so each step is one fma)
    float tail_a = 0.0f, tail_b = 0.0f;
    {
        uint4 k4[4];
#pragma unroll
        for (int v = 0; v < 4; v++) k4[v] = kr[12 + v];
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const uint32_t kw[4] = {k4[v].x, k4[v].y, k4[v].z, k4[v].w};
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int qi = 48 + 4 * v + i;
                if (A) { tail_a = xp_fma_lo(kw[i], qa[qi], tail_a); tail_a = xp_fma_hi(kw[i], qa[qi], tail_a); }
                if (B) { tail_b = xp_fma_lo(kw[i], qb[qi], tail_b); tail_b = xp_fma_hi(kw[i], qb[qi], tail_b); }
            }
        }
    }
    // FP16::block_reduce (vec_util.h:61-71), then result = tail + that sum
    auto reduce = [](float (&sum)[32]) {
#pragma unroll
        for (int l = 0; l < 8; l++) { sum[l] += sum[16 + l]; sum[8 + l] += sum[24 + l]; }
#pragma unroll
        for (int l = 0; l < 8; l++) sum[l] += sum[8 + l];
        const float u0 = sum[0] + sum[4], u1 = sum[1] + sum[5], u2 = sum[2] + sum[6], u3 = sum[3] + sum[7];
        return (u0 + u1) + (u2 + u3);
    };
    if (A) sa = tail_a + reduce(sum_a);
    if (B) sb = tail_b + reduce(sum_b);
}

// ONE: 64 query rows per workgroup, one per lane (short passes: twice the waves per SIMD, half the granularity)
template <bool F16Q, bool ONE>     // q: f32 [T][H * 128] as Rope leaves it, or already rounded to fp16 and laid out [H][T][128]
__global__ __launch_bounds__(256, 2) void xp_scores_kernel(const void *__restrict__ q, const uint16_t *__restrict__ kc, float *__restrict__ S,
                                                           int T, int H, int P, int64_t s_row, int kseg) {
    constexpr int QT = ONE ? 64 : XP_QT;
    __shared__ float s_tile[QT][65];
    __shared__ __align__(16) uint4 s_k[64][16];                  // 64 key rows of 256 bytes
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // The head is the fastest-running index of the grid: consecutive workgroups go to the eight XCDs in turn, and with the query tile
    // there an XCD would get tiles k and k + 8 of 16 only -- under the causal mask 24 to 10 units of work (68 % of the compute units
    // busy over the launch).  With the head there every XCD gets the same mix of tiles, and the key rows of its heads stay in its L2.
    const int t0 = ((int)gridDim.y - 1 - (int)blockIdx.y) * QT, h = blockIdx.x;      // the longest rows first
    const int64_t d = (int64_t)H * 128;
    // the cached positions are dealt out in segments of kseg (a multiple of 64) over blockIdx.z, so that the workgroups are of similar length
    // (one workgroup per 128 query rows would make the longest rows the critical path of the launch)
    const int kv_end = min(P + min(t0 + QT - 1, T - 1) + 1, ((int)blockIdx.z + 1) * kseg);       // cached positions that some row of the tile may see, within this segment
    if ((int)blockIdx.z * kseg >= kv_end) return;
    uint32_t qa[64], qb[ONE ? 1 : 64];
    if constexpr (F16Q) {
        const uint4 *qp = (const uint4 *)((const uint16_t *)q + ((int64_t)h * T + min(t0 + lane, T - 1)) * 128), *qp2 = (const uint4 *)((const uint16_t *)q + ((int64_t)h * T + min(t0 + 64 + lane, T - 1)) * 128);
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const uint4 f = qp[i], f2 = qp2[i];
            qa[4 * i] = f.x; qa[4 * i + 1] = f.y; qa[4 * i + 2] = f.z; qa[4 * i + 3] = f.w;
            if constexpr (!ONE) { qb[4 * i] = f2.x; qb[4 * i + 1] = f2.y; qb[4 * i + 2] = f2.z; qb[4 * i + 3] = f2.w; }
        }
    } else {
        const float4 *qp = (const float4 *)((const float *)q + (int64_t)min(t0 + lane, T - 1) * d + (int64_t)h * 128);
        const float4 *qp2 = (const float4 *)((const float *)q + (int64_t)min(t0 + 64 + lane, T - 1) * d + (int64_t)h * 128);
#pragma unroll
        for (int i = 0; i < 32; i++) {
            const float4 f = qp[i], f2 = qp2[i];
            qa[2 * i] = __builtin_bit_cast(uint32_t, xp_pack(f.x, f.y));
            qa[2 * i + 1] = __builtin_bit_cast(uint32_t, xp_pack(f.z, f.w));
            if constexpr (!ONE) {
                qb[2 * i] = __builtin_bit_cast(uint32_t, xp_pack(f2.x, f2.y));
                qb[2 * i + 1] = __builtin_bit_cast(uint32_t, xp_pack(f2.z, f2.w));
            }
        }
    }
    const int kv_end_a = P + min(t0 + 63, T - 1) + 1;            // cached positions that some row of the tile's first half may see
    // staging: thread -> key row tid / 4 of the tile, 64 of its 256 bytes
    const int st_row = threadIdx.x >> 2, st_q = (threadIdx.x & 3) * 4;
    uint4 kst0, kst1, kst2, kst3;
#define XP_FETCH_K(kv_first) do { \
        const uint4 *src_ = (const uint4 *)(kc + (int64_t)min((kv_first) + st_row, kv_end - 1) * d + (int64_t)h * 128) + st_q; \
        kst0 = src_[0]; kst1 = src_[1]; kst2 = src_[2]; kst3 = src_[3]; } while (0)
    for (int kv0 = (int)blockIdx.z * kseg; kv0 < kv_end; kv0 += 64) {
        // (no key tile travelling in registers during the dots: with 2 x 64 registers of q values and 2 x 32 accumulators there is
        // no room for it; the second workgroup of the compute unit covers the wait)
        XP_FETCH_K(kv0);
        s_k[st_row][st_q] = kst0; s_k[st_row][st_q + 1] = kst1; s_k[st_row][st_q + 2] = kst2; s_k[st_row][st_q + 3] = kst3;
        __syncthreads();
        const bool first_half = kv0 < kv_end_a;                   // else the whole key tile lies behind the mask of query rows t0 .. t0 + 63
#pragma unroll 1
        for (int j = 0; j < 16; j++) {
            const int kvl = wave * 16 + j;
            float sa = 0.0f, sb = 0.0f;
            if (kv0 + kvl < kv_end) {
                if constexpr (ONE) xp_dot128_pair<true, false, 64>(qa, qa, s_k[kvl], sa, sb);
                else if (first_half) xp_dot128_pair<true, true, 64>(qa, qb, s_k[kvl], sa, sb);
                else xp_dot128_pair<false, true, 64>(qa, qb, s_k[kvl], sa, sb);
            }
            s_tile[lane][kvl] = sa;
            if constexpr (!ONE) s_tile[64 + lane][kvl] = sb;
        }
        __syncthreads();
        {
            constexpr int W = ONE ? 16 : 32;                      // scores per thread
            const int row = threadIdx.x / (64 / W), seg = threadIdx.x % (64 / W);
            if (t0 + row < T && (row >= 64 || first_half)) {
                float4 *out = (float4 *)(S + ((int64_t)h * T + t0 + row) * s_row + kv0 + seg * W);
#pragma unroll
                for (int i = 0; i < W / 4; i++)
                    out[i] = make_float4(s_tile[row][seg * W + 4 * i], s_tile[row][seg * W + 4 * i + 1], s_tile[row][seg * W + 4 * i + 2],
                                         s_tile[row][seg * W + 4 * i + 3]);
            }
        }
        // the next tile's key rows go into s_k at the top of the loop: every wave is past its reads of s_k once it has passed the
        // barrier above, and the barrier after the writes orders them against the next reads
    }
#undef XP_FETCH_K
}

// ---------------------------------------------------------------- softmax
// One wave per (head, query row), NW waves per resident workgroup, rows dealt out in turn (the longest first); L = the positions the row may see.  A
// lane keeps its share of the row in registers (groups of four consecutive elements, the unit of the host's sum), so the row is read once
// and written once.  The probabilities leave as fp16 (the first step of the KQV MatMul, mat.cpp:37), followed by zeros up to the end of the
// 32-row tile's last chunk, which the product kernel reads.
// The exponentials: a gather of 64 table entries from memory takes about 64 cycles of the compute unit, so the part of the table that is not zero lies in
// LDS: arguments are <= 0 (or NaN), and exp is 0 from -104 on.  The sum of a row goes through xg_segment_sum: 2 us instead of a chain of up to
// 1024 additions.  2048 rows of 2049 .. 4096 positions and 32 heads (1.2 GB): 462 -> 306 us; 2048 rows of 1 .. 2048: 193 -> 152.
#define XP_LUT 0x5680      // fp16 -104.0 without its sign
#define XP_SM_R 32         // groups per lane: rows of up to 8192 positions
template <int R, int NW>
__global__ __launch_bounds__(64 * NW) void xp_softmax_kernel(const float *__restrict__ S, uint16_t *__restrict__ P16, const float *__restrict__ lut, int T, int H, int P,
                                                             int64_t s_row, int n_total, float scale) {
    extern __shared__ __align__(16) float s_mem[];               // table, then per wave 64 R padded group sums and 4 floats
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    float *s_grp = s_mem + XP_LUT + 4 + wave * (80 * R + 4), *s_rem = s_grp + 80 * R;
    for (int i = threadIdx.x; i <= XP_LUT / 4; i += 64 * NW) ((float4 *)s_mem)[i] = ((const float4 *)(lut + 0x8000))[i];
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
#pragma unroll
                for (int k = 0; k < 4; k++) hx[k] = f2h(mx - e[k]);          // the argument without its sign
#pragma unroll
                for (int k = 0; k < 4; k++) e[k] = s_mem[min(hx[k], (uint32_t)XP_LUT)];      // entry XP_LUT: 0, exp of everything below
                if (__any(max(max(hx[0], hx[1]), max(hx[2], hx[3])) > 0x7C00u)) {            // a NaN somewhere
                    const float w[4] = {v[r].x, v[r].y, v[r].z, v[r].w};
#pragma unroll
                    for (int k = 0; k < 4; k++) if (hx[k] > 0x7C00u && 4 * (lane + 64 * r) + k < L) e[k] = lut[f2h(w[k] - mx)];
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
template <int R, int NW>
int xp_softmax_launch(hipStream_t st, const float *S, uint16_t *P16, const float *lut, int T, int H, int P, int64_t s_row, int n_total, float scale, int ncu) {
    constexpr size_t lds = (XP_LUT + 4 + NW * (80 * R + 4)) * 4;
    static_assert(lds <= 160 * 1024, "");
    const int rc = spy_raise_lds_limit((const void *)xp_softmax_kernel<R, NW>, lds);
    if (rc) return rc;
    const int64_t need = ((int64_t)T * H + NW - 1) / NW;
    xp_softmax_kernel<R, NW><<<dim3((unsigned)(need < ncu ? need : ncu)), dim3(64 * NW), lds, st>>>(S, P16, lut, T, H, P, s_row, n_total, scale);
    return SPY_LAUNCH_RC();
}

// ---------------------------------------------------------------- product with V^T
// One workgroup per (head, 32 query rows, 32 of the 128 output elements); eight groups of 32 lanes, a group takes four
// output elements.  Lane l of a group keeps accumulator l (cached positions 32c + l) of its 4 x 32 outputs, so a V value is
// loaded once for 32 query rows; the probabilities of a chunk come through LDS, transposed to [position][row].
// After the chunks the 32 accumulators of every output are added in the tree of FP16::block_reduce, spread over the lanes so
// that lane l ends with the outputs of query row l, and the scalar tail of the host loop follows.
#define XP_PT 32
#define XP_SC 4            // chunks of 32 positions per stage
__global__ __launch_bounds__(256, 2) void xp_pv_kernel(const uint16_t *__restrict__ P16, const uint16_t *__restrict__ vt, float *__restrict__ out,
                                                       int T, int H, int P, int64_t p_row, int64_t C, int n_total) {
    __shared__ __align__(16) uint16_t s_p[2][32 * XP_SC][40];  // [buffer][position in the stage][query row], rows of 80 bytes
    const int g = threadIdx.x >> 5, l = threadIdx.x & 31;
    const int t0 = ((int)gridDim.z - 1 - (int)blockIdx.z) * XP_PT, h = blockIdx.x;      // head fastest: see xp_scores_kernel
    const int dd0 = blockIdx.y * 32 + g * 4;
    const int Lmax = P + min(t0 + XP_PT - 1, T - 1) + 1;
    const int tail_start = (n_total - 1) / 32 * 32;
    const int nchunk = min(tail_start, (Lmax + 31) & ~31) / 32;
    const int nstage = (nchunk + XP_SC - 1) / XP_SC;
    const uint16_t *vrow[4];
#pragma unroll
    for (int j = 0; j < 4; j++) vrow[j] = vt + ((int64_t)h * 128 + dd0 + j) * C + l;
    // staging of the probabilities: thread -> query row tid % 32, sixteen positions; neighbouring lanes write neighbouring
    // query rows of one position, i.e. neighbouring LDS words (the other way round, 64 lanes would meet in four banks)
    const int st_t = threadIdx.x & 31, st_k = (threadIdx.x >> 5) * 16;
    const uint16_t *prow = P16 + ((int64_t)h * T + min(t0 + st_t, T - 1)) * p_row + st_k;
    float acc[4][32];
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
        for (int i = 0; i < 32; i++) acc[j][i] = 0.0f;
    uint4 pst[2];
    uint16_t vn[XP_SC][4];
    auto fetch = [&](int s) {
        pst[0] = *(const uint4 *)(prow + 32 * XP_SC * s);
        pst[1] = *(const uint4 *)(prow + 32 * XP_SC * s + 8);
#pragma unroll
        for (int c = 0; c < XP_SC; c++) {
            const int pos = 32 * (XP_SC * s + c);
#pragma unroll
            for (int j = 0; j < 4; j++) vn[c][j] = pos + l < Lmax ? vrow[j][pos] : (uint16_t)0;      // past Lmax every probability is 0; the cache may hold anything there
        }
    };
    auto put = [&](int buf) {
#pragma unroll
        for (int v = 0; v < 2; v++) {
            const uint32_t w[4] = {pst[v].x, pst[v].y, pst[v].z, pst[v].w};
#pragma unroll
            for (int i = 0; i < 4; i++) {
                s_p[buf][st_k + 8 * v + 2 * i][st_t] = (uint16_t)(w[i] & 0xFFFFu);
                s_p[buf][st_k + 8 * v + 2 * i + 1][st_t] = (uint16_t)(w[i] >> 16);
            }
        }
    };
    if (nstage > 0) {
        fetch(0);
        put(0);
    }
    __syncthreads();
    for (int s = 0; s < nstage; s++) {
        const int buf = s & 1;
        _Float16 vc[XP_SC][4];
#pragma unroll
        for (int c = 0; c < XP_SC; c++)
#pragma unroll
            for (int j = 0; j < 4; j++) vc[c][j] = __builtin_bit_cast(_Float16, vn[c][j]);
        if (s + 1 < nstage) fetch(s + 1);
#pragma unroll
        for (int c = 0; c < XP_SC; c++) {
            if (XP_SC * s + c < nchunk) {
                const uint4 *pp = (const uint4 *)&s_p[buf][32 * c + l][0];
#pragma unroll
                for (int qd = 0; qd < 4; qd++) {
                    const uint4 w4 = pp[qd];
                    const uint32_t w[4] = {w4.x, w4.y, w4.z, w4.w};
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const xp_half2 p2 = __builtin_bit_cast(xp_half2, w[i]);
#pragma unroll
                        for (int j = 0; j < 4; j++) {
                            acc[j][8 * qd + 2 * i] = fmaf((float)vc[c][j], (float)p2.x, acc[j][8 * qd + 2 * i]);
                            acc[j][8 * qd + 2 * i + 1] = fmaf((float)vc[c][j], (float)p2.y, acc[j][8 * qd + 2 * i + 1]);
                        }
                    }
                }
            }
        }
        if (s + 1 < nstage) put(buf ^ 1);
        __syncthreads();
    }
    // The tree: sum[l] += sum[l + 16], sum[l] += sum[l + 8], t_l = sum[l] + sum[l + 4], (t0 + t1) + (t2 + t3), where l is the lane.
    // At each step a lane keeps the half of its query rows that matches its own lane bit and hands the other half to its
    // partner, so 16 + 8 + 4 + 2 + 1 exchanges per output element leave lane l with the sum of query row l.
    float res[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        float a16[16], a8[8], a4[4], a2[2];
        const bool b4 = l & 16, b3 = l & 8, b2 = l & 4, b0 = l & 1, b1 = l & 2;
#pragma unroll
        for (int k = 0; k < 16; k++) {
            const float keep = b4 ? acc[j][k + 16] : acc[j][k], send = b4 ? acc[j][k] : acc[j][k + 16];
            a16[k] = keep + __shfl_xor(send, 16, SPY_WAVE);
        }
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const float keep = b3 ? a16[k + 8] : a16[k], send = b3 ? a16[k] : a16[k + 8];
            a8[k] = keep + __shfl_xor(send, 8, SPY_WAVE);
        }
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const float keep = b2 ? a8[k + 4] : a8[k], send = b2 ? a8[k] : a8[k + 4];
            a4[k] = keep + __shfl_xor(send, 4, SPY_WAVE);
        }
        // query rows left: 4 per lane, their index = (l & 28) + k; the tree goes on with lane bit 0, then bit 1
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const float keep = b0 ? a4[2 * k + 1] : a4[2 * k], send = b0 ? a4[2 * k] : a4[2 * k + 1];
            a2[k] = keep + __shfl_xor(send, 1, SPY_WAVE);
        }
        {
            const float keep = b1 ? a2[1] : a2[0], send = b1 ? a2[0] : a2[1];
            res[j] = keep + __shfl_xor(send, 2, SPY_WAVE);
        }
    }
    // lane l now holds query row t0 + l: rows were halved by lane bits 4, 3, 2 (index bits 4, 3, 2), then bit 0 chose index bit 0 and
    // bit 1 index bit 1
    const int t = t0 + l;
    if (t >= T) return;
    const int Lt = P + t + 1;                                      // positions row t sees
    const int tail_end = min(n_total, Lt);
    const uint16_t *pr = P16 + ((int64_t)h * T + t) * p_row;
    float o4[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        float tail = 0.0f;
        const uint16_t *vr = vt + ((int64_t)h * 128 + dd0 + j) * C;
        for (int i = tail_start; i < tail_end; i++) {
            const float pr_ = h2f(vr[i]) * h2f(pr[i]);
            tail += pr_;
        }
        o4[j] = tail + res[j];
    }
    *(float4 *)(out + (int64_t)t * H * 128 + (int64_t)h * 128 + dd0) = make_float4(o4[0], o4[1], o4[2], o4[3]);
}

}   // namespace

// q: after Rope, fp32 [T][H][128], or (q_f16) fp16 [H][T][128]; kc: fp16 [position][H][128]; vt: fp16 [H * 128][C]; out: fp32 [T][H][128];
// S: H * T * s_row floats and P16: H * T * s_row halves of scratch, s_row = spy_exact_prompt_attn_row(P + T)
int64_t spy_exact_prompt_attn_row(int64_t n_kv) { return (n_kv + 127) & ~(int64_t)127; }

int spy_exact_prompt_attn(hipStream_t st, const void *q, bool q_f16, const uint16_t *kc, const uint16_t *vt, float *S, uint16_t *P16, float *out, const float *lut,
                          int T, int H, int P, int64_t C, int n_total, float scale) {
    if (T <= 0 || H <= 0 || H > 65535 || P < 0 || (int64_t)P + T > C || n_total < P + T || n_total > C || C % 32) return SPY_HIP_EINVAL;
    if ((int64_t)P + T > 256 * XP_SM_R) return SPY_HIP_EUNSUPPORTED;      // the softmax kernel keeps a row in the registers of a wave
    if (((uintptr_t)q & 15) || ((uintptr_t)kc & 15) || ((uintptr_t)S & 15) || ((uintptr_t)P16 & 7) || ((uintptr_t)out & 15)) return SPY_HIP_EINVAL;
    const int64_t s_row = spy_exact_prompt_attn_row((int64_t)P + T);
    // segments of the cached positions: 512 long where that fills the chip, down to one key tile for short passes (77 tokens on 1000 cached ones
    // gave 96 workgroups: 114 us; one per 64 positions and 64 query rows 29)
    const bool one = T <= 256;
    const int tiles = (T + (one ? 64 : XP_QT) - 1) / (one ? 64 : XP_QT);
    int kseg = XP_KSEG;
    while (kseg > 64 && (int64_t)H * tiles * ((P + T + kseg - 1) / kseg) < 1024) kseg >>= 1;
    const dim3 sgrid((unsigned)H, (unsigned)tiles, (unsigned)((P + T + kseg - 1) / kseg));
    if (q_f16 && one) xp_scores_kernel<true, true><<<sgrid, dim3(256), 0, st>>>(q, kc, S, T, H, P, s_row, kseg);
    else if (q_f16) xp_scores_kernel<true, false><<<sgrid, dim3(256), 0, st>>>(q, kc, S, T, H, P, s_row, kseg);
    else if (one) xp_scores_kernel<false, true><<<sgrid, dim3(256), 0, st>>>(q, kc, S, T, H, P, s_row, kseg);
    else xp_scores_kernel<false, false><<<sgrid, dim3(256), 0, st>>>(q, kc, S, T, H, P, s_row, kseg);
    if (hipGetLastError() != hipSuccess) return SPY_HIP_EINVAL;
    const int ncu = spy_num_cu(), rc = (int64_t)P + T <= 4096 ? xp_softmax_launch<16, 12>(st, S, P16, lut, T, H, P, s_row, n_total, scale, ncu)
                                         : (int64_t)P + T <= 6144 ? xp_softmax_launch<24, 8>(st, S, P16, lut, T, H, P, s_row, n_total, scale, ncu)
                                                                  : xp_softmax_launch<32, 4>(st, S, P16, lut, T, H, P, s_row, n_total, scale, ncu);
    if (rc) return rc;
    xp_pv_kernel<<<dim3((unsigned)H, 4, (unsigned)((T + XP_PT - 1) / XP_PT)), dim3(256), 0, st>>>(P16, vt, out, T, H, P, s_row, C, n_total);
    return SPY_LAUNCH_RC();
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
