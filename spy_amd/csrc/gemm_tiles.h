// Which kernel and tile a MatMul from packed activations (exact_gemm.hip) takes.  Plain C++: a test on the host asks the same functions which tiles its shapes reach.
#pragma once

#include <cstdint>

// Which tile.  n workgroups per compute unit take about lat + (n - 1) * inc: figures in tenths of a microsecond for K = 4096, measured for
// n = 1 .. 16 (whole workgroups count while they are few; everything scales with K).  Small tiles have the shorter chain, large ones unpack a
// weight for more activation rows.
// rest: what a workgroup of the ncg % groups groups that remain takes, 0 if it is a whole one.
struct xt_cost { int rows, groups, lat, inc, rest = 0; };
inline int xt_pick(int64_t M, int nmat, int ncg, int64_t cu, const xt_cost *c, int n) {
    int best = 0;
    int64_t least = 0;
    for (int i = 0; i < n; i++) {
        const int64_t tiles = (M + c[i].rows - 1) / c[i].rows * nmat, wgs = tiles * (c[i].rest ? ncg / c[i].groups : (ncg + c[i].groups - 1) / c[i].groups);
        const int64_t t = c[i].lat + (wgs <= 6 * cu && !c[i].rest ? (wgs + cu - 1) / cu * 10 - 10 : 10 * wgs / cu - 10) * c[i].inc / 10 + tiles * c[i].rest / cu;
        if (!i || t < least) { best = i; least = t; }
    }
    return best;
}
// Q4_0 and Q8_0 in the host's order.  XT_N4, XT_N2: xn_kernel with four and two slots; XT_1 .. XT_4: xt_kernel with so many groups; XT_MIXED + r: four groups, and r for the last ones
enum { XT_N4, XT_N2, XT_1, XT_2, XT_4, XT_MIXED = 4 };
inline int xt_choose(bool q8, int64_t M, int nmat, int ncg, int64_t cu) {
    // the last one: tiles of four groups and one of what remains, where something remains
    static const int of_rest[4] = {0, 60, 100, 132};
    const int rest = ncg > 4 ? ncg % 4 : 0;
    // Q8_0's first two tiles have room for four workgroups on a compute unit, and its chunks are larger: 4096 x 11008 x 150 100.5 -> 93.1 us, 4096 x 4096 x 150 42.2 -> 39.4,
    // 12288 x 4096 x 180 116 -> 108 with its own increments.
    // The third tile's increment: another workgroup on a compute unit that has 8 to 16 takes 95 .. 96 on the scale of the fourth's 165, in either type; but beyond six the
    // rule counts parts of workgroups, where the third is in truth still rounded up (22016 x 4096 x 128, 10.75 of them: 130.7 us, the line between ten and twelve says 125).  Every tile timed
    // at 322 shapes (4096 .. 32000 x 4096 and 4096 x 11008 by 4 .. 512 rows, both types): the choice is 0.12 % slower than the best tile in the mean with 97 or 98, 0.28 % with 96
    // (fourth against third tile: 22016 x 4096 x 128 Q4_0 124 / 132 us, Q8_0 132 / 145; 11008 x 4096 x 256 Q8_0 127 / 142), 0.49 % with 100 (4096 x 11008 x 100 Q4_0: third tile 73.4, mixed fourth 85.1).
    const xt_cost c[5] = {{16, 1, 44, q8 ? 50 : 44}, {32, 1, 106, q8 ? 64 : 56}, {32, 2, 173, 98}, {32, 4, 288, 165}, {32, 4, 288, 165, of_rest[rest]}};
    const int best = xt_pick(M, nmat, ncg, cu, c, rest ? 5 : 4);
    if (best == 0) return (M + 15) / 16 * nmat * ncg <= 2 * cu ? XT_N4 : XT_N2;
    return best == 4 ? XT_MIXED + rest : XT_1 + best - 1;
}

// Tiles of the K-quants, and of Q4_0 in the own order: times in tenths of a microsecond at K = 4096 with 1, 2, 3, 4 and 6 workgroups per compute unit, weights from memory
struct xk_tile { int rows, groups, t[5]; };
inline int xk_pick(int64_t M, int nmat, int ncg, int64_t cu, const xk_tile *c, int n_tiles) {
    int best = 0;
    int64_t least = 0;
    for (int i = 0; i < n_tiles; i++) {
        const int64_t wgs = (M + c[i].rows - 1) / c[i].rows * nmat * ((ncg + c[i].groups - 1) / c[i].groups), n = (wgs + cu - 1) / cu;
        const int64_t t = n <= 4 ? c[i].t[n - 1] : n == 5 ? (c[i].t[3] + c[i].t[4]) / 2 : c[i].t[4] * wgs / (6 * cu);
        if (!i || t < least) { best = i; least = t; }
    }
    return best;
}
// the K-quants in the host's order: xks_kernel, then xk_kernel with waves of 16 rows by groups 2 x 2, 4 x 2, 4 x 4, 8 x 8
enum { XK_TILES = 5 };
inline int xk_choose(bool q4, int64_t M, int nmat, int ncg, int64_t cu) {
    static const xk_tile k4[5] = {{16, 1, {99, 123, 171, 220, 297}}, {32, 2, {226, 264, 278, 319, 517}}, {64, 2, {273, 302, 407, 557, 899}}, {64, 4, {338, 467, 643, 815, 1176}}, {128, 8, {830, 1414, 2069, 2736, 4053}}},
                         k6[5] = {{16, 1, {113, 160, 207, 269, 364}}, {32, 2, {240, 267, 354, 460, 702}}, {64, 2, {305, 455, 635, 832, 1210}}, {64, 4, {357, 526, 756, 987, 1443}}, {128, 8, {827, 1403, 2101, 2768, 4116}}};
    return xk_pick(M, nmat, ncg, cu, q4 ? k4 : k6, XK_TILES);
}
// in the own order: xks_kernel, then xk_kernel 2 x 2, 4 x 2, 2 x 4, 4 x 4, 4 x 8, and with K over sets of waves 2 x 2 (four sets), 2 x 4 (four), 4 x 4 (two)
enum { XKO_TILES = 9 };
inline int xko_choose(bool q4, int64_t M, int nmat, int ncg, int64_t cu) {
    // The last three split K: where a matrix gives a compute unit one workgroup, the chain of its super-blocks is what it takes (8192 x 4096 x 64: Q4_K
    // 35.6 -> 22.6 us, Q6_K 39.8 -> 25.2; 8192 x 11008 x 100: 104 -> 69 and 126 -> 92); with two and more the tiles without a split are faster.
    static const xk_tile k4[9] = {{16, 1, {99, 123, 171, 219, 298}}, {32, 2, {246, 271, 286, 323, 513}}, {64, 2, {287, 320, 405, 556, 802}}, {32, 4, {303, 382, 421, 482, 902}}, {64, 4, {331, 420, 569, 770, 1071}}, {64, 8, {497, 706, 1082, 1333, 1960}}, {32, 2, {148, 259, 380, 499, 736}}, {32, 4, {186, 340, 498, 654, 964}}, {64, 4, {278, 516, 754, 995, 1466}}},
                         k6[9] = {{16, 1, {113, 160, 206, 269, 364}}, {32, 2, {247, 286, 369, 468, 703}}, {64, 2, {316, 468, 643, 841, 1223}}, {32, 4, {295, 408, 480, 586, 1052}}, {64, 4, {354, 532, 762, 1001, 1447}}, {64, 8, {524, 764, 1159, 1473, 2173}}, {32, 2, {174, 317, 462, 606, 892}}, {32, 4, {211, 394, 579, 758, 1122}}, {64, 4, {344, 639, 930, 1230, 1814}}};
    return xk_pick(M, nmat, ncg, cu, q4 ? k4 : k6, XKO_TILES);
}
// Q4_0 in the own order: xo_kernel, xo32_kernel
inline int xo_choose(int64_t M, int nmat, int ncg, int64_t cu) {
    // tiles of 128 rows by four groups (two of 32 x 32 per wave) were the better ones nowhere: 8192 x 4096 x 500 69.1 us, these two 68.9 and 66.2
    static const xk_tile c[2] = {{64, 4, {342, 383, 515, 650, 949}}, {128, 8, {607, 990, 1472, 1933, 2895}}};
    return xk_pick(M, nmat, ncg, cu, c, 2);
}
