// The tile choice of the MatMuls from packed activations (gemm_tiles.h) for the shapes on standard input: lines of "<which> <first type> <M> <T> <compute units>", which = t (Q4_0 / Q8_0,
// host order; first type: 1 for Q8_0), k (K-quants, host order; 1 for Q4_K), o (K-quants, own order; 1 for Q4_K) or q (Q4_0, own order).  One number per line.
#include <cstdio>

#include "../../spy_amd/csrc/gemm_tiles.h"

int main() {
    char which;
    int flag;
    long long M, T, cu;
    while (std::scanf(" %c %d %lld %lld %lld", &which, &flag, &M, &T, &cu) == 5) {
        const int ncg = (int)((T + 15) / 16);
        std::printf("%d\n", which == 't' ? xt_choose(flag, M, 1, ncg, cu) : which == 'k' ? xk_choose(flag, M, 1, ncg, cu) : which == 'o' ? xko_choose(flag, M, 1, ncg, cu) : xo_choose(M, 1, ncg, cu));
    }
    return 0;
}
