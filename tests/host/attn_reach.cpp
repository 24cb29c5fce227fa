// What xattn_short_kernel asks of the caches before it knows the position, walked with the functions it uses (attn_reach.h) over every thread, length
// and context up to the largest the kernel takes.  Prints "ok", or the first request outside the caches (exit status 1).
#include <cstdio>

#include "../../spy_amd/csrc/attn_reach.h"

int main() {
    const int max_kv = 576, threads = 1024;
    for (int in_state = 0; in_state < 2; in_state++)
        for (int n_ctx = 8; n_ctx <= 1024; n_ctx += 8)
            for (int n_kv = 1; n_kv <= (n_ctx < max_kv ? n_ctx : max_kv); n_kv++) {
                const int cap = n_ctx < max_kv ? n_ctx : max_kv, pos_imm = in_state ? 0 : n_kv - 1;
                const int keys = xf_keys_before(in_state, pos_imm, cap), pieces = xf_row_pieces_before(in_state, pos_imm, n_ctx);
                const int key_end = in_state ? cap : n_kv, row_end = in_state ? n_ctx : (n_kv + 7) / 8 * 8;
                if (!in_state && keys != n_kv) { std::printf("n_kv %d of %d: %d keys\n", n_kv, n_ctx, keys); return 1; }
                for (int c = 0; c < threads; c++)
                    if (const int k = xf_piece(c, keys * 16); k < 0 || (k >> 4) >= key_end) { std::printf("n_kv %d of %d, thread %d: key %d\n", n_kv, n_ctx, c, k >> 4); return 1; }
                for (int lane = 0; lane < 64; lane++)
                    if (const int e = xf_piece(lane, pieces) * 8; e < 0 || e + 8 > row_end) { std::printf("n_kv %d of %d, lane %d: element %d\n", n_kv, n_ctx, lane, e); return 1; }
                for (int c = 0; c < (n_kv < threads / 16 ? n_kv : threads / 16) * 16; c++)             // a cached key's own piece is never exchanged for another
                    if (xf_piece(c, keys * 16) != c) { std::printf("n_kv %d of %d: piece %d\n", n_kv, n_ctx, c); return 1; }
                for (int c = 0; c <= (n_kv - 1) / 8 && c < 64; c++)
                    if (xf_piece(c, pieces) != c) { std::printf("n_kv %d of %d: row piece %d\n", n_kv, n_ctx, c); return 1; }
            }
    std::puts("ok");
    return 0;
}
