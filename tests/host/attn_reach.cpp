// What the attention kernels of one token ask of the caches, walked with the functions they use (attn_reach.h): xattn_short_kernel before it knows the position, over every
// thread, length and context up to the largest the kernel takes; xattn_scores_kernel over every number of heads.  Prints "ok", or the first request that is not as it should be (exit status 1).
#include <cstdio>
#include <vector>

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
    // every key of every head once, by a workgroup of its head's group; nothing else is read but a key of the group's own
    for (int n_head = 1; n_head <= 32; n_head++)
        for (int nb : {1, 2, 13, 32})
            for (int n_kv : {1, 3, 16, 17, 300, 577, 1900, 4736}) {
                std::vector<int> seen((size_t)n_head * n_kv);
                for (int b = 0; b < 8 * nb; b++) {
                    const int g = b & 7, tb = b >> 3;
                    if (g >= n_head) continue;
                    const int nh = (n_head - g + 7) / 8, hs = xs_log2(n_head), nt = 16 >> hs;
                    if (nh > 1 << hs) { std::printf("%d heads, group %d: %d heads in units of %d\n", n_head, g, nh, 1 << hs); return 1; }
                    const int tpw = xs_share(n_kv, nb, nt);
                    for (int t = tb * tpw; t < n_kv && t < (tb + 1) * tpw; t += nt)
                        for (int key = 0; key < 16; key++) {
                            const int slot = key & ((1 << hs) - 1), h = xs_head(n_head, g, slot), tt = t + (key >> hs);
                            if (h % 8 != g || h >= n_head) { std::printf("%d heads, group %d: reads head %d\n", n_head, g, h); return 1; }
                            if (slot < nh && tt < n_kv && tt < (tb + 1) * tpw) seen[(size_t)h * n_kv + tt]++;
                        }
                }
                for (int s : seen) if (s != 1) { std::printf("%d heads, %d tokens, %d workgroups a group: a key %d times\n", n_head, n_kv, nb, s); return 1; }
            }
    std::puts("ok");
    return 0;
}
