// Which parts of the caches the attention kernels of one token read.  Plain C++: a test on the host walks the same functions.
#pragma once

// How far xattn_short_kernel (attn_short.hip) reads before it knows the position.
// in_state: the position lies in device memory and is read by the launch itself, so its first requests go out without it, as far as the cache goes (an engine's
// own caches, n_ctx tokens long).  Otherwise it is the number pos_imm, the caches are a caller's, and nothing behind the last token is asked for, but for the
// rest of its 16-byte piece of a V^T row.
// keys (tokens) that may be read; cap: tokens the kernel takes at most
constexpr int xf_keys_before(bool in_state, int pos_imm, int cap) { return in_state ? cap : pos_imm + 1 < cap ? pos_imm + 1 : cap; }
// 16-byte pieces of a V^T row that may be read; n_ctx is a multiple of 8
constexpr int xf_row_pieces_before(bool in_state, int pos_imm, int n_ctx) { return in_state ? n_ctx >> 3 : (pos_imm >> 3) + 1; }
// piece c of `pieces` there are: the last one where c is none of them
constexpr int xf_piece(int c, int pieces) { return c < pieces ? c : pieces - 1; }

// Which keys xattn_scores_kernel (exact_decode.cuh) reads.  Head group g of eight has heads g, g + 8, ...; a unit of a wave is 16 keys: one, two or four heads (as many as the largest
// group has, four at most with 32 heads) of 16, 8 or 4 tokens.
constexpr int xs_log2(int n_head) { return n_head > 16 ? 2 : n_head > 8 ? 1 : 0; }                                // log2 of the heads of a unit
constexpr int xs_head(int n_head, int g, int slot) { return g + 8 * slot < n_head ? g + 8 * slot : g; }           // head of place `slot` in a unit: the group's first where it has none
// tokens of a workgroup where nb share n_kv, a multiple of the nt of a unit
constexpr int xs_share(int n_kv, int nb, int nt) { return ((n_kv + nb - 1) / nb + nt - 1) & -nt; }
