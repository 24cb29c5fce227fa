// How far xattn_short_kernel (attn_short.hip) reads into the caches before it knows the position.  Plain C++: a test on the host walks the same functions.
// in_state: the position lies in device memory and is read by the launch itself, so its first requests go out without it, as far as the cache goes (an engine's
// own caches, n_ctx tokens long).  Otherwise it is the number pos_imm, the caches are a caller's, and nothing behind the last token is asked for, but for the
// rest of its 16-byte piece of a V^T row.
#pragma once

// keys (tokens) that may be read; cap: tokens the kernel takes at most
constexpr int xf_keys_before(bool in_state, int pos_imm, int cap) { return in_state ? cap : pos_imm + 1 < cap ? pos_imm + 1 : cap; }
// 16-byte pieces of a V^T row that may be read; n_ctx is a multiple of 8
constexpr int xf_row_pieces_before(bool in_state, int pos_imm, int n_ctx) { return in_state ? n_ctx >> 3 : (pos_imm >> 3) + 1; }
// piece c of `pieces` there are: the last one where c is none of them
constexpr int xf_piece(int c, int pieces) { return c < pieces ? c : pieces - 1; }
