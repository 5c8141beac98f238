// Which attention kernels the distance between rows allows.  Plain host C++, so that a test can compile it by itself.
//
// The hand-scheduled kernels fetch a tile's rows through one buffer descriptor whose byte offsets and length are 32-bit:
// a row past 2^32 - 1 bytes from the tile's first would wrap, or read as zero.  Rows farther apart take the kernels
// that are staged through registers, whose addresses are 64-bit throughout.  The rule looks at strides alone, not at which
// rows a batch has: the offsets of rows past its end must not wrap into it either.  No ordinary packing comes near it (a 64-row
// tile reaches as long as a token's row is under 65 MiB).
#pragma once

namespace fgrpo {

// `rows` rows of D bf16, `stride` > 0 elements apart (no products of the stride: it may be anything)
inline bool attn_rows_in_reach(long long stride, int rows, int D) { return stride <= ((1LL << 32) - 1 - 2 * D) / (2 * (rows - 1)); }

// What the forward / dQ call takes of `wanted` (Tuning::attn_qside): a wavefront reads 32 rows of Q, O and dO, a step 64 of K and V
inline int attn_query_form(int wanted, long long q_st, long long k_st, long long v_st, int Hq, int D) {
  const bool near = attn_rows_in_reach(q_st, 32, D) && attn_rows_in_reach((long long)Hq * D, 32, D) &&
                    attn_rows_in_reach(k_st, 64, D) && attn_rows_in_reach(v_st, 64, D);
  return near ? wanted : 1;
}

// ... and dK/dV of `wanted` (Tuning::attn_dkv).  3: a work-group takes `keys` rows of K and V at once, an item 32 of Q and dO, and the
// offsets of its per-query scalars, (queries x heads of a group) x 4 bytes, and of the bounds arrays are signed 32-bit.
// 2: 64 rows of Q and dO a tile, its own K or V row by 64-bit address.  1: 64-bit throughout.
inline int attn_key_form(int wanted, long long q_st, long long k_st, long long v_st, int T, int Hq, int Hkv, int D, int keys) {
  const long long o_st = (long long)Hq * D;
  if (wanted != 1 && wanted != 2 && (long long)T * (Hq / Hkv) * 4 < (1LL << 31) && (long long)T * 8 < (1LL << 31) &&
      attn_rows_in_reach(q_st, 32, D) && attn_rows_in_reach(o_st, 32, D) && attn_rows_in_reach(k_st, keys, D) && attn_rows_in_reach(v_st, keys, D))
    return 3;
  return wanted != 1 && attn_rows_in_reach(q_st, 64, D) && attn_rows_in_reach(o_st, 64, D) ? 2 : 1;
}

}  // namespace fgrpo
