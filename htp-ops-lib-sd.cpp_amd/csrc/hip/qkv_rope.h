// Which rows of a rotary table a QKV call reads: token t of the call (t from 0)
// is rotated by row offset + t of the table while offset + t < count.  Plain
// C++ besides the kernels' own qualifiers, so that a host program can walk it.
#pragma once

#include <cstdint>

#if defined(__HIPCC__)
#define QKV_ROPE_FN __host__ __device__ inline
#else
#define QKV_ROPE_FN inline
#endif

// The rotated tokens: 0 .. n - 1, n the result (0: none).  offset >= 0.
QKV_ROPE_FN int qkv_rope_rows(int offset, int count, int tokens) {
  const int64_t left = (int64_t)count - offset;
  return left <= 0 ? 0 : left < tokens ? (int)left : tokens;
}

// The row that token t reads, n > 0: its own where t < n, else the last
// rotated token's.  A kernel that loads for whole tiles of tokens so stays
// within the rows that the call rotates, the only ones the table must hold.
QKV_ROPE_FN int qkv_rope_row(int offset, int n, int t) { return offset + (t < n ? t : n - 1); }
