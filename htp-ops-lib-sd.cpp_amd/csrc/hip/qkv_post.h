// Packed Q / K / V post-processing of the fused QKV opcodes (8/10/11/12),
// shared by the standalone kernel (qkv.hip) and the GEMM with the
// post-processing in its epilogue (f16.hip).
//
// Semantics (reference src/dsp/ops/mat_mul.c): the GEMM output is the HMX
// fp16 readout (:1297-1330, transfer_output_chunk_fp16_to_fp32 :751-778), so
// its f32 values are fp16-exact.  Per 32-token tile and head:
//   Q, K  v = x + bias; sum of squares in the order of the 32-lane vector code
//         (lane j: v[64d+j]^2 then v[64d+32+j]^2 over the 64-column chunks d,
//         then the shifted lane adds of qkv_reduce_sum :1127-1135);
//         inv = rsqrt(sum/hd + 1e-6) by three Newton steps from 0x5f3759df
//         (:1137-1165); y = (v*inv)*gamma (:1167-1208); then the rotary
//         matrices of the token (:1210-1231) while token < rope_count;
//   V     y = x + bias (:1249-1266);
// each value rounded once to fp16 and placed in the packed layouts:
//   Q  row pairs interleaved per 32-column tile, tiles [token tile][column tile]
//      (:1051-1072);
//   K  per 64-column chunk of token r, word w (columns 2w, 2w+1) at byte
//      128w + 4r of the chunk's two tiles (the vscatter of :1078-1101);
//   V  row pairs interleaved per 32-column tile, tiles [column tile][token tile]
//      (:1103-1125, :1359-1369).
// Rows past the call's tokens inside its last tile are zeros.  Every float
// step is one IEEE binary32 operation (the reference computes them in QFloat).
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>

#include <cstdint>

#include "qkv_rope.h"

namespace {

constexpr int kQkvThreads = 256;  // 4 waves; a wave takes two rows at a time (one per 32 lanes)

__device__ inline float qkv_rsqrt(float x) {
  const float half = __fmul_rn(x, 0.5f);
  float y = __uint_as_float(0x5f3759dfu - (__float_as_uint(x) >> 1));
#pragma unroll
  for (int it = 0; it < 3; ++it) {
    const float y2 = __fmul_rn(y, y);
    const float corr = __fsub_rn(1.5f, __fmul_rn(half, y2));
    y = __fmul_rn(y, corr);
  }
  return y;
}

// LDS index of (row r, column c) inside one (token tile, head) block, in the
// order of the destination: Q and K blocks are contiguous, V's column tiles
// are copied to their own places.
template <int WHICH>
__device__ inline int block_index(int r, int c) {
  const int pair = (r >> 1) * 64 + (c & 31) * 2 + (r & 1);
  if (WHICH == 1) return (c >> 6) * 2048 + ((c & 63) >> 1) * 64 + r * 2 + (c & 1);
  return (c >> 5) * 1024 + pair;
}

// One workgroup per (32-token tile, head) of one of Q / K / V (WHICH 0 / 1 / 2).
// Every load of the tile (rows, bias, gamma, rotary matrices) is issued
// before the arithmetic: one round of 4 row pairs per wave keeps enough
// bytes in flight to stream from HBM.
// src: row 0, column 0 of the head's input (rows src_stride elements apart);
// bias: the head's first column (NULL: none); rows: valid rows (1..32);
// token0: the call's token index of row 0; tokens below rope_rows (at most the
// call's tokens) are rotated, token t by row rope_off + t of pe;
// blk: HD * 32 halfwords of LDS, 16-byte aligned, for the packed block, which
// goes to dst + head_base.
template <int HD, int WHICH>
__device__ void qkv_block(uint16_t *__restrict__ blk, uint16_t *__restrict__ dst, const float *__restrict__ src,
                          int src_stride, const float *__restrict__ bias, const float *__restrict__ gamma,
                          const float *__restrict__ pe, int rope_off, int rope_rows, int rows, int token0, int tt,
                          int token_tiles, size_t head_base) {
  constexpr int CH = HD / 64;  // 64-column chunks; lane j holds columns 64d+j and 64d+32+j
  constexpr int E = 2 * CH;    // values per lane and row
  constexpr int PAIRS = 16 / (kQkvThreads / 64);
  constexpr bool ROPE_OK = WHICH < 2;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int half = lane >> 5, j = lane & 31;
  auto col = [&](int e) { return 64 * (e >> 1) + 32 * (e & 1) + j; };

  float v[PAIRS][E];
#pragma unroll
  for (int i = 0; i < PAIRS; ++i) {
    const int r = 2 * (wave + 4 * i) + half;
    const float *x = src + (size_t)r * (size_t)src_stride;
#pragma unroll
    for (int e = 0; e < E; ++e) v[i][e] = r < rows ? x[col(e)] : 0.0f;
  }
  float b[E], g[E];
#pragma unroll
  for (int e = 0; e < E; ++e) {
    b[e] = bias ? bias[col(e)] : 0.0f;
    g[e] = WHICH < 2 ? gamma[col(e)] : 0.0f;
  }
  // rotary matrices (x0, x1 -> m.x x0 + m.y x1, m.z x0 + m.w x1) of each row's token
  float4 m[ROPE_OK ? PAIRS : 1][ROPE_OK ? E : 1];
  bool rot[PAIRS];
#pragma unroll
  for (int i = 0; i < PAIRS; ++i) {
    const int t = token0 + 2 * (wave + 4 * i) + half;
    rot[i] = ROPE_OK && t < rope_rows;
    if (ROPE_OK) {
#pragma unroll
      for (int e = 0; e < E; ++e)
        m[i][e] = rot[i] ? *(const float4 *)(pe + ((size_t)(rope_off + t) * (HD / 2) + (size_t)(col(e) >> 1)) * 4u)
                         : make_float4(0.f, 0.f, 0.f, 0.f);
    }
  }

#pragma unroll
  for (int i = 0; i < PAIRS; ++i) {
    const int r = 2 * (wave + 4 * i) + half;
#pragma unroll
    for (int e = 0; e < E; ++e) v[i][e] = __fadd_rn(v[i][e], b[e]);
    if (WHICH < 2) {
      float acc = 0.0f;
#pragma unroll
      for (int e = 0; e < E; ++e) acc = __fadd_rn(acc, __fmul_rn(v[i][e], v[i][e]));
      // lane i += lane i - s within the 32 lanes of the row, s = 16 .. 1
#pragma unroll
      for (int s = 16; s >= 1; s >>= 1) {
        const float o = __shfl(acc, (lane - s) & 63, 64);
        if (j >= s) acc = __fadd_rn(acc, o);
      }
      const float sum = __shfl(acc, half * 32 + 31, 64);
      const float inv = qkv_rsqrt(__fadd_rn(__fdiv_rn(sum, (float)HD), 1.0e-6f));
#pragma unroll
      for (int e = 0; e < E; ++e) v[i][e] = __fmul_rn(__fmul_rn(v[i][e], inv), g[e]);
      if (rope_rows > 0) {
        // the pair of column c is c ^ 1, held by lane j ^ 1
#pragma unroll
        for (int e = 0; e < E; ++e) {
          const float other = __shfl(v[i][e], lane ^ 1, 64);
          if (rot[i]) {
            const bool odd = j & 1;
            const float x0 = odd ? other : v[i][e], x1 = odd ? v[i][e] : other;
            const float4 mm = m[i][ROPE_OK ? e : 0];
            v[i][e] = odd ? __fadd_rn(__fmul_rn(x0, mm.z), __fmul_rn(x1, mm.w))
                          : __fadd_rn(__fmul_rn(x0, mm.x), __fmul_rn(x1, mm.y));
          }
        }
      }
    }
#pragma unroll
    for (int e = 0; e < E; ++e)
      blk[block_index<WHICH>(r, col(e))] = r < rows ? __half_as_ushort(__float2half_rn(v[i][e])) : (uint16_t)0;
  }
  __syncthreads();
  const uint4 *packed = (const uint4 *)blk;
  uint16_t *hdst = dst + head_base;
  if (WHICH < 2) {
    uint4 *out = (uint4 *)(hdst + (size_t)tt * HD * 32);
    for (int i = threadIdx.x; i < HD * 32 / 8; i += kQkvThreads) out[i] = packed[i];
  } else {
    for (int i = threadIdx.x; i < HD * 32 / 8; i += kQkvThreads) {
      const int ct = i / 128;  // 1024 halfwords = 128 uint4 per column tile
      uint4 *out = (uint4 *)(hdst + ((size_t)ct * token_tiles + tt) * 1024);
      out[i % 128] = packed[i];
    }
  }
}

// ---------------------------------------------------------------------------
// The same post-processing on a GEMM wave's registers: FN 16-column blocks
// (FN / (HD / 16) whole heads) of a 32-row token tile, block (i, j) holding
// rows 16 i + lane % 16 and columns 16 j + 4 * (lane / 16) .. + 3 of the tile
// as fp32 sums.  A row of a head is spread over the 4 lanes that differ in
// lane / 16, so the sum of squares needs two cross-lane adds (its order is the
// one above: column c belongs to vector lane c % 32, so the adds of lanes 16
// and 8, 4 apart are between blocks j, j + 1 and between lane groups); rotary
// pairs are neighbours in a lane; and a token row pair (Q, V) or a column pair
// (K) makes one 32-bit word of the packed layout, stored without passing
// through LDS.
// ---------------------------------------------------------------------------

// The other row of this lane's row pair (lane ^ 1), by DPP quad permutation.
__device__ inline uint32_t qkv_pair_lane(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1 /* quad_perm 1,0,3,2 */, 0xf, 0xf, true);
}

// Row block i of head h of the wave's blocks; rows: valid rows of the token
// tile (others are stored as zeros); base: the head's packed region; rot and
// m: whether this lane's row is rotated, and its rotary matrices for the
// lane's column pairs (8 j + 2 * (lane / 16) + q).
template <int HD, int WHICH, int FN>
__device__ __attribute__((always_inline)) inline void qkv_rows_head(hb_f32x4 (&acc)[2][FN], int i, int h,
                                                                    uint16_t *base, int tt, int token_tiles,
                                                                    const float *bias, const float *gamma, bool rot,
                                                                    const hb_f32x4 (&m)[HD / 16][2], int rows,
                                                                    int lane) {
  typedef float f32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
  constexpr int FH = HD / 16;
  const int g = lane >> 4, r16 = lane & 15;
  float v[FH][4];
#pragma unroll
  for (int j = 0; j < FH; ++j) {
    const hb_f32x4 b = bias ? (hb_f32x4)(*(const f32x4_a4 *)(bias + h * HD + 16 * j + 4 * g)) : hb_f32x4{0, 0, 0, 0};
#pragma unroll
    for (int e = 0; e < 4; ++e) v[j][e] = __fadd_rn((float)(_Float16)acc[i][h * FH + j][e], b[e]);
  }
  if (WHICH < 2) {
    float w[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float p[2];  // vector lanes 4 g + e and 16 + 4 g + e: columns 32 apart, in order
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        p[q] = 0.0f;
#pragma unroll
        for (int j = q; j < FH; j += 2) p[q] = __fadd_rn(p[q], __fmul_rn(v[j][e], v[j][e]));
      }
      w[e] = __fadd_rn(p[1], p[0]);                      // 16 apart
      w[e] = __fadd_rn(w[e], __shfl_xor(w[e], 32, 64));  // 8 apart
      w[e] = __fadd_rn(w[e], __shfl_xor(w[e], 16, 64));  // 4 apart
    }
    const float sum = __fadd_rn(__fadd_rn(w[3], w[1]), __fadd_rn(w[2], w[0]));
    const float inv = qkv_rsqrt(__fadd_rn(__fdiv_rn(sum, (float)HD), 1.0e-6f));
#pragma unroll
    for (int j = 0; j < FH; ++j) {
      const hb_f32x4 gm = *(const f32x4_a4 *)(gamma + 16 * j + 4 * g);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[j][e] = __fmul_rn(__fmul_rn(v[j][e], inv), gm[e]);
    }
    if (rot) {
#pragma unroll
      for (int j = 0; j < FH; ++j)
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const float x0 = v[j][2 * q], x1 = v[j][2 * q + 1];
          v[j][2 * q] = __fadd_rn(__fmul_rn(x0, m[j][q][0]), __fmul_rn(x1, m[j][q][1]));
          v[j][2 * q + 1] = __fadd_rn(__fmul_rn(x0, m[j][q][2]), __fmul_rn(x1, m[j][q][3]));
        }
    }
  }
  const int r = 16 * i + r16;
  const bool valid = r < rows;
  uint32_t *words = (uint32_t *)base;
#pragma unroll
  for (int j = 0; j < FH; ++j) {
    uint32_t c01 = 0, c23 = 0;  // this row's columns 0, 1 and 2, 3 of the block's four
    if (valid) {
      c01 = (uint32_t)__half_as_ushort(__float2half_rn(v[j][0])) |
            (uint32_t)__half_as_ushort(__float2half_rn(v[j][1])) << 16;
      c23 = (uint32_t)__half_as_ushort(__float2half_rn(v[j][2])) |
            (uint32_t)__half_as_ushort(__float2half_rn(v[j][3])) << 16;
    }
    const int c = 16 * j + 4 * g;  // the lane's first column in the head
    if (WHICH == 1) {
      uint32_t *dst = words + (size_t)tt * (HD * 16) + (c >> 6) * 1024 + ((c & 63) >> 1) * 32 + r;
      dst[0] = c01;
      dst[32] = c23;
    } else {
      // the even row's lane takes columns 0, 1 of both rows, the odd row's 2, 3
      const bool odd = lane & 1;
      const uint32_t other = qkv_pair_lane(odd ? c01 : c23);
      const uint32_t lo = odd ? other : c01, hi = odd ? c23 : other;  // even row, odd row
      const uint2 out = make_uint2((lo & 0xffffu) | (hi << 16), (lo >> 16) | (hi & 0xffff0000u));
      const int cc = (c & 31) + (odd ? 2 : 0);
      const size_t tile = WHICH == 0 ? (size_t)tt * (HD / 32) + (size_t)(c >> 5)
                                     : (size_t)(c >> 5) * (size_t)token_tiles + (size_t)tt;
      *(uint2 *)(words + tile * 512 + (r >> 1) * 32 + cc) = out;
    }
  }
}

}  // namespace
