// Main loops of the 256-row-tile MFMA GEMMs, one output tile per 8-wave
// workgroup, operands in HBM as 1 KB tiles in MFMA lane order (16 rows x 64
// bytes of k; hb_lds_ring.h).  Both keep the next fragments' LDS reads and
// the next stages' loads in flight under the multiplications, with one
// workgroup barrier per stage; they differ in how the operands reach the
// registers, which is what bounds a tile:
//  - wide_square: 256 x 256, both operands through an LDS ring, each wave
//    128 x 64 of the tile.  A k-step reads 96 KB from LDS and brings 32 KB in
//    for 1024 cycles of MFMA: the fewest operand bytes per multiplication.
//  - wide_rows: 256 x BN, each wave 32 rows x BN columns, the wave's own
//    activation fragments loaded straight into registers (no other wave needs
//    them) and the weights through an LDS ring shared by the 8 waves.  With
//    activations in LDS too, a 256 x 128 tile moves 88 KB through LDS for 512
//    cycles of MFMA (704 cycles at 128 B per cycle); this way 72 KB, and the
//    cost per column hardly depends on BN, so BN can follow the shape.
// The wave's products are issued with the weights as the first operand: lane
// l of a 16 x 16 block holds row l % 16 and columns 4 * (l / 16) .. + 3.
// Included inside each translation unit's anonymous namespace, after
// hb_lds_ring.h.  The bodies are for the device pass only: the buffer
// resource type does not exist in the host pass.
#ifndef HB_WIDE_TILES_H
#define HB_WIDE_TILES_H

constexpr int kWideWaves = 8;
constexpr int kWideRows = 256;  // rows of a tile

// Tile of workgroup bid, any tile count: workgroups go round-robin over the 8
// XCDs, so each XCD takes one contiguous run of the order that walks groups of
// 4 row blocks column by column (what its L2 then shares).
__device__ inline void xcd_tile(int bid, int tiles_m, int tiles_n, int &tm, int &tn) {
  const int total = tiles_m * tiles_n, each = total / 8, extra = total % 8, xcd = bid % 8;
  group_tile(xcd * each + min(xcd, extra) + bid / 8, tiles_m, tiles_n, tm, tn);
}

// Waits until at most `later` of this wave's stages (PW loads each) issued
// after the awaited one are outstanding, later <= MAX; PW counts the weakest
// wave's loads, so other loads in flight only make the wait longer.
template <int PW, int MAX>
__device__ inline void wait_later(int later) {
  if constexpr (MAX == 0) {
    wait_vmcnt<0>();
  } else {
    if (later >= MAX) wait_vmcnt<MAX * PW>();
    else wait_later<PW, MAX - 1>(later);
  }
}

// A value equal in every lane, kept in a scalar register (a buffer load's
// scalar offset in a vector register becomes a loop over its values).
__device__ inline int wide_uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

// Scalar loads still in flight (kernel arguments) complete out of order, so
// with any pending the compiler can only wait for all LDS reads at once; done
// here, before the loops, it counts the reads.
__device__ inline void wait_scalar_loads() {
#if defined(__HIP_DEVICE_COMPILE__)
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0) alone
#endif
}

// Operands of a tile: a and w point at its first 16-row block of activations
// and 16-column block of weights (blocks of ktc KB), of which ablocks and
// wblocks (from 1 up to the tile's) lie in the image; blocks past them read
// the last one (their sums are never stored).
struct WideOperands {
  const int8_t *a, *w;
  int ablocks, wblocks;
};
__device__ inline WideOperands wide_operands(const int8_t *aimg, int rows, int tile_row, const int8_t *wimg, int cols,
                                             int tile_col, int bn, int ktc) {
  const size_t block = (size_t)ktc * kRingTileBytes;
  return {aimg + (size_t)(tile_row / 16) * block, wimg + (size_t)(tile_col / 16) * block,
          min(kWideRows, rows - tile_row + 15) / 16, min(bn, cols - tile_col) / 16};
}

// acc += rows [wave * FM, + FM) x 16 of the tile times its FN x 16 columns,
// over ktc k-steps.  lds: S stages of 2 * FN KB, one stage = two k-steps of
// weights.  On return every load has landed in this wave, but other waves may
// still read LDS.
//
// Per step of two k-steps: multiply the first, wait for the next stage,
// barrier, issue the loads of a later step, multiply the second.  A wave's
// loads retire in order, so "stage g + 1 has landed" is a count of the loads
// issued after it: S - 3 steps of AL activation and PW weight loads.  The
// prologue issues them in the order that makes that count hold from step 0 on
// (which needs D - 1 >= S - 3 activation steps ahead).
template <class Op, int FM, int FN, int S, int D>
__device__ __attribute__((always_inline)) inline void wide_rows_loop(typename Op::Acc (&acc)[FM][FN], int8_t *lds,
                                                                    const int8_t *a, int ablocks, const int8_t *w,
                                                                    int wblocks, int ktc, int wave, int lane) {
#if defined(__HIP_DEVICE_COMPILE__)
  using Frag = typename Op::Frag;
  constexpr int NB = 2 * FN, PW = (NB + kWideWaves - 1) / kWideWaves, PWL = NB / kWideWaves;
  constexpr int AL = 2 * FM, STAGE = NB * kRingTileBytes, AHEAD = S > D ? S : D;
  static_assert(S >= 4 && D - 1 >= S - 3 && PWL >= 1 && (S - 3) * (AL + PW) < 64, "load counts");
  const uint32_t l16 = (uint32_t)lane * 16u, row_bytes = (uint32_t)ktc * (uint32_t)kRingTileBytes;
  const __amdgpu_buffer_rsrc_t ra =
      __builtin_amdgcn_make_buffer_rsrc((void *)a, 0, (uint32_t)ablocks * row_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t rb =
      __builtin_amdgcn_make_buffer_rsrc((void *)w, 0, (uint32_t)wblocks * row_bytes, 0x00020000);
  const int steps = (ktc + 1) / 2;
  uint32_t soffa[FM], soffb[PW];
  int sub[PW];  // which of the stage's two k-steps a weight block belongs to
#pragma unroll
  for (int i = 0; i < FM; ++i) soffa[i] = (uint32_t)min(wave * FM + i, ablocks - 1) * row_bytes;
#pragma unroll
  for (int i = 0; i < PW; ++i) {
    const int b = min(i * kWideWaves + wave, NB - 1);
    sub[i] = wide_uniform(b / FN);
    soffb[i] = (uint32_t)min(b % FN, wblocks - 1) * row_bytes;
  }
  const bool full = PW == PWL || wave < NB % kWideWaves;  // this wave loads PW blocks of a stage, else PWL
  Frag fa[D][2][FM], fb[2][FN];

#define WIDE_LOAD_A(SET, G, IN)                                                                                         \
  {                                                                                                                  \
    _Pragma("unroll") for (int i = 0; i < FM; ++i) _Pragma("unroll") for (int u = 0; u < 2; ++u) fa[SET][u][i] =     \
        __builtin_bit_cast(Frag, __builtin_amdgcn_raw_buffer_load_b128(                                              \
                                     ra, l16, soffa[i] + (uint32_t)(IN ? 2 * (G) + u : wide_uniform(min(2 * (G) + u, ktc - 1))) * kRingTileBytes, 0)); \
  }
#define WIDE_LOAD_W(SLOT, G, IN)                                                                                        \
  {                                                                                                                  \
    _Pragma("unroll") for (int i = 0; i < PW; ++i) if (i < PWL || full) __builtin_amdgcn_raw_ptr_buffer_load_lds(    \
        rb, HB_LDS_PTR(lds + (SLOT) * STAGE + (i * kWideWaves + wave) * kRingTileBytes), 16, l16,                    \
        soffb[i] + (uint32_t)(IN ? 2 * (G) + sub[i] : wide_uniform(min(2 * (G) + sub[i], ktc - 1))) * kRingTileBytes, 0, 0);        \
  }
#define WIDE_READ_MUL(DST, PTR, SRC, SET, SUB)                                                                       \
  {                                                                                                                  \
    _Pragma("unroll") for (int j = 0; j < FN; ++j) {                                                                 \
      fb[DST][j] = *(const Frag *)((PTR) + j * kRingTileBytes + lane * 16);                                          \
      _Pragma("unroll") for (int i = 0; i < FM; ++i) acc[i][j] = Op::mma(fb[SRC][j], fa[SET][SUB][i], acc[i][j]);    \
    }                                                                                                                \
    _Pragma("unroll") for (int j = 0; j < FN; ++j) {                                                                 \
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0); /* one LDS read, */                                         \
      __builtin_amdgcn_sched_group_barrier(0x8, FM, 0);  /* then FM products */                                      \
    }                                                                                                                \
    __builtin_amdgcn_sched_barrier(0);                                                                               \
  }
#define WIDE_STEP(SET, G, HOT)                                                                                       \
  {                                                                                                                  \
    const int8_t *cur = lds + slot * STAGE;                                                                          \
    if (++slot == S) slot = 0;                                                                                       \
    const int8_t *next = lds + slot * STAGE;                                                                         \
    WIDE_READ_MUL(1, cur + FN * kRingTileBytes, 0, SET, 0)                                                           \
    if (HOT) {                                                                                                       \
      if (full) wait_vmcnt<(S - 3) * (AL + PW)>();                                                                   \
      else wait_vmcnt<(S - 3) * (AL + PWL)>();                                                                       \
    } else {                                                                                                         \
      wait_later<PWL, S - 3>(steps - 2 - (G));                                                                       \
    }                                                                                                                \
    block_barrier(); /* stage G + 1 published; every wave is done with stage G - 1 */                                \
    __builtin_amdgcn_sched_barrier(0);                                                                               \
    if (HOT || (G) + D - 1 < steps) WIDE_LOAD_A(((SET) + D - 1) % D, (G) + D - 1, HOT)                                   \
    if (HOT || (G) + S - 1 < steps) WIDE_LOAD_W(wslot, (G) + S - 1, HOT)                                                 \
    if (++wslot == S) wslot = 0;                                                                                     \
    __builtin_amdgcn_sched_barrier(0);                                                                               \
    if (HOT || 2 * (G) + 1 < ktc) WIDE_READ_MUL(0, next, 1, SET, 1)                                                  \
  }

  // Weights of steps 0 and 1, then activations and weights in turn.  No load
  // here is conditional (past the last step the last k-step is read again,
  // unused): after a branch the compiler counts the loads in flight from the
  // shorter side and would drain the pipeline once per turn of the hot loop.
#pragma unroll
  for (int s = 0; s < S - 1; ++s) {
    if (s >= 2 && s - 2 < D - 1) WIDE_LOAD_A(s - 2, s - 2, false)
    WIDE_LOAD_W(s, s, false)
  }
#pragma unroll
  for (int s = S - 3; s < D - 1; ++s) WIDE_LOAD_A(s, s, false)
  wait_vmcnt<(S - 2) * PWL>();
  block_barrier();
  wait_scalar_loads();
#pragma unroll
  for (int j = 0; j < FN; ++j) fb[0][j] = *(const Frag *)(lds + j * kRingTileBytes + lane * 16);
  int slot = 0, wslot = S - 1, g = 0;
  for (; g + D - 1 + AHEAD - 1 < ktc / 2; g += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) WIDE_STEP(d, g + d, true)
  }
  for (; g < steps; g += D) {
#pragma unroll
    for (int d = 0; d < D; ++d)
      if (g + d < steps) WIDE_STEP(d, g + d, false)
  }
#undef WIDE_STEP
#undef WIDE_READ_MUL
#undef WIDE_LOAD_W
#undef WIDE_LOAD_A
#endif
}

// acc += the 128 x 64 piece (wave / 4, wave % 4) of the 256 x 256 tile, over
// ktc k-steps.
// lds: S stages of 32 KB.  As wide_rows_loop otherwise; 2 of the 8 row blocks
// of a step are multiplied before its barrier, the reads of the next step's
// fragments and this wave's four loads go between the products of the others.
template <class Op, int S>
__device__ __attribute__((always_inline)) inline void wide_square_loop(typename Op::Acc (&acc)[8][4], int8_t *lds,
                                                                      const int8_t *a, int ablocks, const int8_t *w,
                                                                      int wblocks, int ktc, int wave, int lane) {
#if defined(__HIP_DEVICE_COMPILE__)
  using Frag = typename Op::Frag;
  constexpr int FM = 8, FN = 4, PW = 4, FIRST = 2, PHASES = FM - FIRST, READS = FM + FN;
  constexpr int STAGE = 32 * kRingTileBytes;
  static_assert(S >= 4, "at least one stage in flight behind the awaited one");
  const uint32_t l16 = (uint32_t)lane * 16u, row_bytes = (uint32_t)ktc * (uint32_t)kRingTileBytes;
  const __amdgpu_buffer_rsrc_t ra =
      __builtin_amdgcn_make_buffer_rsrc((void *)a, 0, (uint32_t)ablocks * row_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t rb =
      __builtin_amdgcn_make_buffer_rsrc((void *)w, 0, (uint32_t)wblocks * row_bytes, 0x00020000);
  uint32_t soff[PW];  // blocks wave and wave + 8 of each operand
#pragma unroll
  for (int i = 0; i < PW; ++i)
    soff[i] = (uint32_t)(i < 2 ? min(i * 8 + wave, ablocks - 1) : min((i - 2) * 8 + wave, wblocks - 1)) * row_bytes;
  Frag fa[2][FM], fb[2][FN];
  const int aoff = (wave / 4) * FM * kRingTileBytes + lane * 16;
  const int boff = (16 + (wave % 4) * FN) * kRingTileBytes + lane * 16;

#define WIDE_LOAD(I, SLOT, G)                                                                                        \
  __builtin_amdgcn_raw_ptr_buffer_load_lds((I) < 2 ? ra : rb,                                                        \
                                           HB_LDS_PTR(lds + (SLOT) * STAGE + ((I) * 8 + wave) * kRingTileBytes), 16, \
                                           l16, soff[I] + (uint32_t)(G) * kRingTileBytes, 0, 0);
#define WIDE_MUL(P, I)                                                                                               \
  _Pragma("unroll") for (int j = 0; j < FN; ++j) acc[I][j] = Op::mma(fb[P][j], fa[P][I], acc[I][j]);
#define WIDE_STEP(P, G, HOT)                                                                                         \
  {                                                                                                                  \
    _Pragma("unroll") for (int i = 0; i < FIRST; ++i) { WIDE_MUL(P, i) }                                             \
    __builtin_amdgcn_sched_barrier(0);                                                                               \
    if (HOT) wait_vmcnt<(S - 3) * PW>();                                                                             \
    else wait_later<PW, S - 3>(ktc - 2 - (G));                                                                       \
    block_barrier(); /* stage G + 1 published; every wave is done with stage G - 1 */                                \
    __builtin_amdgcn_sched_barrier(0);                                                                               \
    const int8_t *base = lds + rd * STAGE;                                                                           \
    if (++rd == S) rd = 0;                                                                                           \
    const bool more = HOT || (G) + S - 1 < ktc;                                                                      \
    _Pragma("unroll") for (int ph = 0; ph < PHASES; ++ph) {                                                          \
      _Pragma("unroll") for (int q = ph * READS / PHASES; q < (ph + 1) * READS / PHASES; ++q) {                      \
        if (q < FN) fb[1 - (P)][q] = *(const Frag *)(base + boff + q * kRingTileBytes);                              \
        else fa[1 - (P)][q - FN] = *(const Frag *)(base + aoff + (q - FN) * kRingTileBytes);                         \
      }                                                                                                              \
      if (more) {                                                                                                    \
        _Pragma("unroll") for (int q = ph * PW / PHASES; q < (ph + 1) * PW / PHASES; ++q) {                          \
          WIDE_LOAD(q, wr, (G) + S - 1)                                                                              \
        }                                                                                                            \
      }                                                                                                              \
      __builtin_amdgcn_sched_barrier(0);                                                                             \
      WIDE_MUL(P, FIRST + ph)                                                                                        \
      __builtin_amdgcn_sched_barrier(0);                                                                             \
    }                                                                                                                \
    if (++wr == S) wr = 0;                                                                                           \
  }

#pragma unroll
  for (int s = 0; s < S - 1; ++s) {
#pragma unroll
    for (int i = 0; i < PW; ++i) { WIDE_LOAD(i, s, wide_uniform(min(s, ktc - 1))) }
  }
  wait_vmcnt<(S - 2) * PW>();
  block_barrier();
  wait_scalar_loads();
#pragma unroll
  for (int i = 0; i < FM; ++i) fa[0][i] = *(const Frag *)(lds + aoff + i * kRingTileBytes);
#pragma unroll
  for (int j = 0; j < FN; ++j) fb[0][j] = *(const Frag *)(lds + boff + j * kRingTileBytes);
  int rd = 1, wr = S - 1, g = 0;
  for (; g + S < ktc; g += 2) {
    WIDE_STEP(0, g, true)
    WIDE_STEP(1, g + 1, true)
  }
  for (; g < ktc; g += 2) {
    WIDE_STEP(0, g, false)
    if (g + 1 < ktc) WIDE_STEP(1, g + 1, false)
  }
#undef WIDE_STEP
#undef WIDE_MUL
#undef WIDE_LOAD
#endif
}

#endif  // HB_WIDE_TILES_H
