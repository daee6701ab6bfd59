// fk_skinny.h — the GEMM of a step of few rows: C = A · Bᵀ where the tiles of
// fk_gemm.h (256 × 256, one a threadgroup) would leave most of the chip idle.
//
// A step of 8 to 2,000 live rows has 8 to 200 such tiles for 256 CUs, and a
// threadgroup walks the whole of k alone: 46 µs for the QKV projection of 8
// rows, 151 µs for the down projection, where their weights stream from HBM
// in 3 and 6.  Here the k of a tile is split among the wavefronts of its
// threadgroup, so tiles can be small enough to fill the chip and every
// wavefront still has its own loads in flight:
//
// - wavefront w of W takes the steps of 32 columns w, w + W, ... of a tile of
//   MB × NB blocks of 16 × 16, by v_mfma_f32_16x16x32_f16.  Nothing is shared
//   between wavefronts in the loop: a block's operand is one 1 KB chunk of
//   the tile layout (fk_layout.h), loaded straight into the wavefront's own
//   ring of D steps in LDS and read from there as the matrix operation takes
//   it; no barrier.  (Loaded straight into registers instead, 16 lanes of a
//   load on 16 rows 64 bytes apart, the L1 looks 4 lines up where it could
//   look up one: the down projection of 16 rows took 14.6 µs against 13.0,
//   of 704 rows 54 against 44.)
// - The W partial sums meet in LDS, added in the order of the wavefronts, and
//   each wavefront finishes its share of the blocks (the epilogues of
//   fk_gemm.h).
//
// What bounds it: up to 16 live rows the weights' stream from HBM (gate and
// up, 67 MB, in 13.6 µs: 4.9 TB/s; the logits, 131 MB, in 25.5: 5.1) or, of
// fewer than 256 tiles, what one CU draws through its L1 (about 75 GB/s: the
// down projection's 128 tiles read 512 KB each); from 64 rows on the operands'
// reads through the L1s (a tile reads (MB + NB) KB for MB · NB matrix
// operations), which is why tiles grow with the rows.  Measured on MI355X, f16,
// each launch on weights of its own out of HBM, µs, the forms that
// prefill.py's skinny_form picks (fk_gemm's tiles in brackets):
//
//   live rows            16          64         112         208         704        1408
//   QKV  3072 x 2048    7.6 [49]    9.0 [49]  11.3 [49]   11.2 [49]   23.4 [51]   38.7 [57]
//   O    2048 x 2048    5.9 [50]    6.8 [50]   6.5 [50]    8.2 [50]   16.3 [55]   25.6 [55]
//   gate/up 2 x 8192   13.6 [45]   17.7 [45]  21.1 [44]   30.3 [44]    -  [51]     -  [98]
//   down 2048 x 8192   12.9 [160] 15.9 [160]  16.9 [161]  21.7 [161]  46.9 [160]  64.4 [160]
//   head 32000 x 2048  25.5 [62]   36.6 [56]  42.7 [57]     -  [57]    -  [125]    -  [200]
//
// The forms (MB, NB, W, D) and where each is taken: prefill.py's skinny_form.
//
// FK_GEMM_PART splits k among threadgroups too, for the residual projections
// of up to 200 rows, whose tiles are too few to fill the chip: partial sums
// that the norm after them adds (fk_rows_norm.h).
//
// Live rows: the rows that fill a step out to whole tiles (prefill.py) are
// skipped.  Chunk c of the live rows is rows first + i · apart (i = 0 .. 15),
// first = (c / run_chunks) · run + (c mod run_chunks) · 16 · apart: the
// leading rows of each run of a prefill (apart 1), or a decode step's rows,
// one a query block (apart 32, one run; the tiled matrices between its
// kernels then hold the live chunks alone, `compact`: read at their spaced
// rows, 64 bytes each, the down projection of 41 rows took 20 µs against
// 15.5).  A chunk's rows past g.m read zeros and store nothing.
#pragma once

#include "fk_common.h"
#include "fk_gemm.h"
#include "fk_layout.h"
#include "fk_mfma.h"

// MODE: an epilogue of fk_gemm.h.  Blocks per unit of the epilogue: what one
// lane needs of several blocks at once (gate and up; a head's pairs of RoPE).
template <uint32_t MODE, int NB>
struct fk_skinny_unit {
  static constexpr bool PAIRS =
      MODE == FK_GEMM_SILU_MUL || MODE == FK_GEMM_QKV_ROPE || MODE == FK_GEMM_QKV_ROPE_PAGED;
  static constexpr int BLOCKS = PAIRS ? 2 : (MODE == FK_GEMM_STORE_KEYS ? NB : 1);
};

template <uint32_t MODE, int MB, int NB, int W, int D>
__device__ __forceinline__ void skinny_tile(const _Float16 *__restrict__ a, const _Float16 *__restrict__ b0,
                                            const _Float16 *__restrict__ b1, const _Float16 *__restrict__ b2,
                                            void *__restrict__ c0, void *__restrict__ c1, void *__restrict__ c2,
                                            const float *r0, const uint32_t *__restrict__ position,
                                            const uint32_t *__restrict__ slot, const float *__restrict__ rope,
                                            uint64_t *__restrict__ keys, const fk_skinny_params &p) {
  constexpr int U = fk_skinny_unit<MODE, NB>::BLOCKS;
  constexpr bool QKV = MODE == FK_GEMM_QKV_ROPE || MODE == FK_GEMM_QKV_ROPE_PAGED;
  constexpr int NU = NB / U;                       // units a row of blocks
  // Row blocks summed at a time: as many as 128 KB of LDS hold.
  constexpr int MR = MB * NB * W > 128 ? 128 / (NB * W) : MB;
  static_assert(MR >= 1 && MB % MR == 0, "the partial sums of a row of blocks must fit LDS");
  constexpr int CH = MB + NB;                      // chunks (1 KB) a step
  constexpr int RING = W * D * CH * FK_WAVE, SUMS = W * MR * NB * FK_WAVE;
  static_assert(D * CH < 64, "the vector memory counter's range");
  // Every wavefront's ring of D steps; after the loop the partial sums.
  __shared__ uint4 lds[RING > SUMS ? RING : SUMS];
  fk_float4v(*const sums)[MR * NB][FK_WAVE] = reinterpret_cast<fk_float4v(*)[MR * NB][FK_WAVE]>(lds);
  const uint32_t lane = threadIdx.x & (FK_WAVE - 1);
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / FK_WAVE);
  const uint32_t k = p.g.k;
  const uint32_t steps = k / 32;

  // Threadgroups go to the 8 XCDs in turn: the tiles of the same weights (one
  // tile of columns, every tile of rows) follow each other on one XCD, so its
  // L2 fetches them once.
  const uint32_t tiles_m = (p.live + MB - 1) / MB;
  const uint32_t cols = MODE == FK_GEMM_SILU_MUL ? 2 * p.g.ldc[0] : p.g.first_col[p.g.n_anchors];
  const uint32_t tiles_n = cols / (16 * NB);
  const uint32_t at = blockIdx.x / 8;
  const uint32_t tm = at % tiles_m;
  // (FK_GEMM_PART: the parts of a tile follow its tiles of rows)
  const uint32_t parts = MODE == FK_GEMM_PART ? p.parts : 1u;
  const uint32_t part = MODE == FK_GEMM_PART ? at / tiles_m % parts : 0u;
  const uint32_t tn = (at / (tiles_m * parts)) * 8 + blockIdx.x % 8;
  if (tn >= tiles_n) return;

  // The weights' chunks (16 rows) of the tile's column blocks, one 256-row
  // slab: consecutive, but for SiLU·mul gate's then the same of up's (128
  // rows on), and for two blocks of a QKV head its columns d and d + 32.
  uint32_t anchor = 0, n0;
  const _Float16 *b;
  uint32_t slab, chunk0;
  if constexpr (MODE == FK_GEMM_SILU_MUL) {
    n0 = tn * (NB / 2) * 16;
    b = b0;
    slab = n0 / 128;
    chunk0 = (n0 % 128) / 16;
  } else {
    uint32_t col = tn * NB * 16;
    if constexpr (QKV && NB == 2) col = tn / 2 * 64;  // the head's
    anchor = (p.g.n_anchors > 1 && col >= p.g.first_col[1] ? 1u : 0u) +
             (p.g.n_anchors > 2 && col >= p.g.first_col[2] ? 1u : 0u);
    n0 = col - (anchor == 0 ? p.g.first_col[0] : (anchor == 1 ? p.g.first_col[1] : p.g.first_col[2]));
    if constexpr (QKV && NB == 2) n0 += tn % 2 * 16;
    b = anchor == 0 ? b0 : (anchor == 1 ? b1 : b2);
    slab = n0 / 256;
    chunk0 = (n0 % 256) / 16;
  }
  // Block j's chunk, from chunk0.
  auto chunk_of = [](int j) -> uint32_t {
    if constexpr (MODE == FK_GEMM_SILU_MUL) return j < NB / 2 ? j : 8 + j - NB / 2;
    else if constexpr (QKV && NB == 2) return 2 * j;
    else return j;
  };

  // Direct loads: lane L's 16 bytes land at unit L of the staged chunk, row
  // L div 4, the logical unit (L mod 4) ^ swizzle(row).  A weight chunk is
  // staged as it lies; so is a chunk of 16 consecutive rows.
  const auto bsrc = fk::buffer(b + (size_t)slab * 256 * k, (size_t)256 * k * 2);
  const auto asrc = fk::buffer(a, (size_t)p.g.m * k * 2);
  const uint32_t bv = chunk0 * 1024 + lane * 16;
  auto row_of = [&](int i, uint32_t r) -> uint32_t {  // row r of the tile's row chunk i
    const uint32_t c = tm * MB + i;
    return c < p.live ? (c / p.run_chunks) * p.run + ((c % p.run_chunks) * 16 + r) * p.apart : 0xffffffffu;
  };
  uint32_t av[MB];
#pragma unroll
  for (int i = 0; i < MB; i++) {
    // past the rows: past the buffer, where loads read zeros
    const uint32_t c = tm * MB + i;
    const uint32_t row = p.compact ? (c < p.live ? c * 16 + lane / 4 : 0xffffffffu) : row_of(i, lane / 4);
    const uint32_t rr = row % 16;
    av[i] = row < p.g.m ? (row / 256) * (256 * k * 2) + (row % 256 / 16) * 1024 +
                              (rr * 4 + ((lane % 4) ^ fk::tile_swizzle(lane / 4) ^ fk::tile_swizzle(rr))) * 16
                        : 0xfffffff0u;
  }
  // Fragment reads: lane l takes row l mod 16, logical unit l div 16.
  const uint32_t fu = wave * D * CH * FK_WAVE + (lane % 16) * 4 + ((lane / 16) ^ fk::tile_swizzle(lane % 16));
  FK_LDS char *const ring = (FK_LDS char *)lds + wave * (D * CH * 1024);

  // The epilogue's units: a row of blocks has NU, a round of MR rows of blocks
  // UNITS, of which this wavefront takes wave, wave + W, ...: IT a round.
  constexpr int UNITS = MR * NU, IT = (UNITS + W - 1) / W, ROUNDS = MB / MR;
  auto unit_row = [&](int round, int it, uint32_t l) -> uint32_t {  // past the rows for a unit past the last
    const uint32_t u = wave + it * W;
    return u < (uint32_t)UNITS ? row_of(round * MR + u / NU, l % 16) : 0xffffffffu;
  };
  // What the units' rows are stored by is loaded here, and what they are
  // combined with after the loop, all at once: loaded at its unit's turn,
  // each would cost the unit a round trip (O of 1408 rows, 16 units a
  // wavefront: 41 µs a launch in the step, now 26).
  uint32_t upos[QKV ? ROUNDS : 1][QKV ? IT : 1], uslot[QKV ? ROUNDS : 1][QKV ? IT : 1];
  if constexpr (QKV) {
#pragma unroll
    for (int round = 0; round < ROUNDS; round++)
#pragma unroll
      for (int it = 0; it < IT; it++) {
        const uint32_t row = min(unit_row(round, it, lane), p.g.m - 1);
        upos[round][it] = position[row];
        uslot[round][it] = MODE == FK_GEMM_QKV_ROPE && !p.r.staged && anchor != 0 ? slot[row] : 0u;
      }
  }

  fk_float4v acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; i++)
#pragma unroll
    for (int j = 0; j < NB; j++) acc[i][j] = fk_float4v{0.0f, 0.0f, 0.0f, 0.0f};

  // This wavefront's steps: first, first + stride, ...
  const uint32_t first = part * W + wave, stride = parts * W;
  const uint32_t count = first < steps ? (steps - first + stride - 1) / stride : 0;
  // Slot S: step X of this wavefront's.  Steps past the last repeat it, so
  // that every wait counts the same loads; they are never multiplied.
#define FK_SKINNY_LOAD(S, X)                                                                                    \
  do {                                                                                                          \
    const uint32_t at_ = min(first + (uint32_t)(X) * stride, steps - 1) * 16384;                                   \
    FK_LDS char *d_ = ring + (S) * (CH * 1024);                                                                 \
    _Pragma("unroll") for (int j_ = 0; j_ < NB; j_++)                                                           \
      __builtin_amdgcn_raw_ptr_buffer_load_lds(bsrc, d_ + j_ * 1024, 16, bv + chunk_of(j_) * 1024, at_, 0, HINT); \
    _Pragma("unroll") for (int i_ = 0; i_ < MB; i_++)                                                           \
      __builtin_amdgcn_raw_ptr_buffer_load_lds(asrc, d_ + (NB + i_) * 1024, 16, av[i_], at_, 0, 0);             \
  } while (0)
  // Slot S's step once it has landed (the loads of the D - 1 steps after it
  // still in flight): its fragments into registers, its slot loaded again,
  // its matrix operations.
#define FK_SKINNY_VMCNT(N) __builtin_amdgcn_s_waitcnt(((N) & 15) | (((N) >> 4) << 14) | (0x7 << 4) | (0xf << 8))
#define FK_SKINNY_STEP(S, X)                                                                                    \
  do {                                                                                                          \
    fk::Half8 fa[MB], fb[NB];                                                                                   \
    FK_SKINNY_VMCNT((D - 1) * CH);                                                                              \
    asm volatile("" ::: "memory");                                                                              \
    _Pragma("unroll") for (int j_ = 0; j_ < NB; j_++) fb[j_].u = lds[fu + ((S) * CH + j_) * FK_WAVE];           \
    _Pragma("unroll") for (int i_ = 0; i_ < MB; i_++) fa[i_].u = lds[fu + ((S) * CH + NB + i_) * FK_WAVE];      \
    _Pragma("unroll") for (int j_ = 0; j_ < NB; j_++) asm volatile("" : "+v"(fb[j_].h));                        \
    _Pragma("unroll") for (int i_ = 0; i_ < MB; i_++) asm volatile("" : "+v"(fa[i_].h));                        \
    asm volatile("" ::: "memory");                                                                              \
    FK_SKINNY_LOAD(S, (X) + D);                                                                                 \
    _Pragma("unroll") for (int i_ = 0; i_ < MB; i_++)                                                           \
    _Pragma("unroll") for (int j_ = 0; j_ < NB; j_++)                                                           \
      acc[i_][j_] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fb[j_].h, fa[i_].h, acc[i_][j_], 0, 0, 0);           \
    if constexpr (MB * NB >= 64) { /* the accumulators stay in AGPRs from step to step */                       \
      _Pragma("unroll") for (int i_ = 0; i_ < MB; i_++)                                                         \
      _Pragma("unroll") for (int j_ = 0; j_ < NB; j_++) asm volatile("" : "+a"(acc[i_][j_]));                   \
    }                                                                                                           \
  } while (0)
  auto loop = [&](auto streamed) {
    constexpr int HINT = decltype(streamed)::value ? 2 : 0;  // non-temporal
#pragma unroll
    for (int s = 0; s < D; s++) FK_SKINNY_LOAD(s, s);
    uint32_t x = 0;
    for (; x + D <= count; x += D) {
#pragma unroll
      for (int s = 0; s < D; s++) FK_SKINNY_STEP(s, x + s);
    }
#pragma unroll
    for (int s = 0; s < D - 1; s++)
      if (x + s < count) FK_SKINNY_STEP(s, x + s);
  };
  // Weights that one or two tiles of rows read are streamed past the caches
  // (the down projection of 16 rows in 6 % less time, gate and up in 11 %);
  // read by more, they are kept (the down projection of 112 rows, four tiles,
  // in 6 % less).
  if constexpr (MB * NB >= 64) loop(fk_bool_tag<false>{});
  else if (tiles_m <= 2) loop(fk_bool_tag<true>{});
  else loop(fk_bool_tag<false>{});
#undef FK_SKINNY_LOAD
#undef FK_SKINNY_STEP
#undef FK_SKINNY_VMCNT
  // (The lane index is taken anew through an asm statement, so that nothing of
  // the epilogue is computed before the loop and held in registers across it.)
  uint32_t lane_e;
  asm volatile("v_mov_b32 %0, %1" : "=v"(lane_e) : "v"(lane));
  const uint32_t nq = 4 * (lane_e / 16);
  // A unit's first column among its anchor's (QKV: in its head, d).
  auto unit_col = [&](uint32_t un) -> uint32_t {
    if constexpr (MODE == FK_GEMM_SILU_MUL) return n0 + 16 * un + nq;
    else if constexpr (QKV) return (NB == 2 ? n0 % 64 : un % 2 * 16) + nq;
    else return n0 + 16 * un * U + nq;
  };
  const uint32_t ld = anchor == 0 ? p.g.ldc[0] : (anchor == 1 ? p.g.ldc[1] : p.g.ldc[2]);
  fk_float4v with[ROUNDS][IT][QKV ? 2 : 1];  // the residual's columns; QKV: two pairs' (cos, sin) twice
  if constexpr (MODE == FK_GEMM_ADD || QKV) {
#pragma unroll
    for (int round = 0; round < ROUNDS; round++)
#pragma unroll
      for (int it = 0; it < IT; it++) {
        const uint32_t col = unit_col((wave + it * W) % NU);
        if constexpr (QKV) {
          const float *const cs = rope + (size_t)min(upos[round][it], p.r.rope_rows - 1) * 64 + 2 * col;
          with[round][it][0] = *reinterpret_cast<const fk_float4v *>(cs);
          with[round][it][1] = *reinterpret_cast<const fk_float4v *>(cs + 4);
        } else {
          const uint32_t row = min(unit_row(round, it, lane_e), p.g.m - 1);
          with[round][it][0] = *reinterpret_cast<const fk_float4v *>(r0 + (size_t)row * ld + col);
        }
      }
  }
  // Nothing may still be landing in LDS when the sums take the rings' place.
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();

#pragma unroll
  for (int round = 0; round < ROUNDS; round++) {
    if (round) __syncthreads();
#pragma unroll
    for (int i = 0; i < MR; i++)
#pragma unroll
      for (int j = 0; j < NB; j++) sums[wave][i * NB + j][lane_e] = acc[round * MR + i][j];
    __syncthreads();
    // (Unrolled where a unit's operands are in registers; elsewhere a loop,
    // since straight-line code that runs once is fetched at its own cost:
    // gate and up of 208 rows unrolled, 31 µs against 28.)
    constexpr int UNROLL = MODE == FK_GEMM_ADD || QKV ? IT : 1;
#pragma unroll UNROLL
    for (int it = 0; it < IT; it++) {
      const uint32_t u = wave + it * W;
      if (u >= (uint32_t)UNITS) break;
      const uint32_t un = u % NU;
      const uint32_t row = unit_row(round, it, lane_e);
      const uint32_t col = unit_col(un);
      // The sum of the unit's block q.
      auto total = [&](int q) {
        uint32_t j;
        if constexpr (MODE == FK_GEMM_SILU_MUL) j = un + q * (NB / 2);
        else if constexpr (QKV && NB == 2) j = q;
        else if constexpr (QKV) j = un / 2 * 4 + un % 2 + 2 * q;
        else j = un * U + q;
        const uint32_t at = u / NU * NB + j;
        fk_float4v v = sums[0][at][lane_e];
#pragma unroll
        for (int w = 1; w < W; w++) v += sums[w][at][lane_e];
        return v;
      };
      if constexpr (MODE == FK_GEMM_SILU_MUL) {
        const fk_float4v g = total(0), up = total(1);
        if (row >= p.g.m) continue;
        uint16_t h[4];
#pragma unroll
        for (int r = 0; r < 4; r++)
          h[r] = fk::to_f16((p.g.act == FK_ACT_GELU_TANH ? fk::act_hw<true>(g[r]) : fk::act_hw<false>(g[r])) * up[r]);
        *reinterpret_cast<uint2 *>(reinterpret_cast<uint16_t *>(c0) +
                                   fk::tile_offset(p.compact ? (tm * MB + round * MR + u / NU) * 16 + lane_e % 16 : row, col, ld)) =
            make_uint2(h[0] | ((uint32_t)h[1] << 16), h[2] | ((uint32_t)h[3] << 16));
      } else if constexpr (QKV) {
        // The unit's columns d .. d + 3 of its head, and their partners d + 32 ..
        const fk_float4v lo = total(0), hi = total(1);
        if (row >= p.g.m) continue;
        const uint32_t head = n0 / 64 + (NB == 2 ? 0 : un / 2);
        const uint32_t pos = upos[round][it];
        const bool bf16 = p.r.cache_bf16 != 0 && anchor != 0;
        uint16_t l4[4], h4[4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const float cs = with[round][it][r / 2][r % 2 * 2], sn = with[round][it][r / 2][r % 2 * 2 + 1];
          const float xr = anchor != 2 ? lo[r] * cs - hi[r] * sn : lo[r];
          const float yr = anchor != 2 ? hi[r] * cs + lo[r] * sn : hi[r];
          l4[r] = bf16 ? fk::narrow_bf16(xr) : fk::to_f16(xr);
          h4[r] = bf16 ? fk::narrow_bf16(yr) : fk::to_f16(yr);
        }
        uint16_t *dst = reinterpret_cast<uint16_t *>(anchor == 0 ? c0 : (anchor == 1 ? c1 : c2));
        if (anchor == 0) {
          dst += (size_t)row * ld + head * 64;
        } else if constexpr (MODE == FK_GEMM_QKV_ROPE_PAGED) {
          // a position past its table stores nothing
          if (pos / p.pg.block_size >= p.pg.table_len) continue;
          const uint32_t bl = min(slot[(size_t)row * p.pg.table_len + pos / p.pg.block_size], p.pg.blocks - 1);
          dst += (((size_t)bl * p.r.kv_heads + head) * p.pg.block_size + pos % p.pg.block_size) * 64;
        } else if (p.r.staged) {
          dst += ((size_t)row * p.r.kv_heads + head) * 64;
        } else {
          dst += (((size_t)min(uslot[round][it], p.r.slots - 1) * p.r.kv_heads + head) * p.r.length + pos % p.r.length) * 64;
        }
        *reinterpret_cast<uint2 *>(dst + col) =
            make_uint2(l4[0] | ((uint32_t)l4[1] << 16), l4[2] | ((uint32_t)l4[3] << 16));
        *reinterpret_cast<uint2 *>(dst + col + 32) =
            make_uint2(h4[0] | ((uint32_t)h4[1] << 16), h4[2] | ((uint32_t)h4[3] << 16));
      } else {
        float *const out = reinterpret_cast<float *>(anchor == 0 ? c0 : (anchor == 1 ? c1 : c2));
        uint64_t best = 0;
#pragma unroll
        for (int q = 0; q < U; q++) {
          fk_float4v v = total(q);
          if (MODE == FK_GEMM_PART) {
            // [parts][live 16][ld]: every row of a live chunk, the rows past
            // the step's zeros
            const uint32_t c = tm * MB + round * MR + u / NU;
            if (c < p.live)
              *reinterpret_cast<fk_float4v *>(out + ((size_t)part * p.live * 16 + c * 16 + lane_e % 16) * ld + col) = v;
          } else if (row < p.g.m) {
            if (MODE == FK_GEMM_ADD) v = with[round][it][0] + v;
            *reinterpret_cast<fk_float4v *>(out + (size_t)row * ld + col + 16 * q) = v;
          }
          if constexpr (MODE == FK_GEMM_STORE_KEYS) {
#pragma unroll
            for (int r = 0; r < 4; r++) {
              const uint64_t key = fk::argmax_key(v[r], col + 16 * q + r);
              best = key > best ? key : best;
            }
          }
        }
        if constexpr (MODE == FK_GEMM_STORE_KEYS) {
          // Lanes l, l ^ 16, l ^ 32 and l ^ 48 hold the same row's other
          // columns.
#pragma unroll
          for (int s = 16; s <= 32; s <<= 1) {
            const uint64_t other = ((uint64_t)(uint32_t)__shfl_xor((int)(best >> 32), s) << 32) |
                                   (uint64_t)(uint32_t)__shfl_xor((int)(uint32_t)best, s);
            best = other > best ? other : best;
          }
          if (lane_e < 16 && row < p.g.m) keys[(size_t)row * (ld / (16 * NB)) + n0 / (16 * NB)] = best;
        }
      }
    }
  }
}

// Buffers in binding order, then the parameter struct; W wavefronts.  The
// grid: every tile of rows of every tile of columns, the tiles of columns
// rounded up to a multiple of 8.
#define FK_SKINNY_ENTRY(NAME, MODE, MB, NB, W, D)                                                                  \
  extern "C" __global__ void __launch_bounds__(64 * W)                                                             \
      NAME(const _Float16 *__restrict__ a, const _Float16 *__restrict__ b0, const _Float16 *__restrict__ b1,      \
           const _Float16 *__restrict__ b2, void *__restrict__ c0, void *__restrict__ c1, void *__restrict__ c2,  \
           const float *r0, const uint32_t *__restrict__ position, const uint32_t *__restrict__ slot,             \
           const float *__restrict__ rope, uint64_t *__restrict__ keys, fk_skinny_params p) {                     \
    skinny_tile<MODE, MB, NB, W, D>(a, b0, b1, b2, c0, c1, c2, r0, position, slot, rope, keys, p);                \
  }

// S: the ring's steps in the modes that stream many tiles (gate and up, the
// logits), D in the rest.  m8n8's rings take 64 KB a step and its sums 128 KB,
// so a second step costs no LDS, but gate and up are slower with it (112 rows
// 30.9 µs, two steps 33.4; 208, 30.3 and 32.8), the logits about the same (112
// rows 42.7 and 42.0).
#define FK_SKINNY_FORM(FORM, MB, NB, W, D, S)                                   \
  FK_SKINNY_ENTRY(fk_skinny_part_##FORM, FK_GEMM_PART, MB, NB, W, D)            \
  FK_SKINNY_ENTRY(fk_skinny_store_##FORM, FK_GEMM_STORE, MB, NB, W, D)          \
  FK_SKINNY_ENTRY(fk_skinny_add_##FORM, FK_GEMM_ADD, MB, NB, W, D)              \
  FK_SKINNY_ENTRY(fk_skinny_store_keys_##FORM, FK_GEMM_STORE_KEYS, MB, NB, W, S)
#define FK_SKINNY_PAIR_FORM(FORM, MB, NB, W, D, S)                              \
  FK_SKINNY_FORM(FORM, MB, NB, W, D, S)                                         \
  FK_SKINNY_ENTRY(fk_skinny_silu_mul_##FORM, FK_GEMM_SILU_MUL, MB, NB, W, S)    \
  FK_SKINNY_ENTRY(fk_skinny_qkv_rope_##FORM, FK_GEMM_QKV_ROPE, MB, NB, W, D)    \
  FK_SKINNY_ENTRY(fk_skinny_qkv_rope_paged_##FORM, FK_GEMM_QKV_ROPE_PAGED, MB, NB, W, D)

#ifndef FK_SKINNY_FORMS
#define FK_SKINNY_FORMS
FK_SKINNY_FORM(m1n1, 1, 1, 8, 2, 2)
FK_SKINNY_PAIR_FORM(m1n2, 1, 2, 8, 2, 1)
FK_SKINNY_FORM(m2n1, 2, 1, 8, 2, 2)
FK_SKINNY_PAIR_FORM(m2n2, 2, 2, 8, 2, 2)
FK_SKINNY_PAIR_FORM(m2n4, 2, 4, 4, 2, 2)
FK_SKINNY_PAIR_FORM(m4n2, 4, 2, 8, 2, 2)
FK_SKINNY_PAIR_FORM(m4n4, 4, 4, 4, 2, 2)
FK_SKINNY_PAIR_FORM(m4n8, 4, 8, 4, 2, 2)
FK_SKINNY_PAIR_FORM(m8n8, 8, 8, 4, 2, 1)
#endif
