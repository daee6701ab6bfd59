// fk_rows_attend.h — the attention of a step whose rows are each a sequence's
// one (a batch of decode steps, prefill.py's DecodeRows): row i's query is the
// first row of query block i.
//
// fk_prefill_attend takes such a row as a block of 32 queries (31 of them
// filling) and one threadgroup a kv head walks all its keys: 8 rows of up to
// 4096 positions are 64 threadgroups, 58 µs.  Here the keys are split:
//
// - Threadgroup (row, kv head, part j of X) takes the row's tiles of 256 keys
//   j, j + X, ...; each of its 4 wavefronts 64 keys of a tile, their K and V
//   rows loaded straight into the wavefront's own 16 KB of LDS (all of a
//   tile's loads in flight at once; two threadgroups a CU overlap one's loads
//   with the other's arithmetic), with its own running maximum, sum and
//   weighted values.  No barrier until the wavefronts' states meet.
// - The group's query heads (heads / kv heads, up to 16) are the columns of
//   the matrix operations: S = K Qᵀ and Oᵀ = Vᵀ Pᵀ on v_mfma_f32_16x16x32_f16
//   with the probabilities in the registers that made them (the order of the
//   keys is the scores', which the transposed V reads follow).
// - A row whose keys lie in one part is finished there; the rest leave (O, m,
//   l) partials, f32, that fk_rows_combine adds.
//
// What bounds it: the K and V rows' stream (2 KB a position at 8 kv heads of
// 64) once there are many (64 rows, 185 MB: 36.6 µs, 5.1 TB/s), and below that
// a launch's latency (one row of 4096 positions, 8.4 MB: 5.9 µs).  8 rows of
// 256 to 4095 positions: 58 µs in blocks of 32 queries, 10.6 here and 2.3 for
// the combine; 41 rows of up to 700: 18 µs, now 8.9 and 2.1.
//
// The arithmetic is fk_prefill_attend's: f16 operands, binary32 scores,
// probabilities rounded to f16 and summed as rounded, exp2 of scores in log2
// units.  A wavefront's reference lies 8 below its running maximum, so that
// its probabilities reach 2^8 and small ones keep f16's bits at least as long
// as with that kernel's reference, which may lag its maximum by up to 8.
#pragma once

#include "fk_common.h"
#include "fk_layout.h"
#include "fk_mfma.h"

#define FK_ROWS_WAVES 4
#define FK_ROWS_TILE (64 * FK_ROWS_WAVES)  // keys a tile
#define FK_ROWS_LDS __attribute__((address_space(3)))

typedef short fk_rows_short4 __attribute__((ext_vector_type(4)));
typedef _Float16 fk_rows_half2 __attribute__((ext_vector_type(2)));
typedef float fk_rows_float2 __attribute__((ext_vector_type(2)));

namespace fk {

// A row's keys and how they are split: tiles [t0, t1] hold keys first .. pos.
struct RowKeys {
  uint32_t pos, first, t0, t1;
};

__device__ __forceinline__ RowKeys row_keys(const uint32_t *position, uint32_t row, uint32_t window) {
  RowKeys k;
  k.pos = position[row];
  k.first = window && k.pos + 1 > window ? k.pos + 1 - window : 0u;
  k.t0 = k.first / FK_ROWS_TILE;
  k.t1 = k.pos / FK_ROWS_TILE;
  return k;
}

// Over lanes l, l ^ 16, l ^ 32 and l ^ 48.
__device__ __forceinline__ float rows_max(float x) {
  auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = __builtin_fmaxf(__uint_as_float(s[0]), __uint_as_float(s[1]));
  s = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __builtin_fmaxf(__uint_as_float(s[0]), __uint_as_float(s[1]));
}
__device__ __forceinline__ float rows_sum(float x) {
  auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = __uint_as_float(s[0]) + __uint_as_float(s[1]);
  s = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(s[0]) + __uint_as_float(s[1]);
}

// bf16 pairs of a word -> f16 pairs (the matrix operations take f16).
__device__ __forceinline__ uint32_t rows_f16x2(uint32_t w) {
  return to_f16(__uint_as_float(w << 16)) | ((uint32_t)to_f16(__uint_as_float(w & 0xffff0000u)) << 16);
}

}  // namespace fk

template <bool BF16>
__device__ __forceinline__ void rows_attend(const uint16_t *__restrict__ qr, const uint16_t *__restrict__ kc,
                                            const uint16_t *__restrict__ vc, const uint32_t *__restrict__ position,
                                            const uint32_t *__restrict__ slot, uint16_t *__restrict__ out,
                                            float *__restrict__ partials, const fk_rows_attend_params &p) {
  __shared__ __attribute__((aligned(16))) uint16_t kv[FK_ROWS_WAVES][2][64 * 64];
  // (the wavefronts' weighted values take the place of their keys at the end:
  // 65 KB in all, two threadgroups a CU)
  float(*const so)[16][64] = reinterpret_cast<float(*)[16][64]>(kv);
  __shared__ float sm[FK_ROWS_WAVES][16], sl[FK_ROWS_WAVES][16];
  const uint32_t lane = threadIdx.x & (FK_WAVE - 1);
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / FK_WAVE);
  // Part by part, so that the parts past short rows' keys come last.
  const uint32_t pairs = p.rows * p.kv_heads;
  const uint32_t part = blockIdx.x / pairs;
  const uint32_t i = blockIdx.x % pairs / p.kv_heads;
  const uint32_t g = blockIdx.x % p.kv_heads;
  const uint32_t row = i * p.apart;
  const fk::RowKeys ks = fk::row_keys(position, row, p.window);
  const uint32_t tiles = ks.t1 - ks.t0 + 1;
  if (part >= tiles) return;
  const uint32_t G = p.heads / p.kv_heads;
  const uint32_t qw = p.heads * 64;
  const float c = p.scale * 1.4426950408889634f;  // scores to log2 units

  // Q (B of S = K Qᵀ): lane l holds head l mod 16 (past the group: its last),
  // d 32 h + 8 (l div 16) .. + 7.
  fk::Half8 qf[2];
#pragma unroll
  for (int h = 0; h < 2; h++)
    qf[h].u = *reinterpret_cast<const uint4 *>(qr + (size_t)row * qw + (g * G + min(lane % 16, G - 1)) * 64 + 32 * h +
                                               8 * (lane / 16));

  const size_t base = ((size_t)min(slot[row], p.slots - 1) * p.kv_heads + g) * p.length * 64;
  const auto krs = fk::buffer(kc + base, (size_t)p.length * 128);
  const auto vrs = fk::buffer(vc + base, (size_t)p.length * 128);
  uint16_t *const kbuf = kv[wave][0], *const vbuf = kv[wave][1];

  fk_float4v o[4];
#pragma unroll
  for (int d = 0; d < 4; d++) o[d] = fk_float4v{0.0f, 0.0f, 0.0f, 0.0f};
  float m = -__builtin_inff(), l = 0.0f;

  for (uint32_t t = ks.t0 + part; t <= ks.t1; t += p.parts) {
    const uint32_t key0 = t * FK_ROWS_TILE + wave * 64;
    if (key0 > ks.pos || key0 + 63 < ks.first) continue;
    // The 64 keys' rows, 8 a load (lane L 16-byte unit L mod 8 of key L div
    // 8): K's unit u at place u ^ ((key >> 1) mod 8) of its row, V's 32-byte
    // pieces at piece ^ ((key >> 1) mod 4), so that the reads below meet
    // different banks.  Keys past the row's own read its own (masked, finite).
#pragma unroll
    for (int q = 0; q < 8; q++) {
      const uint32_t key = q * 8 + lane / 8;
      const uint32_t at = min(key0 + key, ks.pos) * 128;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(krs, (FK_ROWS_LDS char *)kbuf + q * 1024, 16,
                                               at + (((lane % 8) ^ ((key >> 1) & 7u)) * 16), 0, 0, 2);
    }
#pragma unroll
    for (int q = 0; q < 8; q++) {
      const uint32_t key = q * 8 + lane / 8;
      const uint32_t at = min(key0 + key, ks.pos) * 128;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(vrs, (FK_ROWS_LDS char *)vbuf + q * 1024, 16,
                                               at + (((lane % 8) ^ (((key >> 1) & 3u) << 1)) * 16), 0, 0, 2);
    }
    __builtin_amdgcn_s_waitcnt(8 | (0x7 << 4) | (0xf << 8));  // K landed, V's 8 loads in flight
    asm volatile("" ::: "memory");
    // S: four groups of 16 keys; register r of group s is key 16 s + 4 (l div
    // 16) + r of the 64, head l mod 16.
    fk_float4v sc[4];
#pragma unroll
    for (int s = 0; s < 4; s++) {
      sc[s] = fk_float4v{0.0f, 0.0f, 0.0f, 0.0f};
      const uint32_t key = 16 * s + lane % 16;
#pragma unroll
      for (int h = 0; h < 2; h++) {
        fk::Half8 kf;
        kf.u = *reinterpret_cast<const uint4 *>(&kbuf[key * 64 + ((4 * h + lane / 16) ^ ((key >> 1) & 7u)) * 8]);
        if constexpr (BF16)
          kf.u = make_uint4(fk::rows_f16x2(kf.u.x), fk::rows_f16x2(kf.u.y), fk::rows_f16x2(kf.u.z),
                            fk::rows_f16x2(kf.u.w));
        sc[s] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf.h, qf[h].h, sc[s], 0, 0, 0);
      }
    }
    float mt = -__builtin_inff();
#pragma unroll
    for (int s = 0; s < 4; s++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const uint32_t k = key0 + 16 * s + 4 * (lane / 16) + r;
        sc[s][r] = k <= ks.pos && k >= ks.first ? sc[s][r] * c : -__builtin_inff();
        mt = __builtin_fmaxf(mt, sc[s][r]);
      }
    mt = fk::rows_max(mt) - 8.0f;
    // (a head whose scores are all -inf, or NaN, keeps nothing: 0 in place
    // of its reference)
    const float mn = __builtin_fmaxf(m, mt);
    const float mc = mn == -__builtin_inff() ? 0.0f : mn;
    const float alpha = __builtin_amdgcn_exp2f(m - mc);
    m = mn;
    fk::Half8 pf[2];
    float sum = 0.0f;
    const fk_rows_half2 ones = {(_Float16)1.0f, (_Float16)1.0f};
#pragma unroll
    for (int s = 0; s < 4; s++)
#pragma unroll
      for (int r = 0; r < 4; r += 2) {
        const fk_rows_half2 e = __builtin_convertvector(
            (fk_rows_float2){__builtin_amdgcn_exp2f(sc[s][r] - mc), __builtin_amdgcn_exp2f(sc[s][r + 1] - mc)},
            fk_rows_half2);
        reinterpret_cast<fk_rows_half2 *>(&pf[s / 2])[(s % 2) * 2 + r / 2] = e;
        sum = __builtin_amdgcn_fdot2(e, ones, sum, false);
      }
    l = l * alpha + fk::rows_sum(sum);
#pragma unroll
    for (int d = 0; d < 4; d++) o[d] *= alpha;
    __builtin_amdgcn_s_waitcnt(0x0 | (0x7 << 4) | (0xf << 8));  // V landed
    asm volatile("" ::: "memory");
    // Oᵀ += Vᵀ Pᵀ.  Transposed reads: within 16 lanes, lane 4 k + q reads key
    // K0 + k, d D0 + 4 q .. + 3 and receives keys K0 .. K0 + 3 of d D0 + (its
    // index): keys 32 h + 4 (l div 16) .. + 3 and 16 further, pf[h]'s order.
    const uint32_t tk = 4 * (lane / 16) + lane % 16 / 4, td = 4 * (lane & 3);
#pragma unroll
    for (int d = 0; d < 4; d++)
#pragma unroll
      for (int h = 0; h < 2; h++) {
        uint2 w[2];
#pragma unroll
        for (int q = 0; q < 2; q++) {
          const uint32_t key = 32 * h + 16 * q + tk;
          w[q] = __builtin_bit_cast(
              uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                         (FK_ROWS_LDS fk_rows_short4 *)&vbuf[key * 64 + ((16 * d + td) ^ (((key >> 1) & 3u) << 4))]));
          if constexpr (BF16) w[q] = make_uint2(fk::rows_f16x2(w[q].x), fk::rows_f16x2(w[q].y));
        }
        fk::Half8 vf;
        vf.u = make_uint4(w[0].x, w[0].y, w[1].x, w[1].y);
        o[d] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf.h, pf[h].h, o[d], 0, 0, 0);
      }
    // The reads are done before the next tile's loads land on them.
    asm volatile("" : "+v"(o[0]), "+v"(o[1]), "+v"(o[2]), "+v"(o[3])::"memory");
  }

  // The wavefronts' states: head l mod 16, d 16 dt + 4 (l div 16) + r.
  __syncthreads();
  if (lane % 16 < G) {
#pragma unroll
    for (int d = 0; d < 4; d++)
      *reinterpret_cast<fk_float4v *>(&so[wave][lane % 16][16 * d + 4 * (lane / 16)]) = o[d];
    if (lane < 16) {
      sm[wave][lane] = m;
      sl[wave][lane] = l;
    }
  }
  __syncthreads();
  const bool whole = tiles == 1 || p.parts == 1;
  for (uint32_t e = threadIdx.x; e < G * 64; e += 64 * FK_ROWS_WAVES) {
    const uint32_t q = e / 64, d = e % 64;
    float mm = sm[0][q];
#pragma unroll
    for (int w = 1; w < FK_ROWS_WAVES; w++) mm = __builtin_fmaxf(mm, sm[w][q]);
    const float mc = mm == -__builtin_inff() ? 0.0f : mm;
    float ll = 0.0f, oo = 0.0f;
#pragma unroll
    for (int w = 0; w < FK_ROWS_WAVES; w++) {
      const float f = __builtin_amdgcn_exp2f(sm[w][q] - mc);
      ll += sl[w][q] * f;
      oo += so[w][q][d] * f;
    }
    if (whole) {
      out[fk::tile_offset(p.compact ? i : row, (g * G + q) * 64 + d, qw)] = fk::to_f16(oo / ll);
    } else {
      float *const to = partials + (((size_t)(i * p.kv_heads + g) * p.parts + part) * G + q) * 66;
      to[d] = oo;
      if (d == 0) {
        to[64] = mm;
        to[65] = ll;
      }
    }
  }
}

extern "C" __global__ void __launch_bounds__(64 * FK_ROWS_WAVES, 2)
    fk_rows_attend_f16(const uint16_t *__restrict__ qr, const uint16_t *__restrict__ kc,
                       const uint16_t *__restrict__ vc, const uint32_t *__restrict__ position,
                       const uint32_t *__restrict__ slot, uint16_t *__restrict__ out, float *__restrict__ partials,
                       fk_rows_attend_params p) {
  rows_attend<false>(qr, kc, vc, position, slot, out, partials, p);
}

extern "C" __global__ void __launch_bounds__(64 * FK_ROWS_WAVES, 2)
    fk_rows_attend_bf16(const uint16_t *__restrict__ qr, const uint16_t *__restrict__ kc,
                        const uint16_t *__restrict__ vc, const uint32_t *__restrict__ position,
                        const uint32_t *__restrict__ slot, uint16_t *__restrict__ out, float *__restrict__ partials,
                        fk_rows_attend_params p) {
  rows_attend<true>(qr, kc, vc, position, slot, out, partials, p);
}

// The partials of the rows whose keys took several parts, added in the order
// of the parts: one threadgroup a (row, kv head), one wavefront a query head.
extern "C" __global__ void __launch_bounds__(1024)
    fk_rows_combine(const float *__restrict__ partials, const uint32_t *__restrict__ position,
                    uint16_t *__restrict__ out, fk_rows_attend_params p) {
  const uint32_t i = blockIdx.x / p.kv_heads, g = blockIdx.x % p.kv_heads;
  const uint32_t row = i * p.apart;
  const fk::RowKeys ks = fk::row_keys(position, row, p.window);
  const uint32_t parts = min(ks.t1 - ks.t0 + 1, p.parts);
  if (parts == 1) return;
  const uint32_t G = p.heads / p.kv_heads;
  const uint32_t q = threadIdx.x / FK_WAVE, d = threadIdx.x % FK_WAVE;
  const float *const from = partials + ((size_t)(i * p.kv_heads + g) * p.parts * G + q) * 66;
  float mm = -__builtin_inff(), ll = 0.0f, oo = 0.0f;
  for (uint32_t s0 = 0; s0 < parts; s0 += 8) {
    float m[8], l[8], o[8];
#pragma unroll
    for (uint32_t s = 0; s < 8; s++) {
      const float *const at = from + (size_t)min(s0 + s, parts - 1) * G * 66;
      m[s] = s0 + s < parts ? at[64] : -__builtin_inff();
      l[s] = at[65];
      o[s] = at[d];
    }
    float mn = mm;
#pragma unroll
    for (uint32_t s = 0; s < 8; s++) mn = __builtin_fmaxf(mn, m[s]);
    const float mc = mn == -__builtin_inff() ? 0.0f : mn;
    const float f0 = __builtin_amdgcn_exp2f(mm - mc);
    ll *= f0;
    oo *= f0;
#pragma unroll
    for (uint32_t s = 0; s < 8; s++) {
      const float f = __builtin_amdgcn_exp2f(m[s] - mc);
      ll += l[s] * f;
      oo += o[s] * f;
    }
    mm = mn;
  }
  out[fk::tile_offset(p.compact ? i : row, (g * G + q) * 64 + d, p.heads * 64)] = fk::to_f16(oo / ll);
}
