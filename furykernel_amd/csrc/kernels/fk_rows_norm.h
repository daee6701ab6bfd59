// fk_rows_norm.h — the kernels between the GEMMs of a step of few rows
// (fk_skinny.h), on its live rows alone:
//
//   fk_rows_norm_w*     RMSNorm of f32 rows into the GEMM's f16 tiles, and
//                       before it what makes the row: the token's embedding
//                       gathered, or the residual added to the partial sums a
//                       GEMM left (fk_skinny_part_*)
//   fk_rows_token       the greedy token of each row from the head's keys
//
// A launch of these moves some tens of KB and costs its latency (3 to 6 µs on
// all of a step's rows, fk_prefill_norm_pack and fk_prefill_gather), so they
// are folded into one, a row a threadgroup: a step of 8 rows gathers and norms
// in one launch, and the down projection, split over the chip further than
// its threadgroups' wavefronts can add up, has its partial sums added here.
// Two 1B layers and the head, with that split and the batch's tiled values
// held compact: 8 rows 157 -> 145 µs, 41 rows 216 -> 163, a prompt of 100 rows
// 204 -> 194.
#pragma once

#include "fk_common.h"
#include "fk_layout.h"
#include "fk_mfma.h"

namespace fk {

// Row i of the live rows (fk_skinny.h's chunks).
__device__ __forceinline__ uint32_t live_row(uint32_t i, uint32_t run_chunks, uint32_t run, uint32_t apart) {
  const uint32_t c = i / 16;
  return (c / run_chunks) * run + ((c % run_chunks) * 16 + i % 16) * apart;
}

}  // namespace fk

// Rows of exactly 8 · T · V columns, T threads: thread t holds units t, t + T,
// ... of 8 columns between the row's making, its sum of squares and its tiles.
template <uint32_t T, uint32_t V>
__device__ __forceinline__ void rows_norm(const float *__restrict__ x, const void *__restrict__ table,
                                          const uint32_t *__restrict__ tokens, const float *__restrict__ partials,
                                          const float *__restrict__ gamma, float *__restrict__ xout,
                                          uint16_t *__restrict__ y, const fk_rows_norm_params &p) {
  constexpr uint32_t width = 8 * T * V;
  const uint32_t i = blockIdx.x;
  const uint32_t row = fk::live_row(i, p.run_chunks, p.run, p.apart);
  if (row >= p.m) return;
  const uint32_t t = threadIdx.x;
  float v[V][8], g[V][8];
#pragma unroll
  for (uint32_t u = 0; u < V; u++) {
    const uint32_t c = 8 * (t + u * T);
#pragma unroll
    for (int e = 0; e < 8; e++) g[u][e] = 1.0f;
    if (p.has_gamma) {
#pragma unroll
      for (int q = 0; q < 2; q++) {
        const fk_float4v a = *reinterpret_cast<const fk_float4v *>(gamma + c + 4 * q);
#pragma unroll
        for (int e = 0; e < 4; e++) g[u][4 * q + e] = a[e];
      }
    }
    if (p.source == FK_ROWS_GATHER_F16) {
      const uint4 h = *reinterpret_cast<const uint4 *>(reinterpret_cast<const uint16_t *>(table) +
                                                       (size_t)min(tokens[row], p.table_rows - 1) * width + c);
      const uint32_t w[4] = {h.x, h.y, h.z, h.w};
#pragma unroll
      for (int e = 0; e < 4; e++) {
        v[u][2 * e] = fk::widen_f16(w[e] & 0xffffu) * p.gfactor;
        v[u][2 * e + 1] = fk::widen_f16(w[e] >> 16) * p.gfactor;
      }
    } else {
      const float *const from = p.source == FK_ROWS_GATHER_F32
                                    ? reinterpret_cast<const float *>(table) +
                                          (size_t)min(tokens[row], p.table_rows - 1) * width + c
                                    : x + (size_t)row * width + c;
      const float f = p.source == FK_ROWS_GATHER_F32 ? p.gfactor : 1.0f;
#pragma unroll
      for (int q = 0; q < 2; q++) {
        const fk_float4v a = *reinterpret_cast<const fk_float4v *>(from + 4 * q);
#pragma unroll
        for (int e = 0; e < 4; e++) v[u][4 * q + e] = a[e] * f;
      }
    }
  }
  if (p.source == FK_ROWS_PARTS) {
    // the residual and the parts' sum: (part 0 + part 1 + ...) first
    for (uint32_t u = 0; u < V; u++) {
      const float *const from = partials + (size_t)i * width + 8 * (t + u * T);
      fk_float4v s0 = {0.0f, 0.0f, 0.0f, 0.0f}, s1 = s0;
#pragma unroll 4
      for (uint32_t k = 0; k < p.parts; k++) {
        const float *const at = from + (size_t)k * p.live * 16 * width;
        s0 += *reinterpret_cast<const fk_float4v *>(at);
        s1 += *reinterpret_cast<const fk_float4v *>(at + 4);
      }
#pragma unroll
      for (int e = 0; e < 4; e++) {
        v[u][e] += s0[e];
        v[u][4 + e] += s1[e];
      }
    }
  }
  float ss = 0.0f;
#pragma unroll
  for (uint32_t u = 0; u < V; u++)
#pragma unroll
    for (int e = 0; e < 8; e += 2) ss += v[u][e] * v[u][e] + v[u][e + 1] * v[u][e + 1];
  ss = fk::wave_sum(ss);
  if constexpr (T > FK_WAVE) {
    __shared__ float sums[T / FK_WAVE];
    if (t % FK_WAVE == 0) sums[t / FK_WAVE] = ss;
    __syncthreads();
    ss = sums[0];
#pragma unroll
    for (uint32_t w = 1; w < T / FK_WAVE; w++) ss += sums[w];
  }
  const float s = fk::rsqrt_once(ss / (float)width + p.eps);
  const uint32_t tiled = p.compact ? i : row;
#pragma unroll
  for (uint32_t u = 0; u < V; u++) {
    const uint32_t c = 8 * (t + u * T);
    if (p.source != FK_ROWS_STORED) {
#pragma unroll
      for (int q = 0; q < 2; q++)
        *reinterpret_cast<fk_float4v *>(xout + (size_t)row * width + c + 4 * q) =
            fk_float4v{v[u][4 * q], v[u][4 * q + 1], v[u][4 * q + 2], v[u][4 * q + 3]};
    }
    uint32_t h[4];
#pragma unroll
    for (int e = 0; e < 4; e++)
      h[e] = fk::to_f16(v[u][2 * e] * s * g[u][2 * e] * p.factor) |
             ((uint32_t)fk::to_f16(v[u][2 * e + 1] * s * g[u][2 * e + 1] * p.factor) << 16);
    *reinterpret_cast<uint4 *>(y + fk::tile_offset(tiled, c, width)) = make_uint4(h[0], h[1], h[2], h[3]);
  }
}

#define FK_ROWS_NORM(W, T, V)                                                                                   \
  extern "C" __global__ void __launch_bounds__(T) fk_rows_norm_w##W(                                            \
      const float *__restrict__ x, const void *__restrict__ table, const uint32_t *__restrict__ tokens,        \
      const float *__restrict__ partials, const float *__restrict__ gamma, float *__restrict__ xout,           \
      uint16_t *__restrict__ y, fk_rows_norm_params p) {                                                        \
    rows_norm<T, V>(x, table, tokens, partials, gamma, xout, y, p);                                             \
  }
FK_ROWS_NORM(512, 64, 1)
FK_ROWS_NORM(1024, 128, 1)
FK_ROWS_NORM(2048, 256, 1)
FK_ROWS_NORM(4096, 256, 2)

// The greedy token of each live row: the largest of its keys ([rows][parts],
// as the head's GEMM leaves them), a row a threadgroup.
extern "C" __global__ void __launch_bounds__(256) fk_rows_token(const uint64_t *__restrict__ keys,
                                                                uint32_t *__restrict__ out, fk_rows_token_params p) {
  const uint32_t row = fk::live_row(blockIdx.x, p.run_chunks, p.run, p.apart);
  if (row >= p.m) return;
  const uint64_t *const kr = keys + (size_t)row * p.parts;
  uint64_t best = 0;
#pragma unroll 4
  for (uint32_t j = threadIdx.x; j < p.parts; j += 256) best = kr[j] > best ? kr[j] : best;
#pragma unroll
  for (int s = 32; s >= 1; s >>= 1) {
    const uint64_t other = ((uint64_t)(uint32_t)__shfl_xor((int)(best >> 32), s) << 32) |
                           (uint64_t)(uint32_t)__shfl_xor((int)(uint32_t)best, s);
    best = other > best ? other : best;
  }
  __shared__ uint64_t waves[4];
  if (threadIdx.x % FK_WAVE == 0) waves[threadIdx.x / FK_WAVE] = best;
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int w = 1; w < 4; w++) best = waves[w] > best ? waves[w] : best;
    out[row] = 0xFFFFFFFFu - (uint32_t)best;
  }
}
