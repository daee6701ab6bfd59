// fk_routed.h — the launches of a routed-experts step of one row, three where
// its plan's steps make seven.
//
// A step of few experts is short of work: each of its launches (the norm, the
// router's logits, the route, the gate and up rows, their activation, the
// down rows, the combine) takes 2 to 6 µs, of which the bytes of two experts
// of 1024 at a width of 2048 (25 MB) take 4 altogether, and a launch's start
// and end about 1 µs each.  Each kernel here does what two or three of them
// do, the same operations in the same order, and stores every value that
// they store; the engine takes one where those launches follow each other
// (lower.py's routed_fusions).  MI355X, two experts of 1024 of 16 at 2048, µs:
// the norm, router and route 2.8 + 2.4 + 3.6 apart, 5.7 in one; gate, up and
// activation 5.5 + 2.5, 5.4; down and combine 4.0 + 2.2, 3.7; the step's
// graph 30.2, now 19.9.
#pragma once

#include "fk_common.h"
#include "fk_gemv.h"
#include "fk_step.h"

// The norm, the router's logits and the route in one threadgroup of 16
// wavefronts: a wavefront's rows of the router (at most 2, of 2048 columns)
// are loaded before anything else, so that they arrive while the first four
// wavefronts norm the row (fk_rmsnorm_f32's order over 256 threads) into LDS.
// One CU draws the whole router, of 32 experts at 2048 columns 128 KB, still
// 4.2 µs less than the launches apart.  That is what the wavefronts' registers
// hold; more experts or columns run apart, not measured joined.
#define FK_ROUTER_THREADS 1024
#define FK_ROUTER_WIDTH 2048
#define FK_ROUTER_ROWS 2

namespace fk {

template <typename WT>
__device__ __forceinline__ void step_router(const float *__restrict__ x, const float *__restrict__ gamma,
                                            float *__restrict__ y, const WT *__restrict__ w,
                                            float *__restrict__ logits, const float *__restrict__ scale,
                                            uint32_t *__restrict__ ids, float *__restrict__ ws,
                                            const fk_step_router_params &p) {
  constexpr int P = 8, KPL = FK_ROUTER_WIDTH / P / FK_WAVE, R = FK_ROUTER_ROWS, W = FK_ROUTER_THREADS / FK_WAVE;
  constexpr int NT = 256, NH = FK_ROUTER_WIDTH / 4 / NT;  // the norm's threads and their packs
  __shared__ float4 xs[FK_ROUTER_WIDTH / 4];
  __shared__ float slots[NT / FK_WAVE], lg[R * W];
  const uint32_t t = threadIdx.x, lane = t & (FK_WAVE - 1);
  const uint32_t wave = __builtin_amdgcn_readfirstlane(t / FK_WAVE);
  const uint32_t packs = p.width / P, npacks = p.width / 4;
  float4 v[NH], g[NH];
  if (wave < NT / FK_WAVE) {
#pragma unroll
    for (int i = 0; i < NH; i++) v[i] = *reinterpret_cast<const float4 *>(x + 4 * (size_t)min(t + i * NT, npacks - 1));
    if (p.has_gamma) {
#pragma unroll
      for (int i = 0; i < NH; i++)
        g[i] = *reinterpret_cast<const float4 *>(gamma + 4 * (size_t)min(t + i * NT, npacks - 1));
    }
  }
  uint4 wv[R][KPL];
#pragma unroll
  for (int q = 0; q < R; q++) {
    const WT *wr = w + (size_t)min(wave + q * W, p.experts - 1) * p.width;
#pragma unroll
    for (int it = 0; it < KPL; it++)
      wv[q][it] = load16<false>(wr + (size_t)min(lane + FK_WAVE * (uint32_t)it, packs - 1) * P);
  }
  if (wave < NT / FK_WAVE) {
    float acc = 0.0f;
#pragma unroll
    for (int i = 0; i < NH; i++) {
      float a = acc + v[i].x * v[i].x;
      a = a + v[i].y * v[i].y;
      a = a + v[i].z * v[i].z;
      a = a + v[i].w * v[i].w;
      acc = t + i * NT < npacks ? a : acc;
    }
    acc = wave_sum(acc);
    if (lane == 0) slots[wave] = acc;
  }
  __syncthreads();
  if (wave < NT / FK_WAVE) {
    // block_reduce's second round, by each of the wavefronts
    float acc = -0.0f;
    if (lane < NT / FK_WAVE) acc = acc + slots[lane];
    const float factor = rsqrt_once(wave_sum(acc) / (float)p.width + p.eps);
#pragma unroll
    for (int i = 0; i < NH; i++) {
      if (t + i * NT >= npacks) break;
      float o[4] = {v[i].x * factor, v[i].y * factor, v[i].z * factor, v[i].w * factor};
      if (p.has_gamma) {
        o[0] = o[0] * g[i].x;
        o[1] = o[1] * g[i].y;
        o[2] = o[2] * g[i].z;
        o[3] = o[3] * g[i].w;
      }
      if (p.factor != 1.0f) {
#pragma unroll
        for (int e = 0; e < 4; e++) o[e] = o[e] * p.factor;
      }
      const float4 n = make_float4(o[0], o[1], o[2], o[3]);
      xs[t + i * NT] = n;
      *reinterpret_cast<float4 *>(y + 4 * (size_t)(t + i * NT)) = n;
    }
  }
  __syncthreads();
  float acc[R][P / 4] = {}, sum[R];
#pragma unroll
  for (int it = 0; it < KPL; it++) {
    const uint32_t j = lane + FK_WAVE * (uint32_t)it, jc = min(j, packs - 1);
    const float4 lo = xs[2 * jc], hi = xs[2 * jc + 1];
    const float xf[P] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
#pragma unroll
    for (int q = 0; q < R; q++) {
      float wf[P];
      unpack_w<P>(wv[q][it], wf, WT{});
      add_pack<P>(acc[q], xf, wf, j < packs);
    }
  }
#pragma unroll
  for (int q = 0; q < R; q++) sum[q] = acc[q][0] + acc[q][1];
  wave_sums<R>(sum);
#pragma unroll
  for (int q = 0; q < R; q++) {
    const uint32_t e = wave + q * W;
    if (lane == 0 && e < p.experts) {
      lg[e] = sum[q];
      logits[e] = sum[q];
    }
  }
  __syncthreads();
  if (wave == 0) route_row(lg, scale, ids, ws, p.experts, p.k, p.has_scale != 0);
}

}  // namespace fk

#define FK_ROUTER_ENTRY(NAME, WT)                                                                                 \
  extern "C" __global__ void __launch_bounds__(FK_ROUTER_THREADS)                                                 \
      NAME(const float *__restrict__ x, const float *__restrict__ gamma, float *__restrict__ y,                   \
           const WT *__restrict__ w, float *__restrict__ logits, const float *__restrict__ scale,                 \
           uint32_t *__restrict__ ids, float *__restrict__ ws, fk_step_router_params p) {                         \
    fk::step_router<WT>(x, gamma, y, w, logits, scale, ids, ws, p);                                               \
  }
FK_ROUTER_ENTRY(fk_step_router_f16, _Float16)
FK_ROUTER_ENTRY(fk_step_router_bf16, fk::bf16_t)

// The routed gate and up rows and act(gate) · up: a wavefront takes row i of
// a rank's gate and row i of its up, so that both sums are in its registers.
// A threadgroup is 4 wavefronts, a rank's rows in groups_per_rank of them.
namespace fk {

template <typename WT, int P, int KPL>
__device__ __forceinline__ void routed_pair(const WT *const (&wr)[2], const float *const (&xr)[1], uint32_t packs,
                                            float (&t)[2]) {
  if (packs == FK_WAVE * KPL) gemv_sums_inflight<WT, float, P, 2, 1, KPL, true>(wr, xr, packs, t);
  else gemv_sums_inflight<WT, float, P, 2, 1, KPL, false>(wr, xr, packs, t);
}

template <typename WT, int P>
__device__ __forceinline__ void gemv_routed_act(const uint64_t *__restrict__ table, const uint32_t *__restrict__ ids,
                                                const float *__restrict__ x, float *__restrict__ y,
                                                float *__restrict__ out, const fk_gemv_routed_act_params &p) {
  const uint32_t rank = blockIdx.x / p.groups_per_rank;
  const uint32_t i = blockIdx.x % p.groups_per_rank * (blockDim.x / FK_WAVE) + threadIdx.x / FK_WAVE;
  const uint32_t half = p.n / 2;
  if (rank >= p.ranks || i >= half) return;
  const WT *w = reinterpret_cast<const WT *>(table[min(ids[rank], p.entries - 1)]);
  const WT *const wr[2] = {w + (size_t)i * p.k, w + (size_t)(half + i) * p.k};
  const float *const xr[1] = {x + (p.shared ? (size_t)0 : (size_t)rank * p.k)};
  const uint32_t packs = p.k / P;
  float t[2];
  if (packs <= FK_WAVE * 2) routed_pair<WT, P, 2>(wr, xr, packs, t);
  else if (packs <= FK_WAVE * 4) routed_pair<WT, P, 4>(wr, xr, packs, t);
  else routed_pair<WT, P, 8>(wr, xr, packs, t);
  if ((threadIdx.x & (FK_WAVE - 1)) == 0) {
    y[(size_t)rank * p.n + i] = t[0];
    y[(size_t)rank * p.n + half + i] = t[1];
    out[(size_t)rank * half + i] = act_mul(t[0], t[1], p.act);
  }
}

// The routed down rows, their combine by the route's weights and the residual
// add: a wavefront takes row i of every rank, all of their loads in flight.
template <typename WT, int P, int R, int KPL>
__device__ __forceinline__ void routed_rows(const uint64_t *__restrict__ table, const uint32_t *__restrict__ ids,
                                            const float *__restrict__ x, float *__restrict__ y,
                                            const float *__restrict__ ws, const float *res, float *out,
                                            const fk_gemv_routed_combine_params &p, uint32_t i) {
  const WT *wr[R];
  const float *xr[R];
#pragma unroll
  for (int r = 0; r < R; r++) {
    wr[r] = reinterpret_cast<const WT *>(table[min(ids[r], p.entries - 1)]) + (size_t)i * p.k;
    xr[r] = x + (p.shared ? (size_t)0 : (size_t)r * p.k);
  }
  float t[R];
  gemv_sums_inflight<WT, float, P, R, R, KPL, false>(wr, xr, p.k / P, t);
  if ((threadIdx.x & (FK_WAVE - 1)) == 0) {
    float acc = ws[0] * t[0];
    y[i] = t[0];
#pragma unroll
    for (int r = 1; r < R; r++) {
      y[(size_t)r * p.n + i] = t[r];
      acc = acc + ws[r] * t[r];
    }
    if (p.residual) acc = res[i] + acc;
    out[i] = acc;
  }
}

template <typename WT, int P>
__device__ __forceinline__ void gemv_routed_combine(const uint64_t *__restrict__ table,
                                                    const uint32_t *__restrict__ ids, const float *__restrict__ x,
                                                    float *__restrict__ y, const float *__restrict__ ws,
                                                    const float *res, float *out,
                                                    const fk_gemv_routed_combine_params &p) {
  const uint32_t i = blockIdx.x * (blockDim.x / FK_WAVE) + threadIdx.x / FK_WAVE;
  if (i >= p.n) return;
  // (lanes' packs in flight: at most 8 of all ranks; the host refuses more)
  if (p.k / P > FK_WAVE * 2) {
    if (p.ranks == 1) routed_rows<WT, P, 1, 4>(table, ids, x, y, ws, res, out, p, i);
    else routed_rows<WT, P, 2, 4>(table, ids, x, y, ws, res, out, p, i);
  } else {
    if (p.ranks == 1) routed_rows<WT, P, 1, 2>(table, ids, x, y, ws, res, out, p, i);
    else if (p.ranks == 2) routed_rows<WT, P, 2, 2>(table, ids, x, y, ws, res, out, p, i);
    else if (p.ranks == 3) routed_rows<WT, P, 3, 2>(table, ids, x, y, ws, res, out, p, i);
    else routed_rows<WT, P, 4, 2>(table, ids, x, y, ws, res, out, p, i);
  }
}

}  // namespace fk

#define FK_ROUTED_ENTRIES(TYPE, WT, P)                                                                              \
  extern "C" __global__ void __launch_bounds__(256)                                                                 \
      fk_gemv_routed_act_##TYPE(const uint64_t *__restrict__ table, const uint32_t *__restrict__ ids,               \
                                const float *__restrict__ x, float *__restrict__ y, float *__restrict__ out,        \
                                fk_gemv_routed_act_params p) {                                                      \
    fk::gemv_routed_act<WT, P>(table, ids, x, y, out, p);                                                           \
  }                                                                                                                 \
  extern "C" __global__ void __launch_bounds__(256)                                                                 \
      fk_gemv_routed_combine_##TYPE(const uint64_t *__restrict__ table, const uint32_t *__restrict__ ids,           \
                                    const float *__restrict__ x, float *__restrict__ y,                             \
                                    const float *__restrict__ w, const float *res, float *out,                      \
                                    fk_gemv_routed_combine_params p) {                                              \
    fk::gemv_routed_combine<WT, P>(table, ids, x, y, w, res, out, p);                                               \
  }
FK_ROUTED_ENTRIES(f16, _Float16, 8)
FK_ROUTED_ENTRIES(bf16, fk::bf16_t, 8)
FK_ROUTED_ENTRIES(f32, float, 4)
