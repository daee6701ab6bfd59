// fk_gemv_staged.h — the f32 and f16 matvecs' entries with x staged in LDS
// (fk_gemv.h: gemv_xlds, gemv_staged).  Last in the code object: ahead of the
// step kernels, the addresses that those then had cost the 1B decode step 2 µs
// of 624, their code byte for byte the same.
#pragma once

#include "fk_gemv.h"

// Threadgroups of 256, rows of at most 64 KPL packs: the same sums as the
// entries of any threadgroup.  (Apart from those: beside their form the f16 row
// would keep 110 registers where it needs 80.  Smaller threadgroups would stage
// x more often for the same rows: f16 4096 x 4096 of 64 threads 11.6 µs staged,
// 7.9 from memory; of 256, 7.2 and 7.9.)
#define FK_GEMV_STAGED_ENTRY(NAME, WT, XT, P, R, KPL)                                                        \
  extern "C" __global__ void __launch_bounds__(256) NAME(const WT *__restrict__ w, const XT *__restrict__ x, \
                                                         float *__restrict__ y, fk_gemv_params p) {         \
    __shared__ uint4 xs[FK_WAVE * (KPL) * (P) * sizeof(XT) / 16];                                           \
    static_assert(sizeof xs >= 256 * 16, "a chunk a thread");                                               \
    const uint32_t row0 = (blockIdx.x * 4 + threadIdx.x / FK_WAVE) * (R);                                   \
    if (p.k == FK_WAVE * (KPL) * (P))                                                                       \
      fk::gemv_xlds<WT, XT, P, R, KPL, true, 256>(w, x, nullptr, y, p.n, p.k, row0, xs);                   \
    else                                                                                                     \
      fk::gemv_staged<WT, XT, P, R, KPL>(w, x, nullptr, y, p.n, p.k, row0, xs);                             \
  }

FK_GEMV_STAGED_ENTRY(fk_gemv_f32_f32_staged_r1, float, float, 4, 1, 16)
FK_GEMV_STAGED_ENTRY(fk_gemv_f32_f32_staged_r2, float, float, 4, 2, 16)
FK_GEMV_STAGED_ENTRY(fk_gemv_f32_f32_staged_r4, float, float, 4, 4, 4)
FK_GEMV_STAGED_ENTRY(fk_gemv_f16_f32_staged_r1, _Float16, float, 8, 1, 8)
FK_GEMV_STAGED_ENTRY(fk_gemv_f16_f32_staged_r2, _Float16, float, 8, 2, 8)
FK_GEMV_STAGED_ENTRY(fk_gemv_f16_f32_staged_r4, _Float16, float, 8, 4, 4)
