// fk_split_attend.h — the prefill attention (fk_attend.h)
// with a block's keys split among KS groups of H wavefronts, for
// steps of too few (query block, head) pairs to fill the chip: one wavefront
// walking all of a pair's keys takes about 0.9 µs a block of 64 however few
// there are (512 rows after 3072 positions, 32 heads: 128 threadgroups, 52 µs
// a launch, and 26 in 256 threadgroups of 2 heads and 4 groups).  LDS bounds KS: 32 KB a group.
// Where each (H, KS) is taken: kernels.py's attend_launch.  (Bounds of two
// wavefronts a SIMD: within 256 registers the compiler takes the matrix
// operations' VGPR form; H = 1, whose LDS leaves one a SIMD, keeps AGPRs.)
#pragma once

#include "fk_attend.h"

#define FK_SPLIT_ATTEND(H, KS)                                                                                    \
  extern "C" __global__ void __launch_bounds__(64 * H * KS, 2) fk_split_attend_h##H##k##KS(                         \
      const uint16_t *__restrict__ qr, const uint16_t *__restrict__ kc, const uint16_t *__restrict__ vc,         \
      const uint32_t *__restrict__ position, const uint32_t *__restrict__ slot, uint16_t *__restrict__ out,     \
      const uint16_t *__restrict__ ks, const uint16_t *__restrict__ vs, fk_prefill_attend_params p) {            \
    prefill_attend<H, false, false, KS>(qr, kc, vc, position, slot, out, ks, vs, p);                             \
  }                                                                                                               \
  extern "C" __global__ void __launch_bounds__(64 * H * KS, 2) fk_split_attend_f16_h##H##k##KS(                     \
      const uint16_t *__restrict__ qr, const uint16_t *__restrict__ kc, const uint16_t *__restrict__ vc,         \
      const uint32_t *__restrict__ position, const uint32_t *__restrict__ slot, uint16_t *__restrict__ out,     \
      const uint16_t *__restrict__ ks, const uint16_t *__restrict__ vs, fk_prefill_attend_params p) {            \
    prefill_attend<H, false, true, KS>(qr, kc, vc, position, slot, out, nullptr, nullptr, p);                    \
  }                                                                                                               \
  extern "C" __global__ void __launch_bounds__(64 * H * KS, 2) fk_split_attend_paged_h##H##k##KS(                   \
      const uint16_t *__restrict__ qr, const uint16_t *__restrict__ kc, const uint16_t *__restrict__ vc,         \
      const uint32_t *__restrict__ position, const uint32_t *__restrict__ table, uint16_t *__restrict__ out,     \
      fk_prefill_attend_paged_params p) {                                                                        \
    prefill_attend<H, true, false, KS>(qr, kc, vc, position, table, out, nullptr, nullptr, p.a, p.g);            \
  }                                                                                                               \
  extern "C" __global__ void __launch_bounds__(64 * H * KS, 2) fk_split_attend_paged_f16_h##H##k##KS(               \
      const uint16_t *__restrict__ qr, const uint16_t *__restrict__ kc, const uint16_t *__restrict__ vc,         \
      const uint32_t *__restrict__ position, const uint32_t *__restrict__ table, uint16_t *__restrict__ out,     \
      fk_prefill_attend_paged_params p) {                                                                        \
    prefill_attend<H, true, true, KS>(qr, kc, vc, position, table, out, nullptr, nullptr, p.a, p.g);             \
  }
FK_SPLIT_ATTEND(4, 2)
FK_SPLIT_ATTEND(2, 2)
FK_SPLIT_ATTEND(1, 2)
FK_SPLIT_ATTEND(2, 4)
FK_SPLIT_ATTEND(1, 4)
