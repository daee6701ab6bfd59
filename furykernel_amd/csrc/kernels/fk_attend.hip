// fk_attend.hip — the translation unit of the prefill attention, compiled
// into fk_attend.hsaco (see fk_attend.h for why it is apart).
#include "fk_attend.h"

// One entry a group size G = heads / kv_heads (threads 64 G).
#define FK_PREFILL_ATTEND(G)                                                                                    \
  extern "C" __global__ void __launch_bounds__(64 * G) fk_prefill_attend_g##G(                         \
      const uint16_t *__restrict__ qr, const uint16_t *__restrict__ kc, const uint16_t *__restrict__ vc,       \
      const uint32_t *__restrict__ position, const uint32_t *__restrict__ slot, uint16_t *__restrict__ out,   \
      const uint16_t *__restrict__ ks, const uint16_t *__restrict__ vs, fk_prefill_attend_params p) {          \
    prefill_attend<G>(qr, kc, vc, position, slot, out, ks, vs, p);                                              \
  }
FK_PREFILL_ATTEND(1)
FK_PREFILL_ATTEND(2)
FK_PREFILL_ATTEND(4)

// The same over f16 rings with no staged rows, each block's rows loaded
// straight into LDS (the same bindings; ks and vs unused).
#define FK_PREFILL_ATTEND_F16(G)                                                                                \
  extern "C" __global__ void __launch_bounds__(64 * G) fk_prefill_attend_f16_g##G(                     \
      const uint16_t *__restrict__ qr, const uint16_t *__restrict__ kc, const uint16_t *__restrict__ vc,       \
      const uint32_t *__restrict__ position, const uint32_t *__restrict__ slot, uint16_t *__restrict__ out,   \
      const uint16_t *__restrict__ ks, const uint16_t *__restrict__ vs, fk_prefill_attend_params p) {          \
    prefill_attend<G, false, true>(qr, kc, vc, position, slot, out, nullptr, nullptr, p);                      \
  }
FK_PREFILL_ATTEND_F16(1)
FK_PREFILL_ATTEND_F16(2)
FK_PREFILL_ATTEND_F16(4)

// The same over paged pools: kc and vc the pools, `table` the rows' block
// tables; no staged rows.
#define FK_PREFILL_ATTEND_PAGED(G)                                                                                \
  extern "C" __global__ void __launch_bounds__(64 * G) fk_prefill_attend_paged_g##G(                             \
      const uint16_t *__restrict__ qr, const uint16_t *__restrict__ kc, const uint16_t *__restrict__ vc,         \
      const uint32_t *__restrict__ position, const uint32_t *__restrict__ table, uint16_t *__restrict__ out,     \
      fk_prefill_attend_paged_params p) {                                                                        \
    prefill_attend<G, true>(qr, kc, vc, position, table, out, nullptr, nullptr, p.a, p.g);                       \
  }
FK_PREFILL_ATTEND_PAGED(1)
FK_PREFILL_ATTEND_PAGED(2)
FK_PREFILL_ATTEND_PAGED(4)

// The same over f16 pools (under 4 GiB, tables of at most FK_ATT_TABLE
// blocks), each block's rows loaded straight into LDS.
#define FK_PREFILL_ATTEND_PAGED_F16(G)                                                                            \
  extern "C" __global__ void __launch_bounds__(64 * G) fk_prefill_attend_paged_f16_g##G(                         \
      const uint16_t *__restrict__ qr, const uint16_t *__restrict__ kc, const uint16_t *__restrict__ vc,         \
      const uint32_t *__restrict__ position, const uint32_t *__restrict__ table, uint16_t *__restrict__ out,     \
      fk_prefill_attend_paged_params p) {                                                                        \
    prefill_attend<G, true, true>(qr, kc, vc, position, table, out, nullptr, nullptr, p.a, p.g);                 \
  }
FK_PREFILL_ATTEND_PAGED_F16(1)
FK_PREFILL_ATTEND_PAGED_F16(2)
FK_PREFILL_ATTEND_PAGED_F16(4)
