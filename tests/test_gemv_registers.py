"""The registers of the matvec kernels that keep a whole row's loads in
flight, from the built code object: past 128 a SIMD holds three wavefronts
where it held four, invisible to every numeric test."""

import pytest

from test_code_objects import metadata  # noqa: F401  (the fixture)


@pytest.mark.parametrize("entry", ["fk_gemv_routed_f32_r1", "fk_gemv_routed_f16_r1", "fk_gemv_routed_bf16_r1",
                                   "fk_gemv_f32_f32_r1", "fk_gemv_f16_f32_r1", "fk_gemv_f32_f32_staged_r1"])
def test_a_row_a_wavefront_leaves_four_wavefronts_a_simd(metadata, entry):  # noqa: F811
    assert metadata[entry][".vgpr_count"] <= 128
    assert metadata[entry][".vgpr_spill_count"] == 0
