"""Each form of the few-row GEMM (fk_skinny.h) is one that some size takes
(prefill.skinny_form), on the CPU: a form that none does would be built,
tested and never run."""

import pytest

from furykernel_amd import kernels as K
from furykernel_amd.prefill import SKINNY_COST, skinny_form


def test_every_form_is_taken():
    taken = set()
    for chunks in range(1, 129):
        m = -(-chunks // 16) * 256
        for n, k, mode in ((2048, 8192, "add"), (2048, 2048, "add"), (16384, 2048, "silu_mul"), (3072, 2048, "qkv_rope"),
                           (32000, 2048, "store_keys")):
            picked = skinny_form(chunks, m, n, k, mode, (1, 2, 4, 8) if mode == "add" else (1,))
            taken |= {picked[0]} if picked else set()
    assert taken == set(K.SKINNY_FORMS) == set(SKINNY_COST)


@pytest.mark.parametrize("rows, n, k, mode, slower", [
    (2048, 2 * 2048, 4096, "silu_mul", "m8n8"),
    (1408, 2 * 2048, 4096, "silu_mul", "m8n8"),
    (256, 2 * 12288, 4096, "silu_mul", "m4n8"),
    (1408, 4096, 4096, "store_keys", "m8n8"),
    (2048, 4096, 4096, "store_keys", "m8n8"),
])
def test_a_form_slower_than_the_whole_tiles_is_not_taken(rows, n, k, mode, slower):
    """The form that each measured slower there than fk_gemm's tiles."""
    picked = skinny_form(-(-rows // 16), -(-rows // 256) * 256, n, k, mode)
    assert picked is None or picked[0] != slower
