"""The small probabilities of the attention of a batch of rows
(fk_rows_attend.h) on the GPU: keys whose weights are 2^-24.5 of the largest,
and whose values are all that the output is made of.  The prefill attention
keeps them to 2^-8, its reference lying up to 8 (log2 units) below the
maximum; so they are kept here, in one part and several."""

import numpy as np
import pytest

from furykernel_amd import kernels as K
from furykernel_amd.layout import unpack

pytestmark = pytest.mark.gpu
LENGTH = 512


def inputs():
    """Scores 0 for the first tile's keys, then one of 7.5 and the rest of its
    wavefront's 63 at -17 (log2 units, as f16 rounds them), with values of
    60000 where the others have 0."""
    s = np.zeros(LENGTH, np.float64)
    s[256], s[257:320] = 7.5, -17.0
    k = np.zeros((1, 1, LENGTH, 64), np.float16)
    k[0, 0, :, 0] = s * np.log(2)
    v = np.zeros((1, 1, LENGTH, 64), np.float16)
    v[0, 0, 257:320] = 60000
    score = k[0, 0, :, 0].astype(np.float64)
    e = np.exp(score - score.max())
    return k, v, (e / e.sum()) @ v[0, 0].astype(np.float64)


@pytest.mark.parametrize("parts", [1, 2])
def test_small_probabilities_keep_their_bits(device, kernels, parts):
    k, v, want = inputs()
    q = np.zeros((256, 64), np.float16)
    q[0, 0] = 1
    pos = np.full(256, LENGTH - 1, np.uint32)
    bufs = [device.upload(x) for x in (q, k, v, pos, np.zeros(256, np.uint32), np.zeros(256 * 64, np.float16))]
    part = device.alloc(parts * 66 * 4)
    p = K.RowsAttendParams(1, 32, 1, 1, LENGTH, 1, 0, parts, 0, 1.0)
    bind = dict(zip(("qr", "kc", "vc", "position", "slot", "out"), [b.ptr for b in bufs]), partials=part.ptr)
    print(f"rows attend, small probabilities, {parts} parts", flush=True)
    kernels.launch("fk_rows_attend_f16", parts, 256, bind, p)
    if parts > 1:
        kernels.launch("fk_rows_combine", 1, 64, {n: bind[n] for n in ("partials", "position", "out")}, p)
    device.sync()
    got = unpack(bufs[5].read(np.float16), 256, 64).astype(np.float64)[0]
    for b in (*bufs, part):
        b.free()
    # f16 probabilities of 2^-16.5: half a unit of 2^-24 is 2^-8.5 of them;
    # the output's own rounding 2^-11
    assert np.all(np.abs(got - want) <= np.abs(want) * (2.0**-8 + 2.0**-10)), (got[0], want[0])
