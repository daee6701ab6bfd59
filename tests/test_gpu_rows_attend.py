"""The attention of a batch of rows, each a sequence's one (fk_rows_attend.h),
on the GPU against binary64 attention of the same f16 (bf16) values: rows at
the edges of a wavefront's 64 keys and of a tile's 256, the first and the last
of the ring, one part and several, group sizes of 1 to 16 heads, windows that
start inside and between tiles.

The bound: probabilities are f16 (2^-11 each, of weights that sum to 1), so a
row's error is within 2^-10 of the largest |V| it can reach plus the output's
own f16 rounding; the scores' binary32 sums and exp2 add less than 2^-16.
"""

import numpy as np
import pytest

from furykernel_amd import kernels as K
from furykernel_amd.layout import unpack

pytestmark = pytest.mark.gpu
APART = 32


def attend(device, kernels, heads, kvh, length, positions, parts, window=0, bf16=False, scale=0.125, seed=5):
    rng = np.random.default_rng(seed)
    rows = len(positions)
    m = -(-rows * APART // 256) * 256
    slots = rows + 1
    slot = rng.permutation(slots)[:rows].astype(np.uint32)
    q = rng.standard_normal((m, heads * 64)).astype(np.float16)
    kv = [rng.standard_normal((slots, kvh, length, 64)).astype(np.float32) for _ in range(2)]
    bits = [(x.view(np.uint32) >> 16).astype(np.uint16) if bf16 else x.astype(np.float16).view(np.uint16) for x in kv]
    wide = [((b.astype(np.uint32) << 16).view(np.float32) if bf16 else b.view(np.float16)).astype(np.float64)
            for b in bits]
    pos, sl = np.zeros(m, np.uint32), np.zeros(m, np.uint32)
    pos[:rows * APART:APART], sl[:rows * APART:APART] = positions, slot
    bufs = [device.upload(x) for x in (q, *bits, pos, sl, np.full(m * heads * 64, 3.0, np.float16))]
    part = device.alloc(rows * heads * parts * 66 * 4)
    p = K.RowsAttendParams(rows, APART, heads, kvh, length, slots, window, parts, 0, scale)
    names = ("qr", "kc", "vc", "position", "slot", "out")
    bind = dict({n: b.ptr for n, b in zip(names, bufs)}, partials=part.ptr)
    print(f"rows attend {heads}/{kvh} length {length} rows {rows} parts {parts} window {window}", flush=True)
    try:
        kernels.launch(f"fk_rows_attend_{'bf16' if bf16 else 'f16'}", rows * kvh * parts, 256, bind, p)
        if parts > 1:
            kernels.launch("fk_rows_combine", rows * kvh, 64 * heads // kvh,
                           {n: bind[n] for n in ("partials", "position", "out")}, p)
        device.sync()
        got = unpack(bufs[5].read(np.float16), m, heads * 64).astype(np.float64)
    finally:
        for b in (*bufs, part):
            b.free()
    live = np.arange(rows) * APART
    assert np.all(np.delete(got, live, axis=0) == 3.0)   # the filling rows are left
    for i, at in enumerate(positions):
        ts = slice(max(0, at + 1 - window) if window else 0, at + 1)
        for h in range(heads):
            kk, vv = (x[slot[i], h // (heads // kvh), ts] for x in wide)
            s = scale * (kk @ q[live[i], h * 64:(h + 1) * 64].astype(np.float64))
            e = np.exp(s - s.max())
            want = (e / e.sum()) @ vv
            bar = 2.0**-10 * np.abs(vv).max() + np.abs(want) * 2.0**-11
            assert np.all(np.abs(got[live[i], h * 64:(h + 1) * 64] - want) <= bar), (at, h)


EDGES = [0, 1, 62, 63, 64, 255, 256, 257, 319, 511, 512, 767, 1023]


@pytest.mark.parametrize("parts", [1, 3, 4])
def test_rows_at_the_edges_of_tiles(device, kernels, parts):
    attend(device, kernels, 8, 2, 1024, EDGES, parts)


@pytest.mark.parametrize("heads,kvh", [(2, 2), (4, 2), (16, 1), (12, 4)])
def test_groups_of_heads(device, kernels, heads, kvh):
    attend(device, kernels, heads, kvh, 512, [5, 300, 511], 2)


@pytest.mark.parametrize("window", [1, 48, 64, 300])
def test_windows(device, kernels, window):
    attend(device, kernels, 4, 2, 1024, EDGES, 4, window=window)


@pytest.mark.parametrize("parts", [1, 2])
def test_bf16_rings(device, kernels, parts):
    attend(device, kernels, 8, 2, 512, [0, 100, 256, 511], parts, bf16=True)


def test_a_long_row_in_sixteen_parts(device, kernels):
    attend(device, kernels, 8, 2, 4096, [4095, 17, 2048], 16)


def test_one_row_and_large_scores(device, kernels):
    # scores of hundreds: the running maximum moves between tiles
    attend(device, kernels, 4, 1, 768, [767], 1, scale=8.0)
    attend(device, kernels, 4, 1, 768, [767], 3, scale=8.0)
