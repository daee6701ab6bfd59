"""Softmax of few rows by four threads for one (fk_softmax_f32_wide), against
fk_softmax_f32 on the same rows, bit for bit, at the widths where its forms
meet and with rows of infinities, zeros and NaNs; and against the oracle."""

import numpy as np
import pytest

from furykernel_amd import kernels as K
from oracle import fkref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2052, 4092, 4096, 4100, 8192, 8196, 12288, 16380, 16384])
def test_softmax_wide_bit_exact(device, kernels, n):
    rng = np.random.default_rng(n)
    rows = 9
    x = rng.normal(0, 3, (rows, n)).astype(np.float32)
    x[1] = 0.0
    x[2, n - 1] = 80.0
    x[3, : n // 2] = -np.inf
    x[4] = -np.inf
    x[5, 7] = np.nan
    x[6, 3] = np.inf
    x[7, :4] = np.finfo(np.float32).min
    bx, by, bz = device.upload(x), device.alloc(x.nbytes), device.alloc(x.nbytes)
    print(f"softmax {rows}x{n}", flush=True)
    kernels.softmax(bx, by, rows, n)
    kernels.launch("fk_softmax_f32", rows, 256, {"x": bx.ptr, "y": bz.ptr}, K.SoftmaxParams(rows, n))
    device.sync()
    got, apart = by.read(np.float32).reshape(rows, n), bz.read(np.float32).reshape(rows, n)
    for b in (bx, by, bz):
        b.free()
    nan = np.isnan(apart)
    assert np.array_equal(np.isnan(got), nan)
    assert np.array_equal(got.view(np.uint32)[~nan], apart.view(np.uint32)[~nan])
    want = fkref.softmax(x[:3], threads=256, width=64, pack=4)
    assert np.max(np.abs(got[:3].view(np.int32).astype(np.int64) - want.view(np.int32))) <= 2
