"""The standalone matvecs at the widths where their forms meet (a lane's
packs at and past 1, 2, 4, 8 and 16, rows that end inside a pack's lane, rows
wider than a lane holds), with fewer rows than a threadgroup's and in smaller
threadgroups: bit for bit the oracle, y past n left as it was."""

import numpy as np
import pytest

from furykernel_amd.kernels import GEMV_PACK
from oracle import fkref

pytestmark = pytest.mark.gpu

PACKS = [1, 63, 64, 65, 128, 129, 193, 256, 257, 385, 511, 512, 513, 1023, 1024, 1025]


def bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


@pytest.mark.parametrize("wtype", ["f32", "f16", "i8"])
@pytest.mark.parametrize("r,threads", [(1, 256), (2, 256), (4, 256), (1, 64), (2, 192)])
def test_gemv_widths(device, kernels, wtype, r, threads):
    rng = np.random.default_rng(100 * r + threads)
    pack = GEMV_PACK[wtype]
    for packs in PACKS:
        n, k = 21, packs * pack
        scale = None
        if wtype == "i8":
            w = rng.integers(-128, 128, (n, k)).astype(np.int8)
            x = rng.normal(0, 1, k).astype(np.float16)
            scale = rng.uniform(0.001, 0.01, n).astype(np.float32)
        else:
            w = rng.normal(0, 1, (n, k)).astype(np.float32 if wtype == "f32" else np.float16)
            x = rng.normal(0, 1, k).astype(np.float32)
        bw, bx, by = device.upload(w), device.upload(x), device.upload(np.full(n + 43, 7.0, np.float32))
        bs = None if scale is None else device.upload(scale)
        print(f"gemv {wtype} {n}x{k} r{r} {threads} threads", flush=True)
        kernels.gemv(bw, bx, by, n, k, wtype=wtype, rows_per_wave=r, threads=threads, scale=bs)
        device.sync()
        out = by.read(np.float32, n + 43)
        for b in (bw, bx, by, bs):
            if b is not None:
                b.free()
        kw = {} if scale is None else {"row_scale": scale}
        assert np.array_equal(bits(out[:n]), bits(fkref.gemv(w, x, 64, pack, 1, **kw))), k
        assert np.all(out[n:] == 7.0), k


@pytest.mark.parametrize("n,k", [(4096, 4104), (4099, 4608), (4097, 8184), (4096, 16384), (4095, 4104), (4096, 16392)])
def test_gemv_f16_wide_rows(device, kernels, n, k):
    """Rows wider than a wavefront holds, on both sides of what takes x
    through LDS whole: bit for bit the oracle on the first and last rows."""
    rng = np.random.default_rng(n + k)
    w = rng.integers(-512, 512, (n, k), dtype=np.int16).astype(np.float16) / np.float16(256)
    x = rng.normal(0, 1, k).astype(np.float32)
    bw, bx, by = device.upload(w), device.upload(x), device.upload(np.full(n + 3, 7.0, np.float32))
    print(f"gemv f16 {n}x{k}", flush=True)
    kernels.gemv(bw, bx, by, n, k, wtype="f16")
    device.sync()
    out = by.read(np.float32, n + 3)
    for b in (bw, bx, by):
        b.free()
    rows = np.r_[0:70, n - 70:n]
    assert np.array_equal(bits(out[rows]), bits(fkref.gemv(np.ascontiguousarray(w[rows]), x, 64, 8, 1)))
    assert np.all(out[n:] == 7.0)
