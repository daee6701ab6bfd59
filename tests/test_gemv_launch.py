"""The launch of a standalone matvec (kernels.gemv_launch), on the CPU: in
threadgroups of the caller's threads, its entry one that holds its rows,
covering every row once; and what the launch check refuses."""

import ctypes

import pytest

from furykernel_amd import kernels as K, runtime
from furykernel_amd.tuning import gemv_space, variants
from furykernel_amd.variant import Profile


@pytest.mark.parametrize("wtype", ["f32", "f16", "i8"])
@pytest.mark.parametrize("threads", [64, 128, 192, 256])
def test_every_launch_passes_the_checks(wtype, threads):
    pack = K.GEMV_PACK[wtype]
    for r in (1, 2, 4):
        for n in (1, 37, 4095, 4096):
            for k in (pack, 1024, 1024 + pack, 1800, 2048, 4096, 4096 + pack, 8192, 16384, 16384 + pack):
                k = k // pack * pack
                entry, groups, lds = K.gemv_launch(wtype, n, k, r, threads)
                abi = K.ABIS[entry]
                assert abi.threads in (0, threads)      # the caller's threads, always
                rows = threads // 64 * r
                assert (groups - 1) * rows < n <= groups * rows
                sizes = {"w": n * k * K.ELEM_BYTES[wtype], "x": k * (2 if wtype == "i8" else 4), "y": n * 4,
                         "scale": n * 4}
                spans = [((i + 1) << 40, sizes[b]) for i, b in enumerate(abi.buffers)]
                runtime.launch_check(entry, groups, threads, lds, spans, K.GemvParams(n, k))


def test_x_is_staged_in_threadgroups_of_256_alone():
    for t in (64, 128, 192):
        assert K.gemv_launch("f16", 4096, 4096, 1, t) == ("fk_gemv_f16_f32_r1", 4096 // (t // 64) + (t == 192), 0)
    assert K.gemv_launch("f16", 4096, 4096, 1, 256)[0] == "fk_gemv_f16_f32_staged_r1"
    assert K.gemv_launch("f16", 4096, 8192, 1, 256)[0] == "fk_gemv_f16_f32_wide"
    assert K.gemv_launch("f16", 4095, 8192, 1, 256)[0] == "fk_gemv_f16_f32_r1"
    assert K.gemv_launch("f32", 4096, 8192, 1, 256)[0] == "fk_gemv_f32_f32_r1"
    assert K.gemv_launch("f16", 16384, 2048, 4, 256)[0] == "fk_gemv_f16_f32_r4"


@pytest.mark.parametrize("wtype", ["f32", "f16", "i8"])
def test_tuning_times_what_a_call_launches(wtype):
    space = gemv_space(wtype)
    for shape in space.shapes:
        n, k = dict(shape)["n"], dict(shape)["k"]
        seen = set()
        for v in variants(Profile(256), space, shape):
            r, t = (dict(v.point)[a] for a in "rt")
            L = v.launch
            assert (L.entry, L.groups, L.lds_bytes) == K.gemv_launch(wtype, n, k, r, t) and L.threads == t
            seen.add(t)
        assert seen == {64, 128, 256}


def test_staged_entries_refuse_rows_they_cannot_hold():
    for entry, held in (("fk_gemv_f32_f32_staged_r1", 4096), ("fk_gemv_f32_f32_staged_r4", 1024),
                        ("fk_gemv_f16_f32_staged_r2", 4096), ("fk_gemv_f16_f32_staged_r4", 2048)):
        r, eb = int(entry[-1]), 4 if "_f32_f32" in entry else 2
        for k, groups, threads in ((held, 8, 256), (held + 8, 8, 256), (held, 1, 256), (held, 8, 128)):
            n = 20
            spans = [(1 << 40, n * k * eb), (2 << 40, k * 4), (3 << 40, n * 4)]
            args = (entry, groups, threads, 0, spans, K.GemvParams(n, k))
            if k == held and groups * 4 * r >= n and threads == 256:
                runtime.launch_check(*args)
            else:
                with pytest.raises(runtime.FkError):
                    runtime.launch_check(*args)
    assert ctypes.sizeof(K.GemvParams) == 8


def test_the_wide_softmax_refuses_rows_it_cannot_hold():
    """It holds 16 elements a thread; a longer row would be summed and stored
    short."""
    def check(rows, n, groups, threads=1024, short=0):
        spans = [(1 << 40, rows * n * 4), (2 << 40, rows * n * 4 - short)]
        runtime.launch_check("fk_softmax_f32_wide", groups, threads, 0, spans, K.SoftmaxParams(rows, n))
    check(3, 16384, 3)
    check(3, 4, 3)
    for bad in ((3, 16388, 3), (3, 32768, 3), (3, 4098, 3), (3, 4096, 2), (3, 4096, 3, 512), (3, 4096, 3, 1024, 4)):
        with pytest.raises(runtime.FkError):
            check(*bad)
