"""The prefill attention with its keys split among groups of wavefronts
(fk_split_attend.h) on the GPU, every form, against binary64 attention of the
same values: fewer key blocks than groups, group counts that do not divide
them, a prompt's first rows and a later chunk, windows.

The bar is the f16 one of the other prefill tests: 2e-3 of the largest
magnitude.
"""

import numpy as np
import pytest

from furykernel_amd import kernels as K
from furykernel_amd.layout import unpack

pytestmark = pytest.mark.gpu
BAR = 2e-3
LENGTH, BLOCK = 768, 32


def attend(device, kernels, entry, h, starts, window=0, seed=3):
    """256 rows, 128 of each of two sequences from `starts`, two kv heads of 4
    query heads."""
    rng = np.random.default_rng(seed)
    g = 4
    kvh, rows, slots = 2, 256, 3
    heads = kvh * g
    paged, bf16 = "_paged_" in entry, "_f16_" not in entry
    q = rng.standard_normal((rows, heads * 64)).astype(np.float16)
    kv = [rng.standard_normal((slots, kvh, LENGTH, 64)).astype(np.float32) for _ in range(2)]
    bits = [(x.view(np.uint32) >> 16).astype(np.uint16) if bf16 else x.astype(np.float16).view(np.uint16) for x in kv]
    wide = [((b.astype(np.uint32) << 16).view(np.float32) if bf16 else b.view(np.float16)).astype(np.float64)
            for b in bits]
    pos = np.concatenate([np.arange(s, s + 128) for s in starts]).astype(np.uint32)
    slot = np.repeat([2, 0], 128).astype(np.uint32)
    base = dict(rows=rows, heads=heads, kv_heads=kvh, length=LENGTH, slots=slots, window=window, cache_bf16=int(bf16),
                scale=0.125, run_rows=128)
    if paged:
        per = LENGTH // BLOCK
        order = rng.permutation(slots * per).reshape(slots, per).astype(np.uint32)
        for i, b in enumerate(bits):
            pool = np.empty((slots * per, kvh, BLOCK, 64), np.uint16)
            pool[order] = b.reshape(slots, kvh, per, BLOCK, 64).transpose(0, 2, 1, 3, 4)
            bits[i] = pool
        where = order[slot]
        p = K.PrefillAttendPagedParams(**base, block_size=BLOCK, table_len=per, blocks=slots * per)
    else:
        where, p = slot, K.PrefillAttendParams(**base)
    bufs = [device.upload(x) for x in (q, *bits, pos, where)]
    out = device.alloc(rows * heads * 128)
    bind = dict(zip(("qr", "kc", "vc", "position", "table" if paged else "slot"), [b.ptr for b in bufs]), out=out.ptr,
                ks=0, vs=0)
    print(f"{entry} starts {starts} window {window}", flush=True)
    kernels.launch(entry, rows // 32 * heads // h, K.ATTEND_FORMS[entry], bind, p)
    device.sync()
    got = unpack(out.read(np.float16), rows, heads * 64).astype(np.float64).reshape(rows, heads, 64)
    for b in (*bufs, out):
        b.free()
    for r in range(0, rows, 5):
        ts = slice(max(0, int(pos[r]) + 1 - window) if window else 0, int(pos[r]) + 1)
        for head in range(heads):
            kk, vv = (x[slot[r], head // g, ts] for x in wide)
            s = 0.125 * (kk @ q[r, head * 64:(head + 1) * 64].astype(np.float64))
            e = np.exp(s - s.max())
            want = (e / e.sum()) @ vv
            assert np.max(np.abs(got[r, head] - want)) <= BAR * max(1.0, np.max(np.abs(want))), (r, head)


FORMS = [(f"fk_split_attend_{form}h{h}k{k}", h) for form in ("", "f16_", "paged_", "paged_f16_")
         for h, k in K.ATTEND_SPLITS]


@pytest.mark.parametrize("entry,h", FORMS, ids=lambda x: str(x))
def test_every_form(device, kernels, entry, h):
    attend(device, kernels, entry, h, (0, 77))      # 1 to 4 blocks of keys
    attend(device, kernels, entry, h, (640, 512))   # up to the ring's end


@pytest.mark.parametrize("entry,h", [f for f in FORMS if "f16" in f[0]], ids=lambda x: str(x))
def test_windows(device, kernels, entry, h):
    attend(device, kernels, entry, h, (500, 300), window=48)
    attend(device, kernels, entry, h, (500, 300), window=200)


@pytest.mark.parametrize("rows,heads,kvh", [(256, 32, 8), (512, 32, 8), (1024, 32, 8), (512, 8, 8), (1536, 32, 8)])
def test_the_launcher_takes_them(device, kernels, rows, heads, kvh):
    """kernels.prefill_attend where it splits, sampled rows."""
    entry, groups, threads = K.attend_launch("f16_", rows, heads, kvh, 2048)
    assert "split" in entry and threads == K.ATTEND_FORMS[entry]
    rng = np.random.default_rng(8)
    q = rng.standard_normal((rows, heads * 64)).astype(np.float16)
    kc, vc = (rng.standard_normal((1, kvh, 2048, 64)).astype(np.float16) for _ in range(2))
    pos = np.arange(2048 - rows, 2048).astype(np.uint32)
    bufs = [device.upload(x) for x in (q, kc, vc, pos, np.zeros(rows, np.uint32))]
    out = device.alloc(rows * heads * 128)
    kernels.prefill_attend(*bufs, out, rows, heads, kvh, 2048, 1, 0.125, positions=pos, seqs=np.zeros(rows, int))
    device.sync()
    got = unpack(out.read(np.float16), rows, heads * 64).astype(np.float64).reshape(rows, heads, 64)
    for r in (0, 1, 31, 32, rows // 2 + 7, rows - 1):
        for head in range(0, heads, 3):
            kk, vv = (x[0, head // (heads // kvh), :pos[r] + 1].astype(np.float64) for x in (kc, vc))
            s = 0.125 * (kk @ q[r, head * 64:(head + 1) * 64].astype(np.float64))
            e = np.exp(s - s.max())
            want = (e / e.sum()) @ vv
            assert np.max(np.abs(got[r, head] - want)) <= BAR, (r, head)
    for b in (*bufs, out):
        b.free()
