"""The GEMM of a step of few rows (fk_skinny.h) on the GPU against f64 sums of
its f16 operands, each form with each epilogue at the sizes where it can go
wrong: fewer steps of k than wavefronts, steps that the wavefronts do not
divide, chunks of rows that do not fill a tile, rows of runs and rows 32
apart, rows past the step's.

The bound of binary32 accumulation is fk_gemm's (test_gpu_gemm.bound); f16
and bf16 outputs round once more (2^-11, 2^-8 of the value).  Rows that are
not live are left as they were.
"""

import ctypes

import numpy as np
import pytest

from furykernel_amd import kernels as K
from furykernel_amd.layout import pack, pair, unpack
from furykernel_amd.lower import rope_table
from test_gpu_gemm import bound, f16, gelu_mul, silu_mul

pytestmark = pytest.mark.gpu
MARK = 777.0

# (m, live chunks, chunks a run, run, apart, k)
ROWS = [(256, 1, 1, 256, 1, 64), (256, 16, 16, 256, 1, 192), (512, 9, 9, 512, 1, 1088),
        (512, 10, 5, 256, 1, 320),            # two runs, 80 rows of each
        (256, 1, 1, 256, 32, 1024),           # 8 rows 32 apart, 8 more past the step
        (1536, 3, 3, 1536, 32, 576)]


def live_rows(m, live, run_chunks, run, apart):
    c = np.arange(live)
    first = (c // run_chunks) * run + (c % run_chunks) * 16 * apart
    rows = (first[:, None] + np.arange(16) * apart).reshape(-1)
    return rows[rows < m]


def launch(device, kernels, mode, form, shape, bs, cs, n, bind=None, **params):
    m, live, run_chunks, run, apart, k = shape
    mb, nb, waves = K.SKINNY_FORMS[form]
    params.setdefault("parts", 1)
    p = K.SkinnyParams(m=m, k=k, n_anchors=len(n), live=live, run_chunks=run_chunks, run=run, apart=apart, **params)
    first = np.concatenate([[0], np.cumsum(n)]).tolist()
    for i in range(4):
        p.first_col[i] = first[min(i, len(n))]
    for i, w in enumerate(n):
        p.ldc[i] = w
    tiles_n = (2 if mode == "silu_mul" else 1) * sum(n) // (16 * nb)
    bound_to = {b: 0 for b in K.SKINNY_BUFFERS}
    bound_to.update({f"b{i}": b.ptr for i, b in enumerate(bs)})
    bound_to.update({f"c{i}": c.ptr for i, c in enumerate(cs)})
    bound_to.update({name: b.ptr for name, b in (bind or {}).items()})
    print(f"skinny {mode} {form} {shape} {n}", flush=True)
    kernels.launch(f"fk_skinny_{mode}_{form}", -(-tiles_n // 8) * 8 * -(-live // mb) * params["parts"],
                   64 * waves, bound_to, p)
    device.sync()


FORMS = list(K.SKINNY_FORMS)
PAIRS = [f for f in FORMS if K.SKINNY_FORMS[f][1] > 1]


@pytest.mark.parametrize("shape", ROWS, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("form", FORMS)
def test_rows_within_the_accumulation_bound(device, kernels, form, shape):
    """The plain store (two anchors), the residual and the keys epilogues."""
    m, k = shape[0], shape[-1]
    live = live_rows(*shape[:-1])
    rest = np.setdiff1d(np.arange(m), live)
    a, ws = f16((m, k)), [f16((256, k)), f16((512, k))]
    r = np.random.default_rng(1).standard_normal((m, 256)).astype(np.float32)
    ba, bs = device.upload(pack(a)), [device.upload(pack(w)) for w in ws]
    cs = [device.upload(np.full((m, w.shape[0]), MARK, np.float32)) for w in ws]
    br = device.upload(r)
    parts = 512 // (16 * K.SKINNY_FORMS[form][1])
    bk = device.upload(np.full((m, parts), 5, np.uint64))
    exact = [a.astype(np.float64) @ w.astype(np.float64).T for w in ws]
    try:
        launch(device, kernels, "store", form, shape, bs, cs, [256, 512], {"a": ba})
        for c, w, e in zip(cs, ws, exact):
            got = c.read(np.float32).reshape(m, -1)
            assert np.all(np.abs(got - e)[live] <= bound(a, w)[live]) and np.all(got[rest] == MARK)
        # in place: the residual's rows are the output's
        launch(device, kernels, "add", form, shape, bs[:1], [br], [256], {"a": ba, "r0": br})
        got = br.read(np.float32).reshape(m, 256)
        want = r + exact[0]
        assert np.all(np.abs(got - want)[live] <= (bound(a, ws[0]) + np.abs(want) * 2.0**-24)[live])
        assert np.array_equal(got[rest], r[rest])
        launch(device, kernels, "store_keys", form, shape, bs[1:], cs[1:], [512], {"a": ba, "keys": bk})
        got, keys = cs[1].read(np.float32).reshape(m, 512), bk.read(np.uint64).reshape(m, parts)
        best = np.max(keys, axis=1)
        assert np.array_equal((0xFFFFFFFF - (best & 0xFFFFFFFF)).astype(np.int64)[live], np.argmax(got, axis=1)[live])
        assert np.all(keys[rest] == 5)
    finally:
        for b in [ba, br, bk, *bs, *cs]:
            b.free()


@pytest.mark.parametrize("act", [0, 1], ids=["silu", "gelu-tanh"])
@pytest.mark.parametrize("form", PAIRS)
def test_act_mul_writes_the_tile_layout(device, kernels, form, act):
    shape = ROWS[3]
    m, k = shape[0], shape[-1]
    live = live_rows(*shape[:-1])
    a, g, u = f16((m, k), 0.5), f16((256, k), 0.4), f16((256, k), 0.4)
    ba, bb = device.upload(pack(a)), device.upload(pack(pair(g, u)))
    bc = device.upload(np.full(m * 256, MARK, np.float16))
    try:
        launch(device, kernels, "silu_mul", form, shape, [bb], [bc], [256], {"a": ba}, act=act)
        got = unpack(bc.read(np.float16), m, 256).astype(np.float64)
        exact = (gelu_mul if act else silu_mul)(a, g, u)
        assert np.max(np.abs(got - exact)[live]) <= 2e-3 * np.max(np.abs(exact))
        assert np.all(np.delete(got, live, axis=0) == MARK)
    finally:
        for b in (ba, bb, bc):
            b.free()


@pytest.mark.parametrize("where", ["ring", "bf16 ring", "staged", "paged"])
@pytest.mark.parametrize("form", PAIRS)
def test_qkv_turns_and_stores_the_heads(device, kernels, form, where):
    """4 query heads over 4 kv heads: q in f16 rows, k and v in the caches at
    each row's place, every other element of the caches as it was."""
    shape = ROWS[5] if where == "ring" else ROWS[3]
    m, k = shape[0], shape[-1]
    live = live_rows(*shape[:-1])
    heads, length, slots, block = 4, 128, 17, 16
    rng = np.random.default_rng(3)
    pos = rng.integers(0, length, m).astype(np.uint32)
    # every live row its own place
    slot = (np.arange(m) % slots).astype(np.uint32)
    pos[live] = (np.arange(live.size) // slots % length).astype(np.uint32)
    slot[live] = (np.arange(live.size) % slots).astype(np.uint32)
    a, ws = f16((m, k)), [f16((256, k), k ** -0.5) for _ in range(3)]
    rope = rope_table(10000.0, 64, 32, length)
    ba, bs = device.upload(pack(a)), [device.upload(pack(w)) for w in ws]
    bp, br = device.upload(pos), device.upload(rope)
    bq = device.upload(np.full((m, 256), MARK, np.float16))
    bf16 = where == "bf16 ring"
    if where == "paged":
        blocks = slots * length // block
        order = rng.permutation(blocks).reshape(slots, -1).astype(np.uint32)
        bt, units = device.upload(order[slot]), (blocks, heads, block, 64)
    else:
        bt, units = device.upload(slot), ((m, heads, 64) if where == "staged" else (slots, heads, length, 64))
    fill = np.full(units, 0x4321, np.uint16)
    caches = [device.upload(fill) for _ in range(2)]
    try:
        launch(device, kernels, "qkv_rope_paged" if where == "paged" else "qkv_rope", form, shape, bs, [bq, *caches],
               [256] * 3, {"a": ba, "position": bp, "slot": bt, "rope": br}, kv_heads=heads, rope_rows=length,
               length=length, slots=slots, cache_bf16=int(bf16), staged=int(where == "staged"),
               block_size=block if where == "paged" else 0, table_len=length // block if where == "paged" else 0,
               blocks=slots * length // block if where == "paged" else 0)
        lim = [bound(a, w) for w in ws]
        raw = [(a.astype(np.float64) @ w.astype(np.float64).T).reshape(m, heads, 64) for w in ws]
        c, s = (rope[pos, :, i].astype(np.float64)[:, None] for i in (0, 1))

        def turn(x):
            return np.concatenate([x[..., :32] * c - x[..., 32:] * s, x[..., 32:] * c + x[..., :32] * s], -1)

        def check(got, want, lim, ulp):
            # the sums' bounds of a pair, the turn's roundings, the narrowing
            wide = lim.reshape(m, heads, 64)
            wide = wide + np.roll(wide, 32, -1) + 2.0**-22 * (np.abs(want) + 1)
            assert np.all((np.abs(got - want) <= wide + np.abs(want) * ulp + 2.0**-25)[live])

        q = bq.read(np.float16).reshape(m, heads, 64)
        check(q.astype(np.float64), turn(raw[0]), lim[0], 2.0**-11)
        assert np.all(np.delete(q, live, axis=0) == MARK)
        for j, want in ((1, turn(raw[1])), (2, raw[2])):
            held = caches[j - 1].read(np.uint16).reshape(units)
            if where == "staged":
                at = (np.arange(m),)
            elif where == "paged":
                at = (order[slot, pos // block], slice(None), pos % block)
            else:
                at = (slot, slice(None), pos)
            bits = held[at]
            got = (bits.astype(np.uint32) << 16).view(np.float32) if bf16 else bits.view(np.float16)
            check(got.astype(np.float64), want, lim[j], 2.0**-8 if bf16 else 2.0**-11)
            others = np.ones(units, bool)
            others[tuple(i[live] if isinstance(i, np.ndarray) else i for i in at)] = False
            assert np.all(held[others] == 0x4321)
    finally:
        for b in [ba, bp, br, bq, bt, *bs, *caches]:
            b.free()


def test_the_params_are_the_kernels():
    assert ctypes.sizeof(K.SkinnyParams) == ctypes.sizeof(K.GemmParams) + 15 * 4


@pytest.mark.parametrize("parts", [1, 2, 5])
@pytest.mark.parametrize("form", FORMS)
def test_parts_sum_to_the_product(device, kernels, form, parts):
    """Partial sums over parts of k (more than it has steps for, at 5), every
    row of a live chunk, the live chunks one after another in A and C."""
    for shape in (ROWS[2], ROWS[5], (256, 3, 3, 256, 1, 64)):
        m, live, k = shape[0], shape[1], shape[-1]
        a, w = f16((live * 16, k)), f16((256, k))
        full = np.zeros((m, k), np.float16)
        full[:live * 16] = a
        ba, bw = device.upload(pack(full)), device.upload(pack(w))
        bc = device.upload(np.full((parts * live * 16 + 1, 256), MARK, np.float32))
        try:
            launch(device, kernels, "part", form, shape, [bw], [bc], [256], {"a": ba}, parts=parts, compact=1)
            got = bc.read(np.float32).reshape(-1, 256)
            assert np.all(got[-1] == MARK)
            got = got[:-1].reshape(parts, live * 16, 256).astype(np.float64).sum(axis=0)
            exact = a.astype(np.float64) @ w.astype(np.float64).T
            assert np.all(np.abs(got - exact) <= bound(a, w))
        finally:
            for b in (ba, bw, bc):
                b.free()


@pytest.mark.parametrize("shape", [ROWS[3], ROWS[5]], ids=["runs", "apart"])
@pytest.mark.parametrize("source", [K.ROWS_STORED, K.ROWS_GATHER_F16, K.ROWS_GATHER_F32, K.ROWS_PARTS])
@pytest.mark.parametrize("width", list(K.ROWS_NORM_THREADS))
def test_rows_norm(device, kernels, width, source, shape):
    """fk_rows_norm: each way a row is made, then its RMSNorm within one f16
    rounding of binary64's, tiled in place or live rows alone."""
    m, live, run_chunks, run, apart, _ = shape
    rows = live_rows(*shape[:-1])
    index = np.arange(live * 16)[:rows.size] if apart > 1 else None
    rng = np.random.default_rng(width + source)
    x = rng.standard_normal((m, width)).astype(np.float32)
    gain = (1 + 0.1 * rng.standard_normal(width)).astype(np.float32)
    table = rng.standard_normal((50, width)).astype(np.float16 if source == K.ROWS_GATHER_F16 else np.float32)
    tokens = rng.integers(0, 60, m).astype(np.uint32)      # past the table: its last row
    parts = rng.standard_normal((3, live * 16, width)).astype(np.float32)
    where = np.concatenate([np.arange(c * 16, c * 16 + 16) for c in range(live)])[:rows.size]
    if source == K.ROWS_STORED:
        want = x[rows].astype(np.float64)
    elif source == K.ROWS_PARTS:
        want = x[rows].astype(np.float64) + parts[:, where].astype(np.float64).sum(axis=0)
    else:
        want = table[np.minimum(tokens[rows], 49)].astype(np.float64) * 1.25
    bufs = {"x": device.upload(x), "table": device.upload(table), "tokens": device.upload(tokens),
            "partials": device.upload(parts), "gamma": device.upload(gain),
            "xout": device.upload(np.full((m, width), MARK, np.float32)),
            "y": device.upload(np.full(m * width, MARK, np.float16))}
    p = K.RowsNormParams(m, width, live, run_chunks, run, apart, int(apart > 1), 1e-5, 1.0, 1, source, 50, 1.25, 3)
    try:
        kernels.launch(f"fk_rows_norm_w{width}", live * 16, K.ROWS_NORM_THREADS[width],
                       {n: b.ptr for n, b in bufs.items()}, p)
        device.sync()
        y = unpack(bufs["y"].read(np.float16), m, width).astype(np.float64)
        xout = bufs["xout"].read(np.float32).reshape(m, width)
        if source == K.ROWS_STORED:
            assert np.all(xout == MARK)
        else:
            # three additions of binary32 rounding, or a product
            assert np.all(np.abs(xout[rows] - want) <= 4 * 2.0**-24 * (np.abs(want) + 8))
            assert np.all(np.delete(xout, rows, axis=0) == MARK)
        tiles = rows if apart == 1 else index
        normed = want * (np.mean(want * want, axis=1, keepdims=True) + 1e-5) ** -0.5 * gain
        assert np.all(np.abs(y[tiles] - normed) <= np.abs(normed) * (2.0**-11 + 2.0**-18) + 2.0**-20)
        assert np.all(np.delete(y, tiles, axis=0) == MARK)
    finally:
        for b in bufs.values():
            b.free()


@pytest.mark.parametrize("parts", [1, 250, 2000])
def test_rows_token(device, kernels, parts):
    m, live, run_chunks, run, apart, _ = shape = ROWS[5]
    rows = live_rows(*shape[:-1])
    keys = np.random.default_rng(parts).integers(0, 1 << 63, (m, parts), dtype=np.uint64)
    bk, out = device.upload(keys), device.upload(np.full(m, 9, np.uint32))
    kernels.launch("fk_rows_token", live * 16, 256, {"keys": bk.ptr, "out": out.ptr},
                   K.RowsTokenParams(m, live, run_chunks, run, apart, parts))
    device.sync()
    got = out.read(np.uint32)
    want = 0xFFFFFFFF - (keys.max(axis=1) & 0xFFFFFFFF)
    assert np.array_equal(got[rows], want[rows].astype(np.uint32)) and np.all(np.delete(got, rows) == 9)
    bk.free()
    out.free()
