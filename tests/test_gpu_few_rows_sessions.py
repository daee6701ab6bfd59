"""Sessions of few rows on the GPU, through the kernels of few rows
(fk_skinny.h, fk_rows_norm.h, fk_split_attend.h), one layer of the 1B
model's: against the f64 evaluator (the f16 bar, 2e-3 of the largest
magnitude), with every buffer that a step makes holding NaN bits before it,
so that no output may come from a row that the step has not made."""

import dataclasses

import numpy as np
import pytest

from furykernel_amd.program.decoder import ONE_B
from oracle.eval import Bindings, evaluate_fast
from test_gpu_prefill import BAR, rel
from test_gpu_rows import caches_of, host_weights

pytestmark = pytest.mark.gpu

DIMS = dataclasses.replace(ONE_B, vocab=4096, context=1024)


def fill_nan(s):
    """NaN bits (f16's, bf16's and f32's) in what a step makes."""
    given = ("weight:", "widen:", "table:", "ints:", "rope:", "cache:")
    for name in s.lowered.buffers:
        if name not in s.lowered.layouts and not name.startswith(given):
            s.kernels.fill_u32(s.engine.buffers[name], 0xFFFFFFFF)


def open_session(device, kernels, seqs, rows, bound=None, paging=None):
    from furykernel_amd.prefill import PrefillSession
    s = PrefillSession(device, kernels, dataclasses.replace(DIMS, slots=seqs), seqs, rows, layers=1,
                       position_bound=bound, paging=paging)
    for name in s.lowered.buffers:
        if name.startswith("cache:"):
            s.engine.zero(name)
    s.write_weights(host_weights(s.checked, 0.02))
    fill_nan(s)
    device.sync()
    return s


def evaluated(s, seqs, rows, tokens, start=0, caches=None):
    dims = s.dims
    per = dims.kv_heads * dims.context * dims.head_dim
    if caches is None:
        caches = {src.name: {u: np.zeros(per) for u in range(dims.slots)} for src in s.checked.program.sources
                  if type(src.kind).__name__ == "SCache"}
    weights = host_weights(s.checked, 0.02)
    return evaluate_fast(s.checked, Bindings(
        seqs * rows, weights={k: np.asarray(v, np.float64) for k, v in weights.items()},
        row_ints={"tokens": tokens[:, None], "position": np.tile(np.arange(start, start + rows), seqs)[:, None],
                  "slot": np.repeat(np.arange(seqs), rows)[:, None]}, caches=caches))


def check(s, ev, seqs, rows, start=0):
    assert rel(s.logits(), ev.outputs["logits"]) <= BAR
    held = caches_of(s, s.dims)
    for name in held:
        for u in range(seqs):
            g = held[name][u].reshape(s.dims.kv_heads, s.dims.context, s.dims.head_dim)
            w = ev.caches[name][u].reshape(g.shape)
            assert rel(g[:, start:start + rows], w[:, start:start + rows]) <= BAR, (name, u)


@pytest.mark.parametrize("seqs,rows", [(1, 100), (1, 9), (2, 70)])
def test_staged_prefills_read_only_rows_they_made(device, kernels, seqs, rows):
    """Counts whose last query block is half real rows and less."""
    tokens = np.random.default_rng(rows).integers(0, DIMS.vocab, seqs * rows)
    s = open_session(device, kernels, seqs, rows, bound=DIMS.context)
    try:
        assert s.staged and any(L.entry.startswith("fk_skinny_qkv_rope") for L in s.lowered.launches)
        s.set_tokens(tokens)
        print(f"staged prefill {seqs} x {rows}", flush=True)
        s.run()
        device.sync()
        check(s, evaluated(s, seqs, rows, tokens), seqs, rows)
    finally:
        s.close()


@pytest.mark.parametrize("seqs,rows", [(1, 100), (1, 9), (2, 70), (1, 400)])
def test_a_staged_prefill_is_the_in_place_one_bit_for_bit(device, kernels, seqs, rows):
    """The rows that a staged step makes past the live ones change no form."""
    tokens = np.random.default_rng(rows).integers(0, DIMS.vocab, seqs * rows)
    got = []
    for bound in (DIMS.context, None):
        s = open_session(device, kernels, seqs, rows, bound=bound)
        try:
            assert s.staged == (bound is not None)
            s.set_tokens(tokens)
            print(f"prefill {seqs} x {rows}, staged {s.staged}", flush=True)
            s.run()
            device.sync()
            held = caches_of(s, s.dims)
            got.append((s.logits(), s.tokens(),
                        [held[n][u].reshape(8, -1, 64)[:, :rows] for n in sorted(held) for u in range(seqs)]))
        finally:
            s.close()
    (la, ta, ca), (lb, tb, cb) = got
    assert np.array_equal(la.view(np.uint32), lb.view(np.uint32)) and np.array_equal(ta, tb)
    assert all(np.array_equal(a, b) for a, b in zip(ca, cb))


@pytest.mark.parametrize("seqs,rows", [(1, 100), (2, 9), (2, 70), (1, 209)])
def test_ragged_prefills_in_place(device, kernels, seqs, rows):
    """Last query blocks half real rows and less, rings zeroed past them."""
    tokens = np.random.default_rng(rows + 1).integers(0, DIMS.vocab, seqs * rows)
    s = open_session(device, kernels, seqs, rows)
    try:
        entries = {L.entry.rsplit("_", 1)[0] for L in s.lowered.launches}
        assert not s.staged and {"fk_skinny_qkv_rope", "fk_rows_norm"} <= entries
        s.set_tokens(tokens)
        print(f"prefill {seqs} x {rows} in place", flush=True)
        for _ in range(2):      # the second over what the first left
            s.run()
            device.sync()
            check(s, evaluated(s, seqs, rows, tokens), seqs, rows)
        held = caches_of(s, s.dims)
        for name in held:       # the rings past the prompts as they were
            for u in range(seqs):
                assert np.all(held[name][u].reshape(8, -1, 64)[:, rows:] == 0)
    finally:
        s.close()


@pytest.mark.parametrize("seqs,rows", [(1, 100), (2, 300)])
def test_ragged_paged_prefills_are_the_ring_ones(device, kernels, seqs, rows):
    """Pools through scrambled tables: logits and tokens bit for bit the ring
    session's, unsplit attention (100 rows) and split (300)."""
    tokens = np.random.default_rng(rows + 2).integers(0, DIMS.vocab, seqs * rows)
    got = []
    for paging in (None, (64, seqs * DIMS.context // 64 + 3)):
        s = open_session(device, kernels, seqs, rows, paging=paging)
        try:
            store = "fk_skinny_qkv_rope" + ("_paged" if paging else "")
            assert any(L.entry.startswith(store) for L in s.lowered.launches)
            split = any(L.entry.startswith("fk_split_attend") for L in s.lowered.launches)
            assert split == (rows == 300)
            s.set_tokens(tokens)
            print(f"prefill {seqs} x {rows}, paged {paging}", flush=True)
            s.run()
            device.sync()
            got.append((s.logits(), s.tokens()))
        finally:
            s.close()
    assert np.array_equal(got[0][0].view(np.uint32), got[1][0].view(np.uint32))
    assert np.array_equal(got[0][1], got[1][1]) and np.isfinite(got[0][0]).all()


def test_a_later_chunk_of_a_staged_prefill(device, kernels):
    """100 rows at positions 512 .. 611 over what the rings hold: the earlier
    keys from the ring, the step's own from its staging rows."""
    rows, start = 100, 512
    tokens = np.random.default_rng(7).integers(0, DIMS.vocab, rows)
    s = open_session(device, kernels, 1, rows, bound=DIMS.context)
    try:
        for i, name in enumerate(sorted(n for n in s.lowered.buffers if n.startswith("cache:"))):
            s.engine.init_normal(name, 99 + i, 0.5)
        device.sync()
        before = caches_of(s, s.dims)
        s.engine.set_ints("position", s.positions + start, DIMS.context)
        s.set_tokens(tokens)
        print(f"staged prefill 1 x {rows} from {start}", flush=True)
        s.run()
        device.sync()
        check(s, evaluated(s, 1, rows, tokens, start, {n: dict(b) for n, b in before.items()}), 1, rows, start)
        after = caches_of(s, s.dims)
        for n in before:
            b, a = (x[n][0].reshape(8, -1, 64) for x in (before, after))
            own = np.s_[start:start + rows]
            assert np.array_equal(np.delete(a, own, 1), np.delete(b, own, 1))
    finally:
        s.close()


@pytest.mark.parametrize("m", [20, 33])
def test_a_batch_of_more_rows_than_a_chunk(device, kernels, m):
    """Decode rows past one chunk of 16, the last one not whole, their tiled
    values held one after another."""
    from furykernel_amd.prefill import DecodeRows
    dims = dataclasses.replace(DIMS, slots=m, context=512)
    rng = np.random.default_rng(m)
    positions, slots = rng.integers(0, dims.context, m), rng.permutation(m)
    s = DecodeRows(device, kernels, dims, positions, slots, layers=1)
    try:
        assert any(L.params.get("compact") for L in s.lowered.launches)
        s.write_weights(host_weights(s.checked, 0.02))
        for i, name in enumerate(sorted(n for n in s.lowered.buffers if n.startswith("cache:"))):
            s.engine.init_normal(name, 5 + i, 0.5)
        fill_nan(s)
        device.sync()
        before = caches_of(s, dims)
        tokens = rng.integers(0, dims.vocab, m)
        s.set_tokens(tokens)
        print(f"decode batch of {m}", flush=True)
        s.run()
        device.sync()
        ev = evaluate_fast(s.checked, Bindings(
            m, weights={k: np.asarray(v, np.float64) for k, v in host_weights(s.checked, 0.02).items()},
            row_ints={"tokens": tokens[:, None], "position": positions[:, None], "slot": slots[:, None]},
            caches=before))
        assert rel(s.logits(), ev.outputs["logits"]) <= BAR
        assert np.array_equal(s.tokens(), np.argmax(s.logits(), axis=1))
    finally:
        s.close()
