"""Sessions of few rows on the GPU, through the kernels of few rows
(fk_skinny.h, fk_rows_norm.h, fk_split_attend.h), one layer of the 1B
model's: against the f64 evaluator (the f16 bar, 2e-3 of the largest
magnitude), with every buffer that a step makes holding NaN bits before it,
so that no output may come from a row that the step has not made."""

import dataclasses

import numpy as np
import pytest

from furykernel_amd import kernels as K
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
