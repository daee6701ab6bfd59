"""Which rows of a step hold a value once its launches have run, on the CPU:
a staged prefill's attention reads its run's staging rows by whole query
blocks, so a step of few live rows has to make all of those (a weight of 0
times an unwritten row's NaN or infinity is NaN), and the real rows' outputs
have to come from rows that were made."""

import dataclasses

import numpy as np
import pytest

from furykernel_amd import kernels as K
from furykernel_amd.prefill import QBLOCK, LiveRows, lower_prefill, prefill_placement
from furykernel_amd.program.check import check_program
from furykernel_amd.program.decoder import ONE_B, decoder_step
from furykernel_amd.program.plan import PlanOptions, plan


def live_rows(p, rows):
    c = np.arange(p["live"])
    first = (c // p["run_chunks"]) * p["run"] + (c % p["run_chunks"]) * 16 * p["apart"]
    at = (first[:, None] + np.arange(16) * p["apart"]).reshape(-1)
    out = np.zeros(rows, bool)
    out[at[at < rows]] = True
    return out


def made_rows(low, rows):
    """Buffer -> its rows that hold a value, after the step; and how many
    attentions read staging rows.  Inputs, weights and what the rings held
    before hold one."""
    made, staged = {}, 0

    def of(L, *names):
        return np.logical_and.reduce([made.get(L.bind[b], np.ones(rows, bool)) for b in names])

    for L in low.launches:
        p, e = L.params, L.entry
        live = live_rows(p, rows) if "live" in p else np.ones(rows, bool)
        if e == "fk_prefill_gather":
            made[L.bind["x"]] = live
        elif e.startswith(("fk_prefill_norm_pack", "fk_rows_norm")):
            source = p.get("source", K.ROWS_STORED)
            got = live & (of(L, "x") if source in (K.ROWS_STORED, K.ROWS_PARTS) else live)
            if source == K.ROWS_PARTS:
                got &= made[L.bind["partials"]]
            made[L.bind["y"]] = got
            if source != K.ROWS_STORED:
                made[L.bind["xout"]] = got
        elif e.startswith(("fk_gemm_f16_", "fk_skinny_")):
            got = live & of(L, "a", *(["r0"] if "_add" in e else []))
            for c in ("c0", "c1", "c2"):
                if L.bind.get(c) is not None and not L.bind[c].startswith("cache:"):
                    made[L.bind[c]] = got
            if "keys" in e:
                made[L.bind["keys"]] = got
        elif e == "fk_prefill_rope_store":
            for b, to in (("q", "qr"), ("k", "kc"), ("v", "vc")):
                if not L.bind[to].startswith("cache:"):
                    made[L.bind[to]] = of(L, b)
        elif e in K.ATTEND_FORMS:
            got = of(L, "qr").copy()
            if p["staged"]:
                staged += 1
                held = of(L, "ks", "vs")
                for r0 in range(0, rows, QBLOCK):
                    # the run's rows up to the block's last query
                    run = r0 // p["run_rows"] * p["run_rows"]
                    got[r0:r0 + QBLOCK] &= held[run:r0 + QBLOCK].all()
            made[L.bind["out"]] = got
        elif e in ("fk_rows_token", "fk_prefill_argmax_keys"):
            made[L.bind["out"]] = live & of(L, "keys")
        else:
            assert e == "fk_prefill_land", e
    return made, staged


def prefill(dims, seqs, seq_rows, layers, **kw):
    """(the lowering, the step's real rows, its rows), as ``PrefillSession``
    makes it."""
    dims = dataclasses.replace(dims, slots=seqs)
    rows, run, _, _, real = prefill_placement(seqs, seq_rows, dims.slots)
    chunks = -(-seq_rows // 16)
    c = check_program(decoder_step(dims, layers=layers, **kw))
    return lower_prefill(c, plan(PlanOptions(sequence_rows=seq_rows), c), rows, run, True,
                         LiveRows(seqs * chunks, chunks, run, keys=run)), real, rows


# Every count up to past a run of 256 rows' query blocks, and rows on both
# sides of a block's half from there on.
ROWS = [*range(2, 290), *(b + d for b in range(320, 1501, 128) for d in (1, 15, 16, 17, 31, 32))]


@pytest.mark.parametrize("seqs", [1, 3])
def test_staged_steps_make_every_row_they_read(seqs):
    for seq_rows in ROWS:
        low, real, rows = prefill(ONE_B, seqs, seq_rows, 2, position_bound=4096)
        made, staged = made_rows(low, rows)
        assert staged == 2
        for name in ("value:logits", "value:token"):
            assert made[name][real].all(), (seq_rows, name)


@pytest.mark.parametrize("seq_rows", [5, 16, 17, 100, 700])
def test_staged_rows_that_the_rope_kernel_stores(seq_rows):
    """With 16 of 32 pairs turned, RoPE is a kernel of its own between the
    GEMMs of the live rows and the staging rows."""
    low, real, rows = prefill(ONE_B, 2, seq_rows, 2, position_bound=4096, rope_rotated=16)
    assert any(L.entry == "fk_prefill_rope_store" and L.bind["kc"].startswith("staged:") for L in low.launches)
    made, staged = made_rows(low, rows)
    assert staged == 2 and made["value:logits"][real].all()


@pytest.mark.parametrize("seq_rows", [650, 656, 657])
def test_fk_gemm_after_a_norm_of_the_live_rows(seq_rows):
    """A wide QKV stays fk_gemm's, which makes every row, while the split down
    projection's norm before it makes the live ones alone: the staging rows
    that a live block reads are still made from rows that were."""
    wide = dataclasses.replace(ONE_B, heads=128, kv_heads=32)
    low, real, rows = prefill(wide, 1, seq_rows, 2, position_bound=4096)
    entries = [L.entry for L in low.launches]
    i = len(entries) - 1 - entries[::-1].index("fk_gemm_f16_qkv_rope")
    assert entries[i - 1].startswith("fk_rows_norm") and low.launches[i - 1].params["source"] == K.ROWS_PARTS
    made, staged = made_rows(low, rows)
    assert staged == 2 and made["value:logits"][real].all()


def test_in_place_steps_make_their_real_rows():
    for seqs, seq_rows in [(1, 1), (1, 100), (2, 700), (3, 9), (1, 1300)]:
        for kw in ({}, {"paging": (64, 256)}):
            low, real, rows = prefill(ONE_B, seqs, seq_rows, 2, position_bound=seq_rows, **kw)
            made, staged = made_rows(low, rows)
            assert staged == 0 and made["value:logits"][real].all()


@pytest.mark.parametrize("seqs", [1, 2])
def test_a_staged_step_takes_the_in_place_ones_forms(seqs):
    """Whatever the rows that it makes beside the live ones, so that the two
    agree bit for bit: the same launches but for where keys and values go."""
    for seq_rows in ROWS:
        steps = [prefill(ONE_B, seqs, seq_rows, 2, position_bound=bound)[0] for bound in (seq_rows, 4096)]
        entries = [[L.entry.replace("_attend_f16_", "_attend_") for L in low.launches if L.entry != "fk_prefill_land"]
                   for low in steps]
        parts = [[L.params.get("parts") for L in low.launches if L.entry.startswith("fk_skinny")] for low in steps]
        assert entries[0] == entries[1] and parts[0] == parts[1], seq_rows
