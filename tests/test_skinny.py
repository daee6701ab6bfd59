"""Which GEMMs of a step go to the kernel of few rows (fk_skinny.h), on the
CPU: every launch that does passes the engine's and the launch table's
checks, reaches every live row once, and no other shape is moved."""

import dataclasses

import numpy as np
import pytest

from furykernel_amd import kernels as K, runtime
from furykernel_amd.engine import check_launch, params_struct
from furykernel_amd.prefill import (QBLOCK, LiveRows, decode_placement, lower_prefill, prefill_placement, skinny_form)
from furykernel_amd.program.check import check_program
from furykernel_amd.program.decoder import ONE_B, SMALL_PREFILL, decoder_step
from furykernel_amd.program.plan import PlanOptions, plan


def lowered(dims, seqs, seq_rows, decode=False, bound=None, **kw):
    """(the lowering, the step's real rows, its rows) as the sessions make it."""
    dims = dataclasses.replace(dims, slots=max(seqs, 1))
    if decode:
        rows, _, _, real = decode_placement([0] * seqs, range(seqs), dims.slots)
        run, chunks, at = QBLOCK, -(-seqs // 16), 1
        live = LiveRows(chunks, chunks, rows, QBLOCK, seqs)
    else:
        rows, run, _, _, real = prefill_placement(seqs, seq_rows, dims.slots)
        chunks, at = -(-seq_rows // 16), seq_rows
        live = LiveRows(seqs * chunks, chunks, run, keys=run)
    c = check_program(decoder_step(dims, layers=1, position_bound=bound or (dims.context if decode else seq_rows), **kw))
    return lower_prefill(c, plan(PlanOptions(sequence_rows=at), c), rows, run, True, live), real, rows


CASES = {"1 x 100": (1, 100), "3 x 9": (3, 9), "2 x 700": (2, 700), "1 x 256": (1, 256), "4 x 1500": (4, 1500)}


@pytest.mark.parametrize("case", [*CASES, "staged", "paged", "batch 1", "batch 8", "batch 41"])
def test_every_launch_passes_the_checks_and_makes_the_live_rows(case):
    if case.startswith("batch"):
        low, real, rows = lowered(ONE_B, int(case[6:]), 1, decode=True)
    elif case == "staged":
        low, real, rows = lowered(ONE_B, 2, 64, bound=4096)
    elif case == "paged":
        low, real, rows = lowered(ONE_B, 2, 64, paging=(64, 128))
    else:
        low, real, rows = lowered(ONE_B, *CASES[case])
    at, addr = 1 << 40, {}
    for name, spec in low.buffers.items():
        addr[name] = at
        at += (spec.nbytes + 4095) // 4096 * 4096
    skinny = 0
    for L in low.launches:
        check_launch(L, low.buffers)
        spans = [(0, 0) if L.bind.get(b) is None else (addr[L.bind[b]], low.buffers[L.bind[b]].nbytes)
                 for b in K.ABIS[L.entry].buffers]
        runtime.launch_check(L.entry, L.groups, L.threads, L.lds_bytes, spans, params_struct(L))
        if L.entry.startswith("fk_skinny_"):
            skinny += 1
            p = L.params
            c = np.arange(p["live"])
            first = (c // p["run_chunks"]) * p["run"] + (c % p["run_chunks"]) * 16 * p["apart"]
            made = (first[:, None] + np.arange(16) * p["apart"]).reshape(-1)
            made = made[made < rows]
            assert np.unique(made).size == made.size and np.isin(real, made).all()
            # a grid that misses a tile, a buffer short of its last byte
            with pytest.raises(runtime.FkError):
                runtime.launch_check(L.entry, L.groups - 8, L.threads, L.lds_bytes, spans, params_struct(L))
            for b in ("a", "b0", "c0", "r0", "keys", "position", "rope", "c2"):
                i = K.ABIS[L.entry].buffers.index(b)
                if b in K.launch_reads(L.entry, p) and not (b == "c0" and "_part_" in L.entry):
                    short = list(spans)
                    short[i] = (short[i][0], short[i][1] - 1)
                    with pytest.raises(runtime.FkError):
                        runtime.launch_check(L.entry, L.groups, L.threads, L.lds_bytes, short, params_struct(L))
    assert skinny == {"4 x 1500": 0, "2 x 700": 3, "1 x 256": 4}.get(case, 5)


def test_the_keys_of_the_head_follow_its_tile():
    low, _, rows = lowered(ONE_B, 1, 100)
    head, token = low.launches[-2:]
    mode, (_, nb, _) = K.skinny_entry(head.entry)
    assert mode == "store_keys" and token.entry == "fk_rows_token"
    assert token.params["parts"] == 32000 // (16 * nb)
    assert low.buffers[head.bind["keys"]].count == rows * token.params["parts"]


@pytest.mark.parametrize("rows,context,parts", [(8, 4096, 16), (41, 4096, 4), (64, 4096, 4), (3, 256, 1), (1, 512, 2)])
def test_a_batchs_attention_splits_its_keys(rows, context, parts):
    low, _, _ = lowered(dataclasses.replace(ONE_B, context=context), rows, 1, decode=True)
    entries = [L.entry for L in low.launches]
    at = low.launches[entries.index("fk_rows_attend_f16")]
    assert (at.groups, at.params["rows"], at.params["parts"]) == (rows * 8 * parts, rows, parts)
    assert ("fk_rows_combine" in entries) == (parts > 1)
    assert not any(e.startswith("fk_prefill_attend") for e in entries)


@pytest.mark.parametrize("seqs,seq_rows,kw,entry", [
    (3, 9, {}, "fk_prefill_attend_f16_g4"), (1, 500, {}, "fk_split_attend_f16_h2k4"),
    (2, 700, {}, "fk_split_attend_f16_h4k2"), (2, 700, {"paging": (64, 128)}, "fk_split_attend_paged_f16_h4k2"),
    (1, 512, {"bound": 4096}, "fk_split_attend_h2k4"), (4, 2048, {}, "fk_prefill_attend_f16_g4")])
def test_a_prefills_attention_splits_its_keys_where_its_blocks_are_few(seqs, seq_rows, kw, entry):
    low, _, rows = lowered(ONE_B, seqs, seq_rows, **kw)
    at = [L for L in low.launches if L.entry in K.ATTEND_FORMS]
    assert [L.entry for L in at] == [entry]
    h = int(entry[entry.rindex("h") + 1]) if "split" in entry else 4
    assert at[0].groups == rows // 32 * 32 // h and at[0].threads == K.ATTEND_FORMS[entry]


def test_forms_by_size():
    def down(c, splits=(1,)):
        return skinny_form(c, -(-c // 16) * 256, 2048, 8192, "add", splits)
    # larger tiles as the rows grow; fk_gemm where its rounds are full
    assert [down(c) and down(c)[0] for c in (1, 3, 4, 7, 13, 22, 88, 128, 512)] == \
        ["m1n1", "m2n1", "m2n1", "m2n2", "m4n2", "m4n4", "m8n8", "m8n8", None]
    # k split further where a norm adds the parts, until they cost what they save
    assert [down(c, (1, 2, 4, 8)) for c in (1, 4, 7, 13, 64)] == \
        [("m1n2", 4), ("m4n2", 4), ("m4n4", 4), ("m4n4", 2), ("m4n8", 1)]
    assert skinny_form(1, 256, 3072, 2048, "qkv_rope") == ("m1n2", 1)      # pairs of columns
    assert skinny_form(22, 512, 16384, 2048, "silu_mul") is None
    assert skinny_form(1, 256, 2048, 960, "add") is None                   # a short k
    for c in range(1, 400):
        m = -(-c // 16) * 256
        for n, k, mode in ((3072, 2048, "qkv_rope_paged"), (16384, 2048, "silu_mul"), (32000, 2048, "store_keys"),
                           (256, 1024, "store"), (512, 16384, "add")):
            picked = skinny_form(c, m, n, k, mode)
            if picked is not None:
                mb, nb, _ = K.SKINNY_FORMS[picked[0]]
                assert mb < 2 * c and n % (16 * nb) == 0 and (nb > 1 or mode not in K.SKINNY_PAIR_MODES)
    assert all(L.entry.startswith("fk_skinny") is False
               for L in lowered(SMALL_PREFILL, 2, 100)[0].launches)


def test_the_kernels_between_the_gemms_take_the_live_rows():
    low, real, rows = lowered(ONE_B, 41, 1, decode=True)
    norms = [L for L in low.launches if L.entry == "fk_rows_norm_w2048"]
    assert [L.params["source"] for L in norms] == [K.ROWS_GATHER_F16, K.ROWS_PARTS, K.ROWS_PARTS]
    assert all(L.groups == 48 for L in norms)     # 41 rows in chunks of 16
    assert not any(L.entry.startswith(("fk_prefill_norm", "fk_prefill_gather", "fk_prefill_argmax"))
                   for L in low.launches)
    # each part's sums are read, and only by the norm after it
    for i, L in enumerate(low.launches):
        if "_part_" in L.entry:
            norm = low.launches[i + 1]
            assert norm.bind["partials"] == L.bind["c0"] and norm.params["parts"] == L.params["parts"] > 1
            assert low.buffers[L.bind["c0"]].count >= L.params["parts"] * 48 * 2048
    # the tiled values hold the live rows one after another, everywhere
    assert all(L.params["compact"] == 1 for L in low.launches if L.entry != "fk_rows_token")


def test_a_prefills_tiled_values_stay_in_place():
    low, _, _ = lowered(ONE_B, 1, 100)
    assert not any(L.params.get("compact") for L in low.launches)
    # past ROWS_NORM_CHUNKS the plain kernels stay
    low, _, _ = lowered(ONE_B, 4, 700)
    assert not any(L.entry.startswith(("fk_rows", "fk_skinny_part")) for L in low.launches)


def test_a_batch_through_fk_gemm_is_not_compact():
    # k 512: fk_gemm's, which reads the step's rows in place
    low, _, _ = lowered(SMALL_PREFILL, 4, 1, decode=True)
    assert any(L.entry.startswith("fk_gemm") for L in low.launches)
    assert not any(L.params.get("compact") for L in low.launches)
