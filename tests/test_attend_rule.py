"""Which form the prefill attention takes (kernels.attend_launch), on the
CPU: a windowed launch only forms that hold its blocks at once, few keys none,
and each listed form for some shape."""

import pytest

from furykernel_amd import kernels as K

HEADS = [(kvh * g, kvh) for kvh in (2, 4, 8) for g in (1, 2, 4)]


def forms(window=0, keys=4096, **kw):
    for form in ("", "f16_", "paged_", "paged_f16_"):
        for rows in range(256, 8193, 256):
            for heads, kvh in HEADS:
                yield rows, heads, kvh, K.attend_launch(form, rows, heads, kvh, keys, window, **kw)


def split(entry):
    """(heads a group, groups), or None of an unsplit form."""
    return (int(entry[-3]), int(entry[-1])) if entry.startswith("fk_split") else None


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("window", [64, 128, 200, 256, 512, 1024, 4000])
def test_a_windowed_launch_fits_the_chip(window, bf16):
    for rows, heads, kvh, (entry, groups, threads) in forms(window, bf16=bf16):
        assert threads == K.ATTEND_FORMS[entry] and groups * threads == rows // 32 * heads * 64 * (
            split(entry) or (1, 1))[1]
        if split(entry):
            # LDS: 32 KB a group of wavefronts, 160 KB a CU, 256 CUs
            assert groups <= 256 * (160 // (32 * split(entry)[1])), (rows, heads, kvh, entry)


def test_few_keys_stay_unsplit():
    assert not any(split(e) for *_, (e, _, _) in forms(keys=448))
    assert not any(split(e) for *_, (e, _, _) in forms(window=100))
    # a window's rows never walk more than it, however long the ring
    assert not any(split(e) and split(e)[1] == 2 for *_, (e, _, _) in forms(window=200))


def test_picks_by_what_was_measured():
    def pick(form, rows, heads, kvh, **kw):
        return split(K.attend_launch(form, rows, heads, kvh, 4096, **kw)[0])
    assert pick("f16_", 512, 32, 8) == (2, 4) and pick("f16_", 1024, 32, 8) == (2, 2)
    assert pick("f16_", 2048, 32, 8) == (4, 2) and pick("f16_", 3072, 32, 8) is None
    assert pick("f16_", 2048, 32, 8, window=256) is None
    assert pick("f16_", 768, 16, 8, window=256) == (2, 4)      # 384 pairs: h1k4 would take two rounds
    assert pick("f16_", 8192, 8, 8) is None and pick("f16_", 3584, 8, 8) == (1, 2)
    # rows through registers: past 1280 pairs for a prompt's first rows alone
    assert pick("", 2048, 32, 8, bf16=True) is None and pick("", 2048, 32, 8) is None
    assert pick("", 2048, 32, 8, bf16=True, prompts=True) == (4, 2) == pick("", 2048, 32, 8, prompts=True)
    assert pick("", 256, 32, 8, bf16=True) == (2, 4)


def test_every_form_is_taken():
    taken = {split(e) for bf16 in (False, True) for *_, (e, _, _) in forms(bf16=bf16)}
    assert taken == {None, *K.ATTEND_SPLITS}


@pytest.mark.parametrize("bf16", [False, True])
def test_a_sessions_forms_agree(bf16):
    """Ring, staged and paged steps of one shape split their keys alike."""
    for keys in (256, 512, 768, 1536, 2048):
        got = [[split(e) for *_, (e, _, _) in [(0, K.attend_launch(form, rows, heads, kvh, keys, bf16=bf16,
                                                                   prompts=True))]]
               for rows in range(256, 8193, 256) for heads, kvh in HEADS
               for form in ("", "f16_", "paged_", "paged_f16_")]
        assert all(got[i] == got[i - i % 4] for i in range(len(got)))
