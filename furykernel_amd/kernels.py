"""The launch table of the hand-written gfx950 kernels.

What a ``Lowered``'s ``loweredKernels`` carries for a runtime
(src/FuryKernel/Backend.hs:76-101): each kernel's entry, its buffers in
binding order, its parameter struct in C layout (src/FuryKernel/Abi.hs:
113-133) and its threads.  Kernargs are the buffers' device addresses in that
order, then the struct.

Every launcher checks the shapes it is given against what its kernel assumes
(packs dividing rows, buffers large enough for every access) before it
launches, and raises ``LaunchError`` otherwise: a kernel is never launched on
a shape it would read or write past.
"""

from __future__ import annotations

import ctypes
import re
import struct
from dataclasses import dataclass
from pathlib import Path

import numpy as np

from . import runtime

PACKAGE = Path(__file__).resolve().parent
CODE_OBJECT = PACKAGE / "fk_kernels.hsaco"
ATTEND_OBJECT = PACKAGE / "fk_attend.hsaco"   # the prefill attention, built apart (fk_attend.h)
# Both code objects as read-only data of one shared library (build.py
# build_kernel_library): what the device runs is mapped into the process.
KERNEL_LIBRARY = PACKAGE / "libfkkernels.so"
WAVE = 64


class LaunchError(ValueError):
    """A launch whose shapes or buffers don't fit its kernel."""


class GemvParams(ctypes.Structure):
    _fields_ = [("n", ctypes.c_uint32), ("k", ctypes.c_uint32)]


class RmsNormParams(ctypes.Structure):
    _fields_ = [
        ("rows", ctypes.c_uint32),
        ("width", ctypes.c_uint32),
        ("seg", ctypes.c_uint32),
        ("eps", ctypes.c_float),
        ("factor", ctypes.c_float),
        ("has_gamma", ctypes.c_uint32),
    ]


class SoftmaxParams(ctypes.Structure):
    _fields_ = [("rows", ctypes.c_uint32), ("n", ctypes.c_uint32)]


class FillParams(ctypes.Structure):
    _fields_ = [("count", ctypes.c_uint32), ("value", ctypes.c_uint32)]


class StreamReadParams(ctypes.Structure):
    _fields_ = [("words", ctypes.c_uint64)]


class NoopParams(ctypes.Structure):
    _fields_ = [("unused", ctypes.c_uint32)]


class StepGemvParams(ctypes.Structure):
    _fields_ = [
        ("n_anchors", ctypes.c_uint32),
        ("rows", ctypes.c_uint32 * 3),
        ("first_row", ctypes.c_uint32 * 4),
        ("k", ctypes.c_uint32),
        ("pro_mode", ctypes.c_uint32),
        ("seg", ctypes.c_uint32),
        ("eps", ctypes.c_float),
        ("factor", ctypes.c_float),
        ("gfactor", ctypes.c_float),
        ("has_gamma", ctypes.c_uint32),
        ("epi_mode", ctypes.c_uint32),
        ("store_tile", ctypes.c_uint32),
        ("table_rows", ctypes.c_uint32),
        ("blocks", ctypes.c_uint32),
        ("arg_slots", ctypes.c_uint32),
        ("act", ctypes.c_uint32),
        ("src2_off", ctypes.c_uint32),
        ("cap", ctypes.c_float),
        ("splits", ctypes.c_uint32),
        ("head_dim", ctypes.c_uint32),
    ]


class GemmParams(ctypes.Structure):
    _fields_ = [("m", ctypes.c_uint32), ("k", ctypes.c_uint32), ("n_anchors", ctypes.c_uint32),
                ("first_col", ctypes.c_uint32 * 4), ("ldc", ctypes.c_uint32 * 3), ("act", ctypes.c_uint32)]


class GemmQkvParams(ctypes.Structure):
    """fk_gemm_qkv_params: the GEMM's parameters, then the RoPE and caches'."""
    _fields_ = GemmParams._fields_ + [("kv_heads", ctypes.c_uint32), ("rope_rows", ctypes.c_uint32),
                                      ("length", ctypes.c_uint32), ("slots", ctypes.c_uint32),
                                      ("cache_bf16", ctypes.c_uint32), ("staged", ctypes.c_uint32)]


class SkinnyParams(ctypes.Structure):
    """fk_skinny_params: the GEMM's, the rows it makes, then the QKV
    epilogue's RoPE, caches and paging."""
    _fields_ = GemmParams._fields_ + [("live", ctypes.c_uint32), ("run_chunks", ctypes.c_uint32),
                                      ("run", ctypes.c_uint32), ("apart", ctypes.c_uint32),
                                      ("compact", ctypes.c_uint32), ("parts", ctypes.c_uint32)] + \
        GemmQkvParams._fields_[len(GemmParams._fields_):] + \
        [("block_size", ctypes.c_uint32), ("table_len", ctypes.c_uint32), ("blocks", ctypes.c_uint32)]


class RowsAttendParams(ctypes.Structure):
    """fk_rows_attend_params: the attention of rows each a sequence's one."""
    _fields_ = [("rows", ctypes.c_uint32), ("apart", ctypes.c_uint32), ("heads", ctypes.c_uint32),
                ("kv_heads", ctypes.c_uint32), ("length", ctypes.c_uint32), ("slots", ctypes.c_uint32),
                ("window", ctypes.c_uint32), ("parts", ctypes.c_uint32), ("compact", ctypes.c_uint32),
                ("scale", ctypes.c_float)]


class RowsNormParams(ctypes.Structure):
    """fk_rows_norm_params: the live rows made (`source`), stored and normed."""
    _fields_ = [(f, ctypes.c_uint32) for f in ("m", "width", "live", "run_chunks", "run", "apart", "compact")] + \
        [("eps", ctypes.c_float), ("factor", ctypes.c_float), ("has_gamma", ctypes.c_uint32),
         ("source", ctypes.c_uint32), ("table_rows", ctypes.c_uint32), ("gfactor", ctypes.c_float),
         ("parts", ctypes.c_uint32)]


class RowsTokenParams(ctypes.Structure):
    _fields_ = [(f, ctypes.c_uint32) for f in ("m", "live", "run_chunks", "run", "apart", "parts")]


class PrefillGatherParams(ctypes.Structure):
    _fields_ = [("rows", ctypes.c_uint32), ("width", ctypes.c_uint32), ("table_rows", ctypes.c_uint32),
                ("table_f16", ctypes.c_uint32), ("factor", ctypes.c_float)]


class PrefillNormParams(ctypes.Structure):
    _fields_ = [("rows", ctypes.c_uint32), ("width", ctypes.c_uint32), ("eps", ctypes.c_float),
                ("factor", ctypes.c_float), ("has_gamma", ctypes.c_uint32)]


class PrefillRopeParams(ctypes.Structure):
    _fields_ = [("rows", ctypes.c_uint32), ("heads", ctypes.c_uint32), ("kv_heads", ctypes.c_uint32),
                ("head_dim", ctypes.c_uint32), ("rotated", ctypes.c_uint32), ("rope_rows", ctypes.c_uint32),
                ("length", ctypes.c_uint32), ("slots", ctypes.c_uint32), ("cache_bf16", ctypes.c_uint32),
                ("staged", ctypes.c_uint32)]


class PrefillAttendParams(ctypes.Structure):
    _fields_ = [("rows", ctypes.c_uint32), ("heads", ctypes.c_uint32), ("kv_heads", ctypes.c_uint32),
                ("length", ctypes.c_uint32), ("slots", ctypes.c_uint32), ("window", ctypes.c_uint32),
                ("cache_bf16", ctypes.c_uint32), ("scale", ctypes.c_float), ("staged", ctypes.c_uint32),
                ("run_rows", ctypes.c_uint32)]


class GemmQkvPagedParams(ctypes.Structure):
    """fk_gemm_qkv_paged_params: the QKV GEMM's, then the pools' paging."""
    _fields_ = GemmQkvParams._fields_ + [("block_size", ctypes.c_uint32), ("table_len", ctypes.c_uint32),
                                         ("blocks", ctypes.c_uint32)]


class PrefillRopePagedParams(ctypes.Structure):
    """fk_prefill_rope_paged_params: the RoPE store's, then the pools' paging."""
    _fields_ = PrefillRopeParams._fields_ + [("block_size", ctypes.c_uint32), ("table_len", ctypes.c_uint32),
                                             ("blocks", ctypes.c_uint32)]


class PrefillAttendPagedParams(ctypes.Structure):
    """fk_prefill_attend_paged_params: the attention's, then the pools' paging."""
    _fields_ = PrefillAttendParams._fields_ + [("block_size", ctypes.c_uint32), ("table_len", ctypes.c_uint32),
                                               ("blocks", ctypes.c_uint32)]


class PrefillLandParams(ctypes.Structure):
    _fields_ = [("rows", ctypes.c_uint32), ("kv_heads", ctypes.c_uint32), ("head_dim", ctypes.c_uint32),
                ("length", ctypes.c_uint32), ("slots", ctypes.c_uint32)]


class PrefillSoftcapParams(ctypes.Structure):
    _fields_ = [("count", ctypes.c_uint32), ("cap", ctypes.c_float)]


class ActMulParams(ctypes.Structure):
    _fields_ = [("n", ctypes.c_uint32), ("act", ctypes.c_uint32), ("b_off", ctypes.c_uint32), ("half", ctypes.c_uint32)]


class ElementwiseParams(ctypes.Structure):
    _fields_ = [("n", ctypes.c_uint32), ("op", ctypes.c_uint32), ("width", ctypes.c_uint32),
                ("width_b", ctypes.c_uint32), ("factor", ctypes.c_float)]


class GatherParams(ctypes.Structure):
    _fields_ = [("rows", ctypes.c_uint32), ("width", ctypes.c_uint32), ("count", ctypes.c_uint32),
                ("table_rows", ctypes.c_uint32), ("factor", ctypes.c_float)]


# fk_step_elementwise's operations.
ELT_ADD, ELT_SCALE, ELT_STANDARDIZE, ELT_CONCAT = range(4)


class PrefillArgmaxParams(ctypes.Structure):
    _fields_ = [("rows", ctypes.c_uint32), ("width", ctypes.c_uint32)]


class PrefillArgmaxKeysParams(ctypes.Structure):
    _fields_ = [("rows", ctypes.c_uint32), ("parts", ctypes.c_uint32)]


class StepTokenParams(ctypes.Structure):
    _fields_ = [("slots", ctypes.c_uint32), ("context", ctypes.c_uint32), ("step", ctypes.c_uint32),
                ("advance", ctypes.c_uint32)]


class StepStoreParams(ctypes.Structure):
    _fields_ = [
        ("n_stores", ctypes.c_uint32),
        ("rope", ctypes.c_uint32 * 2),
        ("kv_heads", ctypes.c_uint32),
        ("head_dim", ctypes.c_uint32),
        ("length", ctypes.c_uint32),
        ("slots", ctypes.c_uint32),
        ("rotated", ctypes.c_uint32),
        ("rope_rows", ctypes.c_uint32),
        ("cache_bf16", ctypes.c_uint32),
    ]


class StepAttendParams(ctypes.Structure):
    _fields_ = [
        ("heads", ctypes.c_uint32),
        ("kv_heads", ctypes.c_uint32),
        ("head_dim", ctypes.c_uint32),
        ("length", ctypes.c_uint32),
        ("slots", ctypes.c_uint32),
        ("splits", ctypes.c_uint32),
        ("split", ctypes.c_uint32),
        ("rope", ctypes.c_uint32),
        ("rotated", ctypes.c_uint32),
        ("rope_rows", ctypes.c_uint32),
        ("scale", ctypes.c_float),
        ("window", ctypes.c_uint32),
        ("cache_bf16", ctypes.c_uint32),
        ("store", ctypes.c_uint32),
        ("krope", ctypes.c_uint32),
        ("has_reach", ctypes.c_uint32),
    ]


class Paging(ctypes.Structure):
    """``fk_paging``: a paged pool's blocks of block_size positions, a row's
    table of table_len blocks, the pool's `blocks`."""
    _fields_ = [("block_size", ctypes.c_uint32), ("table_len", ctypes.c_uint32), ("blocks", ctypes.c_uint32)]


class StepAttendPagedParams(ctypes.Structure):
    _fields_ = [("a", StepAttendParams), ("g", Paging)]


class StepStorePagedParams(ctypes.Structure):
    _fields_ = [("s", StepStoreParams), ("g", Paging)]


class AttendArgs(ctypes.Structure):
    """``fk_attend_args`` (include/fkrocm_ops.h): device addresses, then the
    attention's parameters."""
    _fields_ = [("q", ctypes.c_uint64), ("knew", ctypes.c_uint64), ("vnew", ctypes.c_uint64),
                ("kc", ctypes.c_uint64), ("vc", ctypes.c_uint64), ("position", ctypes.c_uint64),
                ("slot", ctypes.c_uint64), ("rope", ctypes.c_uint64), ("out", ctypes.c_uint64),
                ("p", StepAttendParams)]


class RouteParams(ctypes.Structure):
    _fields_ = [("n", ctypes.c_uint32), ("k", ctypes.c_uint32), ("has_scale", ctypes.c_uint32)]


class GemvRoutedParams(ctypes.Structure):
    _fields_ = [("n", ctypes.c_uint32), ("k", ctypes.c_uint32), ("ranks", ctypes.c_uint32),
                ("shared", ctypes.c_uint32), ("entries", ctypes.c_uint32), ("groups_per_rank", ctypes.c_uint32)]


class CombineRanksParams(ctypes.Structure):
    _fields_ = [("seg", ctypes.c_uint32), ("ranks", ctypes.c_uint32), ("residual", ctypes.c_uint32)]


class RouterParams(ctypes.Structure):
    _fields_ = [(f, ctypes.c_uint32) for f in ("width", "experts", "k", "has_gamma", "has_scale")] + \
        [("eps", ctypes.c_float), ("factor", ctypes.c_float)]


class GemvRoutedActParams(ctypes.Structure):
    _fields_ = GemvRoutedParams._fields_ + [("act", ctypes.c_uint32)]


class GemvRoutedCombineParams(ctypes.Structure):
    _fields_ = GemvRoutedParams._fields_[:5] + [("residual", ctypes.c_uint32)]


class StepCombineParams(ctypes.Structure):
    _fields_ = [("heads", ctypes.c_uint32), ("head_dim", ctypes.c_uint32), ("splits", ctypes.c_uint32)]


class CountParams(ctypes.Structure):
    _fields_ = [("n", ctypes.c_uint32)]


class AdvanceParams(ctypes.Structure):
    _fields_ = [("context", ctypes.c_uint32), ("step", ctypes.c_uint32)]


class InitNormalParams(ctypes.Structure):
    _fields_ = [("count", ctypes.c_uint64), ("seed", ctypes.c_uint64), ("std", ctypes.c_float),
                ("dtype", ctypes.c_uint32)]


@dataclass(frozen=True)
class KernelAbi:
    """A kernel's binary interface: buffers in binding order, then the params struct."""

    entry: str
    buffers: tuple[str, ...]
    params: type
    threads: int = 0  # the threads a launch must have, when the kernel is compiled for one count

    def kernarg(self, bound: dict[str, int], params: ctypes.Structure) -> bytes:
        missing = [b for b in self.buffers if b not in bound]
        if missing:
            raise LaunchError(f"{self.entry}: buffers {missing} not bound")
        ptrs = struct.pack(f"<{len(self.buffers)}Q", *[int(bound[b]) for b in self.buffers])
        return ptrs + bytes(params)


def _gemv_abis() -> dict[str, KernelAbi]:
    out = {}
    for wt, xt in (("f32", "f32"), ("f16", "f32")):
        for r in (1, 2, 4):
            e = f"fk_gemv_{wt}_{xt}_r{r}"
            out[e] = KernelAbi(e, ("w", "x", "y"), GemvParams)
    for r in (1, 2, 4):
        e = f"fk_gemv_i8_f16_r{r}"
        out[e] = KernelAbi(e, ("w", "scale", "x", "y"), GemvParams)
    for wt in ("f32", "f16", "bf16"):
        e = f"fk_gemv_p4_{wt}"
        out[e] = KernelAbi(e, ("w", "x", "y"), GemvParams)
    return out


# The GEMV step kernels (fk_step_gemv.h): <shape>_p<prologue>_e<epilogue>, a
# shape being the weight type, the largest input width it takes and its rows a
# block; the SiLU·mul epilogue (3) on every shape but the widest inputs' (at
# one row a block, a wavefront's row meets its neighbour's in LDS).
STEP_GEMV_SHAPES = {"fk_step_gemv_f16_k2048_r1": True, "fk_step_gemv_f16_k2048_r2": True,
                    "fk_step_gemv_f16_k8192_r1": False, "fk_step_gemv_bf16_k2048_r1": True,
                    "fk_step_gemv_bf16_k2048_r2": True, "fk_step_gemv_bf16_k8192_r1": False,
                    "fk_step_gemv_f32_k256_r1": True,
                    "fk_step_gemv_f32_k256_r2": True, "fk_step_gemv_f32_k1024_r1": True,
                    "fk_step_gemv_f32_k1024_r2": True}
STEP_GEMV_ENTRIES = tuple(f"{shape}_p{pro}_e{epi}" for shape, pairs in STEP_GEMV_SHAPES.items() for pro in range(6)
                          for epi in ((0, 1, 2, 3, 4, 5) if pairs else (0, 1, 2, 4, 5)))
STEP_GEMV_BUFFERS = ("w0", "w1", "w2", "y0", "y1", "y2", "src", "src2", "gamma", "table", "token", "res", "res_table",
                     "res_token", "epi_out", "arg")

# The GEMM of few rows (fk_skinny.h): fk_skinny_<mode>_<form>, a form being the
# (16-row, 16-column) blocks of a tile and the wavefronts its k is split
# among; forms of one column block have no pairs of columns (gate and up, a
# head's RoPE pairs).
SKINNY_FORMS = {"m1n1": (1, 1, 8), "m1n2": (1, 2, 8), "m2n1": (2, 1, 8), "m2n2": (2, 2, 8), "m2n4": (2, 4, 4),
                "m4n2": (4, 2, 8), "m4n4": (4, 4, 4), "m4n8": (4, 8, 4), "m8n8": (8, 8, 4)}
SKINNY_PAIR_MODES = ("silu_mul", "qkv_rope", "qkv_rope_paged")
SKINNY_MODES = ("store", "add", "part", "store_keys") + SKINNY_PAIR_MODES
SKINNY_BUFFERS = ("a", "b0", "b1", "b2", "c0", "c1", "c2", "r0", "position", "slot", "rope", "keys")
_SKINNY = re.compile(r"^fk_skinny_(\w+)_(m\dn\d)$")


def skinny_entry(entry: str) -> tuple[str, tuple]:
    """(mode, (row blocks, column blocks, wavefronts)) of a fk_skinny entry."""
    m = _SKINNY.match(entry)
    return m.group(1), SKINNY_FORMS[m.group(2)]


# What makes a row that fk_rows_norm norms (fk_rows_norm.h); its threads by the
# row's width.
ROWS_STORED, ROWS_GATHER_F16, ROWS_GATHER_F32, ROWS_PARTS = range(4)
ROWS_NORM_THREADS = {512: 64, 1024: 128, 2048: 256, 4096: 256}

# Keys a threadgroup of the attention of a batch of rows takes at a time
# (fk_rows_attend.h).
ROWS_TILE = 256

# Keys a block of the prefill attention stages (fk_attend.h): ring lengths are
# multiples of it.
ATTEND_KEYS = 64

# The prefill attention's forms with a block's keys split among groups of
# wavefronts (fk_attend.h): heads (wavefronts) a group, groups.
ATTEND_SPLITS = ((4, 2), (2, 2), (1, 2), (2, 4), (1, 4))
# Entry -> threads: rings and paged pools, staged through registers or (f16)
# loaded straight into LDS, by the heads a kv head or split.
ATTEND_FORMS = {f"fk_prefill_attend_{form}g{g}": 64 * g for form in ("", "f16_", "paged_", "paged_f16_")
                for g in (1, 2, 4)}
ATTEND_FORMS.update({f"fk_split_attend_{form}h{h}k{k}": 64 * h * k for form in ("", "f16_", "paged_", "paged_f16_")
                     for h, k in ATTEND_SPLITS})


# Where each split form is taken, by the query heads a kv head, tried in order:
# (heads a group, groups), the most pairs of a block of 32 rows and a head, and
# with a window the most pairs and the least window.  See attend_launch.
ATTEND_RULE = {1: (((1, 4), 511, 256, 128), ((1, 2), 1024, 512, 256)),
               2: (((1, 4), 256, 256, 128), ((2, 4), 767, 512, 128), ((2, 2), 2559, 1024, 256)),
               4: (((1, 4), 256, 256, 128), ((2, 4), 767, 512, 128), ((2, 2), 1279, 1024, 512))}
ATTEND_RULE_BF16 = {1: (((1, 4), 767, 256, 1), ((1, 2), 1024, 512, 1)),
                    2: (((2, 4), 767, 512, 1), ((2, 2), 2559, 1024, 1)),
                    4: (((2, 4), 767, 512, 128), ((4, 2), 1279, 1024, 256))}
ATTEND_RULE_MANY = ((4, 2), 2559, 2048, 1024)  # 4 heads, past those
# (form, heads a kv head or (heads a group, groups)) -> entry
ATTEND_ENTRIES = {(form, g): f"fk_prefill_attend_{form}g{g}" for form in ("", "f16_", "paged_", "paged_f16_")
                  for g in (1, 2, 4)}
ATTEND_ENTRIES.update({(form, hk): f"fk_split_attend_{form}h{hk[0]}k{hk[1]}"
                       for form in ("", "f16_", "paged_", "paged_f16_") for hk in ATTEND_SPLITS})


def attend_launch(form: str, rows: int, heads: int, kv_heads: int, keys: int, window: int = 0, bf16: bool = False,
                  prompts: bool = False) -> tuple[str, int, int]:
    """The entry, threadgroups and threads of the prefill attention of `rows`
    rows ("", "f16_", "paged_", "paged_f16_": where its keys come from), the
    rows' positions below `keys`, over `bf16` caches or f16 ones; `prompts`:
    the rows are taken to be sequences' first `keys` ones.

    A wavefront takes a block of 32 rows and a query head and walks the
    block's keys, 64 at a time; few such pairs leave SIMDs idle (1024 on the
    chip, and up to four wavefronts a SIMD to hide a block's latency), so
    their keys are split among groups of wavefronts (fk_split_attend_*), 32
    KB of LDS a group: in four while a threadgroup a CU holds the pairs, in
    two while two a CU do; and the heads of a kv head go to threadgroups of
    their own, for 256 or more.  MI355X, f16, 8 kv heads of 4, µs unsplit and
    split:

    - 256 rows from position 3000 (256 pairs): 48.0, h1k4 22.9, h4k2 36.4;
    - 512 from 3072: 52.1, h2k4 25.9, h1k4 43.2; from 0: 11.0, h2k4 8.7;
    - 1024 from 0: 18.5, h2k2 13.6, h4k2 15.8; from 3072: 59.5, 46.9, 46.7;
    - 2048 from 0 (2048 pairs): 36.6, h4k2 31.3, h2k2 34.7;
    - 2 x 1536 (3072 pairs): 32.0, h4k2 33.5;
    - 8 kv heads of one, 2 x 1792 from 2048 (896 pairs): 55.5, h1k2 55.3; 4
      of one, 2048 pairs, h1k2 at 0.80 to 0.93 of unsplit's speed.

    The blocks of a sequence's first rows differ in their keys and fill in
    behind each other, so there a second round costs little; those of a
    window are all the same, so a form has to hold them at once, and a window
    of few blocks leaves nothing to split.  From 2048, 512 rows: window 64
    6.4, h2k4 6.3; 256 8.9, 8.2; 512 12.2, 9.5.  2048 rows: window 256 12.4,
    h4k2 13.0; 512 17.6, 17.6; 1024 28.1, 26.5.  1536 rows of 4 kv heads of 2
    (384 pairs), window 256: 8.5, h1k4 14.2, h2k4 7.9.

    Rows that go through registers (bf16 ones, converted by the group that
    takes them; f16 ones of staged steps) share the work of a group's heads:
    bf16, 512 rows from 2048, 54.1, h2k4 31.4, h1k4 63.3.  Their h4k2 holds a
    threadgroup a CU, so past 1280 pairs it is for `prompts` alone (bf16, 2 x
    768 from 0 20.7, h4k2 17.5; from 2048 73.1, 76.5).

    Fewer than eight blocks of keys stay: their merge would cost what the
    split saves (256 rows from 0: 7.8, at best 6.7); past 1280 pairs eight do
    too (4 x 512 from 0: 12.4, h4k2 12.8).  The rule is the same for every
    place that a session's keys come from, so that its staged, paged and ring
    steps of one shape agree bit for bit."""
    g, pairs = heads // kv_heads, rows // 32 * heads
    if keys >= 512 and pairs < 2560:
        rule = (ATTEND_RULE_BF16 if bf16 else ATTEND_RULE)[g]
        if g == 4 and keys > 512 and (prompts or "f16" in form):
            rule += (ATTEND_RULE_MANY,)
        for split, most, most_windowed, least in rule:
            if pairs <= (most_windowed if window else most):
                if window and window < least:
                    break
                return ATTEND_ENTRIES[form, split], pairs // split[0], 64 * split[0] * split[1]
    return ATTEND_ENTRIES[form, g], rows // 32 * kv_heads, 64 * g


# Row widths the one-pass RMSNorm-to-tiles holds in registers (fk_prefill.h).
NORM_PACK_HELD = (512, 1024, 2048, 4096)

ABIS: dict[str, KernelAbi] = {
    **_gemv_abis(),
    **{e: KernelAbi(e, ("w", "x", "y"), GemvParams, 256)
       for e in ("fk_gemv_f16_f32_wide",
                 *(f"fk_gemv_{t}_f32_staged_r{r}" for t in ("f32", "f16") for r in (1, 2, 4)))},
    "fk_rmsnorm_f32": KernelAbi("fk_rmsnorm_f32", ("x", "gamma", "y"), RmsNormParams),
    "fk_softmax_f32": KernelAbi("fk_softmax_f32", ("x", "y"), SoftmaxParams),
    "fk_softmax_f32_wide": KernelAbi("fk_softmax_f32_wide", ("x", "y"), SoftmaxParams, 1024),
    "fk_fill_u32": KernelAbi("fk_fill_u32", ("dst",), FillParams),
    **{e: KernelAbi(e, STEP_GEMV_BUFFERS, StepGemvParams, 512) for e in STEP_GEMV_ENTRIES},
    "fk_step_token": KernelAbi("fk_step_token", ("arg", "out", "token", "position"), StepTokenParams, 64),
    **{f"fk_gemm_f16_{mode}": KernelAbi(f"fk_gemm_f16_{mode}", ("a", "b0", "b1", "b2", "c0", "c1", "c2", "r0"),
                                        GemmParams, 256) for mode in ("store", "add", "silu_mul")},
    "fk_gemm_f16_store_keys": KernelAbi("fk_gemm_f16_store_keys", ("a", "b0", "b1", "b2", "c0", "c1", "c2", "r0",
                                                                   "keys"), GemmParams, 256),
    "fk_gemm_f16_qkv_rope": KernelAbi("fk_gemm_f16_qkv_rope", ("a", "b0", "b1", "b2", "c0", "c1", "c2", "r0",
                                                               "position", "slot", "rope"), GemmQkvParams, 256),
    "fk_gemm_f16_qkv_rope_paged": KernelAbi("fk_gemm_f16_qkv_rope_paged", ("a", "b0", "b1", "b2", "c0", "c1", "c2",
                                                                           "r0", "position", "table", "rope"),
                                            GemmQkvPagedParams, 256),
    **{f"fk_skinny_{mode}_{form}": KernelAbi(f"fk_skinny_{mode}_{form}", SKINNY_BUFFERS, SkinnyParams, 64 * w)
       for form, (_, nb, w) in SKINNY_FORMS.items() for mode in SKINNY_MODES
       if nb > 1 or mode not in SKINNY_PAIR_MODES},
    **{e: KernelAbi(e, ("qr", "kc", "vc", "position", "slot", "out", "partials"), RowsAttendParams, 256)
       for e in ("fk_rows_attend_f16", "fk_rows_attend_bf16")},
    **{f"fk_rows_norm_w{w}": KernelAbi(f"fk_rows_norm_w{w}", ("x", "table", "tokens", "partials", "gamma", "xout", "y"),
                                       RowsNormParams, t) for w, t in ROWS_NORM_THREADS.items()},
    "fk_rows_token": KernelAbi("fk_rows_token", ("keys", "out"), RowsTokenParams, 256),
    "fk_rows_combine": KernelAbi("fk_rows_combine", ("partials", "position", "out"), RowsAttendParams),
    "fk_prefill_gather": KernelAbi("fk_prefill_gather", ("table", "tokens", "x"), PrefillGatherParams, 256),
    "fk_prefill_norm_pack": KernelAbi("fk_prefill_norm_pack", ("x", "gamma", "y"), PrefillNormParams, 256),
    **{f"fk_prefill_norm_pack_w{w}": KernelAbi(f"fk_prefill_norm_pack_w{w}", ("x", "gamma", "y"), PrefillNormParams,
                                               256) for w in NORM_PACK_HELD},
    "fk_prefill_rope_store_paged": KernelAbi("fk_prefill_rope_store_paged", ("q", "k", "v", "position", "table",
                                                                             "rope", "qr", "kc", "vc"),
                                             PrefillRopePagedParams),
    "fk_prefill_rope_store": KernelAbi("fk_prefill_rope_store", ("q", "k", "v", "position", "slot", "rope", "qr",
                                                                 "kc", "vc"), PrefillRopeParams),
    **{e: KernelAbi(e, ("qr", "kc", "vc", "position", "slot", "out", "ks", "vs"), PrefillAttendParams, threads)
       for e, threads in ATTEND_FORMS.items() if "_paged_" not in e},
    **{e: KernelAbi(e, ("qr", "kc", "vc", "position", "table", "out"), PrefillAttendPagedParams, threads)
       for e, threads in ATTEND_FORMS.items() if "_paged_" in e},
    "fk_prefill_land": KernelAbi("fk_prefill_land", ("ks", "vs", "position", "slot", "kc", "vc"),
                                 PrefillLandParams, 256),
    "fk_prefill_argmax": KernelAbi("fk_prefill_argmax", ("x", "out"), PrefillArgmaxParams, 256),
    "fk_prefill_argmax_keys": KernelAbi("fk_prefill_argmax_keys", ("keys", "out"), PrefillArgmaxKeysParams, 256),
    "fk_prefill_softcap": KernelAbi("fk_prefill_softcap", ("x", "y"), PrefillSoftcapParams, 256),
    "fk_step_store": KernelAbi("fk_step_store", ("x0", "x1", "c0", "c1", "position", "slot", "rope"),
                               StepStoreParams),
    "fk_step_store_paged": KernelAbi("fk_step_store_paged", ("x0", "x1", "p0", "p1", "position", "table", "rope"),
                                     StepStorePagedParams),
    "fk_step_attend": KernelAbi("fk_step_attend", ("q", "knew", "vnew", "kc", "vc", "position", "slot", "rope",
                                                   "partials", "reach"), StepAttendParams),
    "fk_step_attend_wide": KernelAbi("fk_step_attend_wide", ("q", "knew", "vnew", "kc", "vc", "position", "slot",
                                                             "rope", "partials", "reach"), StepAttendParams),
    "fk_step_attend_paged": KernelAbi("fk_step_attend_paged", ("q", "knew", "vnew", "kpool", "vpool", "position",
                                                               "table", "rope", "partials", "reach"),
                                      StepAttendPagedParams),
    "fk_step_combine": KernelAbi("fk_step_combine", ("partials", "out"), StepCombineParams, 64),
    "fk_step_argmax": KernelAbi("fk_step_argmax", ("x", "out"), CountParams),
    "fk_step_act_mul": KernelAbi("fk_step_act_mul", ("a", "b", "y"), ActMulParams),
    "fk_step_route": KernelAbi("fk_step_route", ("x", "scale", "ids", "ws"), RouteParams, 64),
    "fk_step_combine_ranks": KernelAbi("fk_step_combine_ranks", ("w", "x", "res", "y"), CombineRanksParams),
    **{e: KernelAbi(e, ("table", "ids", "x", "y"), GemvRoutedParams)
       for e in ("fk_gemv_routed_f16_r1", "fk_gemv_routed_f16_r2", "fk_gemv_routed_f32_r1",
                 "fk_gemv_routed_bf16_r1", "fk_gemv_routed_bf16_r2")},
    **{f"fk_step_router_{t}": KernelAbi(f"fk_step_router_{t}", ("x", "gamma", "y", "w", "logits", "scale", "ids", "ws"),
                                        RouterParams, 1024) for t in ("f16", "bf16")},
    **{f"fk_gemv_routed_act_{t}": KernelAbi(f"fk_gemv_routed_act_{t}", ("table", "ids", "x", "y", "out"),
                                            GemvRoutedActParams, 256) for t in ("f16", "bf16", "f32")},
    **{f"fk_gemv_routed_combine_{t}": KernelAbi(f"fk_gemv_routed_combine_{t}",
                                                ("table", "ids", "x", "y", "w", "res", "out"),
                                                GemvRoutedCombineParams, 256) for t in ("f16", "bf16", "f32")},
    "fk_step_elementwise": KernelAbi("fk_step_elementwise", ("a", "b", "c", "y"), ElementwiseParams),
    **{f"fk_step_gather_{t}": KernelAbi(f"fk_step_gather_{t}", ("table", "tokens", "y"), GatherParams)
       for t in ("f32", "f16", "bf16")},
    "fk_step_advance": KernelAbi("fk_step_advance", ("next_token", "token", "position"), AdvanceParams),
    "fk_init_normal": KernelAbi("fk_init_normal", ("dst",), InitNormalParams),
    "fk_noop": KernelAbi("fk_noop", (), NoopParams),
    "fk_stream_read": KernelAbi("fk_stream_read", ("src", "out"), StreamReadParams),
}

# Elements a lane loads at once, by weight type: one 16-byte load of W.
GEMV_PACK = {"f32": 4, "f16": 8, "i8": 16}
ELEM_BYTES = {"f32": 4, "f16": 2, "i8": 1}

# Matvecs (fk_gemv.h): the columns up to which a row takes x staged in LDS, by
# the weights and the rows a wavefront takes: what it holds, of four f16 rows
# (2048) a little less (16384 x 1800 12.7 µs, staged 11.2; x 2040 14.1, 14.9).
# Of wider f16 rows the x that a threadgroup holds whole in LDS, and the rows
# from which that pays.
GEMV_HELD = {("f32", 1): 4096, ("f32", 2): 4096, ("f32", 4): 1024,
             ("f16", 1): 4096, ("f16", 2): 4096, ("f16", 4): 1800}
# (weights, rows a wavefront) -> the entry of any threads, the staged one and
# the columns up to which it is taken; the elements of a pack, the bytes of an
# element of W and of x.
GEMV_ENTRIES = {(t, r): (f"fk_gemv_{t}_f32_r{r}", f"fk_gemv_{t}_f32_staged_r{r}", held, GEMV_PACK[t], ELEM_BYTES[t], 4)
                for (t, r), held in GEMV_HELD.items()}
GEMV_ENTRIES.update({("i8", r): (f"fk_gemv_i8_f16_r{r}", "", 0, 16, 1, 2) for r in (1, 2, 4)})
GEMV_WIDE, GEMV_WIDE_ROWS = 16384, 4096

# Softmax rows that four times the threads make, in the same order (fk_rows.h):
# more than 2048 elements (64 rows of 2048: 3.65 µs, so 3.73; of 4096 4.9, 4.1),
# up to what LDS holds, and at most 512 rows, past which the chip is full
# without (512 of 16384 31.8, 18.6; 1024 of 4096 10.4, 10.1).
SOFTMAX_WIDE_FROM, SOFTMAX_WIDE, SOFTMAX_WIDE_ROWS = 2048, 16384, 512


def gemv_launch(wtype: str, n: int, k: int, rows_per_wave: int, threads: int) -> tuple[str, int, int]:
    """The entry, threadgroups and LDS bytes of a standalone matvec in
    threadgroups of `threads`: of 256, x is staged in LDS (fk_gemv.h says
    where that pays); the sums are the same in any."""
    entry, staged, held, _, _, _ = GEMV_ENTRIES[wtype, rows_per_wave]
    lds = 0
    if threads == 256:
        if k <= held:
            entry = staged
        elif rows_per_wave == 1 and wtype == "f16" and n >= GEMV_WIDE_ROWS and k <= GEMV_WIDE:
            entry, lds = "fk_gemv_f16_f32_wide", -(-k // 512) * 512 * 4
    return entry, -(-n // (threads // WAVE * rows_per_wave)), lds


def _need(buf: runtime.Buffer, nbytes: int, what: str, entry: str) -> None:
    if buf.size < nbytes:
        raise LaunchError(f"{entry}: {what} holds {buf.size} bytes, the launch reads or writes {nbytes}")
    if buf.ptr % 16:
        raise LaunchError(f"{entry}: {what} is not 16-byte aligned")


ATTEND_PREFIX = "fk_prefill_attend"


class Kernels:
    """The code object loaded on a device, and a launcher per kernel family."""

    def __init__(self, device: runtime.Device, library: Path = KERNEL_LIBRARY):
        if not Path(library).exists():
            raise runtime.NativeMissing(f"{library} is not built; run __graft_entry__.build()")
        self.device = device
        self.library = ctypes.CDLL(str(library))
        images = []
        for sym in ("fk_kernels_co", "fk_attend_co"):
            start = ctypes.addressof(ctypes.c_char.in_dll(self.library, sym))
            end = ctypes.addressof(ctypes.c_char.in_dll(self.library, sym + "_end"))
            if end <= start:
                raise runtime.NativeMissing(f"{library}: {sym} is empty")
            images.append((start, end - start))
        self.module = device.load_module_image(*images[0])
        self.attend_module = device.load_module_image(*images[1])

    def fn(self, entry: str) -> runtime.Function:
        module = self.attend_module if entry.startswith(ATTEND_PREFIX) else self.module
        return module.function(entry)

    def launch(self, entry: str, groups: int, threads: int, bound: dict[str, int], params: ctypes.Structure,
               stream: runtime.Stream | None = None, lds_bytes: int = 0) -> None:
        abi = ABIS[entry]
        self.fn(entry).launch(groups, threads, abi.kernarg(bound, params), lds_bytes, stream)

    # y = W x: the GEMV family (test/Test/FuryKernel/Gemv.hs:131-191) at split 1.
    def gemv(self, w: runtime.Buffer, x: runtime.Buffer, y: runtime.Buffer, n: int, k: int, wtype: str = "f32",
             rows_per_wave: int = 1, threads: int = 256, scale: runtime.Buffer | None = None,
             stream: runtime.Stream | None = None) -> None:
        if (wtype, rows_per_wave) not in GEMV_ENTRIES:
            raise LaunchError(f"no GEMV kernel fk_gemv_{wtype}_{'f16' if wtype == 'i8' else 'f32'}_r{rows_per_wave}")
        entry, _, _, pack, w_bytes, x_bytes = GEMV_ENTRIES[wtype, rows_per_wave]
        if n <= 0 or k <= 0 or k % pack:
            raise LaunchError(f"{entry}: k = {k} is not a positive multiple of the pack width {pack}")
        if threads % WAVE or not 0 < threads <= 256:
            raise LaunchError(f"{entry}: {threads} threads is not 1 to 4 wavefronts")
        _need(w, n * k * w_bytes, "W", entry)
        _need(x, k * x_bytes, "x", entry)
        _need(y, n * 4, "y", entry)
        bound = {"w": w.ptr, "x": x.ptr, "y": y.ptr}
        if wtype == "i8":
            if scale is None:
                raise LaunchError(f"{entry}: the int8 layer needs its per-row scales")
            _need(scale, n * 4, "scale", entry)
            bound["scale"] = scale.ptr
        entry, groups, lds = gemv_launch(wtype, n, k, rows_per_wave, threads)
        self.launch(entry, groups, threads, bound, GemvParams(n, k), stream, lds)

    # C = A Bᵀ on the matrix cores (fk_gemm.h): the prefill GEMM.  256 × 256
    # tiles, K steps of 32 taken in pairs; LDS: a ring of 4 stages of A's and
    # B's 256 rows × 32 halves.
    GEMM_TILE, GEMM_K, GEMM_LDS = 256, 64, 4 * 2 * 256 * 32 * 2

    def gemm(self, a: runtime.Buffer, bs: list, cs: list, m: int, k: int, rows: list, mode: str = "store",
             r: runtime.Buffer | None = None, stream: runtime.Stream | None = None, act: int = 0,
             keys: runtime.Buffer | None = None) -> None:
        """A [m, k] f16 in the tile layout (furykernel_amd.layout) times the
        weights bs[j] ([rows[j], k] f16, tiled: the anchors) into cs[j]
        ([m, rows[j]] f32 rows; "add": plus r, [m, rows[0]] f32, which may be
        cs[0]).  "silu_mul": one weight, the pair of gate and up ([2 rows[0],
        k], layout.pair), into cs[0] [m, rows[0]] f16 tiled as silu(gate) up.
        "store_keys": one anchor stored as "store" does, and `keys` [m,
        rows[0] / 128] u64 the greedy token's keys (prefill_argmax_keys)."""
        entry = f"fk_gemm_f16_{mode}"
        if entry not in ABIS:
            raise LaunchError(f"no GEMM {entry}")
        if (mode == "store_keys") != (keys is not None) or (keys is not None and len(bs) != 1):
            raise LaunchError(f"{entry}: keys go with the store_keys mode and one anchor")
        t = self.GEMM_TILE
        if m <= 0 or m % t or k <= 0 or k % self.GEMM_K:
            raise LaunchError(f"{entry}: m = {m} must be a multiple of {t}, k = {k} of {self.GEMM_K}")
        silu = mode == "silu_mul"
        if not 1 <= len(bs) <= (1 if silu else 3) or len(bs) != len(rows) or len(cs) != len(bs):
            raise LaunchError(f"{entry}: {len(bs)} weights, {len(cs)} outputs, {len(rows)} row counts")
        unit = t // 2 if silu else t
        if any(n <= 0 or n % unit for n in rows):
            raise LaunchError(f"{entry}: anchors of {rows} rows, not multiples of {unit}")
        if mode == "add" and (len(bs) != 1 or r is None):
            raise LaunchError(f"{entry}: the residual epilogue takes one anchor and its residual")
        if mode != "add" and r is not None:
            raise LaunchError(f"{entry}: a residual without the residual epilogue")
        _need(a, m * k * 2, "A", entry)
        if silu:
            _need(bs[0], 2 * rows[0] * k * 2, "the gate/up pair", entry)
            _need(cs[0], m * rows[0] * 2, "C", entry)
            groups = (m // t) * (rows[0] // unit)
        else:
            for j, (b, n) in enumerate(zip(bs, rows)):
                _need(b, n * k * 2, f"B{j}", entry)
            for j, (c, n) in enumerate(zip(cs, rows)):
                _need(c, m * n * 4, f"C{j}", entry)
            groups = (m // t) * (sum(rows) // t)
        if r is not None:
            _need(r, m * rows[0] * 4, "R", entry)
        if keys is not None:
            _need(keys, m * (rows[0] // 128) * 8, "keys", entry)
        first = [0]
        for n in rows:
            first.append(first[-1] + n)
        first += [first[-1]] * (4 - len(first))
        ldc = (list(rows) + [0, 0, 0])[:3]
        bufs = {"a": a.ptr, "r0": r.ptr if r is not None else 0}
        if keys is not None:
            bufs["keys"] = keys.ptr
        for j in range(3):
            bufs[f"b{j}"] = bs[j].ptr if j < len(bs) else 0
            bufs[f"c{j}"] = cs[j].ptr if j < len(cs) else 0
        if act not in (ACT_SILU, ACT_GELU_TANH):
            raise LaunchError(f"{entry}: activation {act}")
        params = GemmParams(m, k, len(bs), (ctypes.c_uint32 * 4)(*first), (ctypes.c_uint32 * 3)(*ldc), act)
        self.launch(entry, groups, 256, bufs, params, stream, lds_bytes=self.GEMM_LDS)

    # The kernels around the prefill GEMM (fk_prefill.h).

    def prefill_norm_pack(self, x: runtime.Buffer, gamma: runtime.Buffer | None, y: runtime.Buffer, rows: int,
                          width: int, eps: float = 1e-5, factor: float = 1.0,
                          stream: runtime.Stream | None = None) -> None:
        """RMSNorm of f32 rows [rows, width] into f16 tiles (the GEMM's A)."""
        entry = f"fk_prefill_norm_pack_w{width}" if width in NORM_PACK_HELD else "fk_prefill_norm_pack"
        if rows <= 0 or rows % 256 or width <= 0 or width % 32:
            raise LaunchError(f"{entry}: [{rows}, {width}] does not tile (rows of 256, columns of 32)")
        _need(x, rows * width * 4, "x", entry)
        _need(y, rows * width * 2, "y", entry)
        if gamma is not None:
            _need(gamma, width * 4, "gamma", entry)
        self.launch(entry, rows // 4, 256, {"x": x.ptr, "gamma": gamma.ptr if gamma is not None else 0, "y": y.ptr},
                    PrefillNormParams(rows, width, eps, factor, int(gamma is not None)), stream)

    def prefill_argmax(self, x: runtime.Buffer, out: runtime.Buffer, rows: int, width: int,
                       stream: runtime.Stream | None = None) -> None:
        """The greedy token of each f32 row [rows, width] into out (u32)."""
        entry = "fk_prefill_argmax"
        if rows <= 0 or width <= 0:
            raise LaunchError(f"{entry}: [{rows}, {width}]")
        _need(x, rows * width * 4, "x", entry)
        _need(out, rows * 4, "out", entry)
        self.launch(entry, (rows + 3) // 4, 256, {"x": x.ptr, "out": out.ptr}, PrefillArgmaxParams(rows, width), stream)

    def prefill_argmax_keys(self, keys: runtime.Buffer, out: runtime.Buffer, rows: int, parts: int,
                            stream: runtime.Stream | None = None) -> None:
        """The greedy token of each row from its `parts` keys (u64, [rows,
        parts], as gemm's store_keys mode leaves them) into out (u32)."""
        entry = "fk_prefill_argmax_keys"
        if rows <= 0 or parts <= 0:
            raise LaunchError(f"{entry}: {rows} rows of {parts} keys")
        _need(keys, rows * parts * 8, "keys", entry)
        _need(out, rows * 4, "out", entry)
        self.launch(entry, (rows + 3) // 4, 256, {"keys": keys.ptr, "out": out.ptr},
                    PrefillArgmaxKeysParams(rows, parts), stream)

    def prefill_attend(self, qr: runtime.Buffer, kc: runtime.Buffer, vc: runtime.Buffer, position: runtime.Buffer,
                       slot: runtime.Buffer, out: runtime.Buffer, rows: int, heads: int, kv_heads: int,
                       length: int, slots: int, scale: float, window: int = 0, cache_bf16: bool = False,
                       positions=None, seqs=None, stream: runtime.Stream | None = None) -> None:
        """Causal attention of f16 rows q [rows, heads · 64] (RoPE'd) over the
        caches [slots][kv_heads][length][64] into f16 tiles [rows, heads · 64].
        Every block of 32 rows must be one sequence's consecutive positions:
        given the host copies (positions, seqs), that is checked here.  A bf16
        cache is converted to f16 as it is staged (the matrix operations take
        f16): an element beyond f16's range (|x| > 65504) becomes infinite and
        one below 2^-24 flushes to zero, so bf16 caches are for values inside
        f16's range, as the prefill's own stores of f16-range rows are."""
        form = "" if cache_bf16 else "f16_"
        g = heads // kv_heads if kv_heads > 0 and heads % kv_heads == 0 else 0
        entry = ATTEND_ENTRIES.get((form, g), "fk_prefill_attend")
        if rows <= 0 or rows % 256 or g not in ATTEND_RULE:
            raise LaunchError(f"{entry}: {rows} rows, {heads} heads over {kv_heads}")
        if length <= 0 or length % ATTEND_KEYS:
            raise LaunchError(f"{entry}: a ring of {length}; keys go by blocks of {ATTEND_KEYS} that must not wrap")
        if positions is not None:
            from .prefill import check_rows
            check_rows(positions, seqs)
            if np.max(np.asarray(positions)) >= length:
                raise LaunchError(f"{entry}: positions past the ring's {length}")
        q_bytes, cache_bytes = rows * heads * 128, slots * kv_heads * length * 128
        _need(qr, q_bytes, "q", entry)
        _need(kc, cache_bytes, "K cache", entry)
        _need(vc, cache_bytes, "V cache", entry)
        _need(position, rows * 4, "position", entry)
        _need(slot, rows * 4, "slot", entry)
        _need(out, q_bytes, "out", entry)
        bound = {"qr": qr.ptr, "kc": kc.ptr, "vc": vc.ptr, "position": position.ptr, "slot": slot.ptr, "out": out.ptr,
                 "ks": 0, "vs": 0}
        entry, groups, threads = attend_launch(form, rows, heads, kv_heads, length, window, cache_bf16)
        self.launch(entry, groups, threads, bound,
                    PrefillAttendParams(rows, heads, kv_heads, length, slots, window, int(cache_bf16), scale), stream)

    def rmsnorm(self, x: runtime.Buffer, gamma: runtime.Buffer | None, y: runtime.Buffer, rows: int, width: int,
                seg: int | None = None, eps: float = 1e-6, factor: float = 1.0, threads: int = 256,
                stream: runtime.Stream | None = None) -> None:
        entry = "fk_rmsnorm_f32"
        seg = width if seg is None else seg
        if rows <= 0 or seg <= 0 or width % seg or seg % 4:
            raise LaunchError(f"{entry}: segments of {seg} don't divide rows of {width} into packs of 4")
        if threads % WAVE or not 0 < threads <= 1024:
            raise LaunchError(f"{entry}: {threads} threads is not 1 to 16 wavefronts")
        _need(x, rows * width * 4, "x", entry)
        _need(y, rows * width * 4, "y", entry)
        if gamma is not None:
            _need(gamma, seg * 4, "gamma", entry)
        bound = {"x": x.ptr, "gamma": gamma.ptr if gamma is not None else 0, "y": y.ptr}
        params = RmsNormParams(rows, width, seg, eps, factor, 1 if gamma is not None else 0)
        self.launch(entry, rows * (width // seg), threads, bound, params, stream)

    def fill_u32(self, dst: runtime.Buffer, value: int = 0, count: int | None = None,
                 stream: runtime.Stream | None = None) -> None:
        """Sets 32-bit words of a buffer: what a graph clears memory with."""
        count = dst.size // 4 if count is None else count
        if count * 4 > dst.size:
            raise LaunchError(f"fk_fill_u32: {count} words past a buffer of {dst.size} bytes")
        groups = min(max((count + 255) // 256, 1), 4096)
        self.launch("fk_fill_u32", groups, 256, {"dst": dst.ptr}, FillParams(count, value & 0xFFFFFFFF), stream)

    def stream_read(self, src: runtime.Buffer, out: runtime.Buffer, groups: int, nbytes: int | None = None,
                    stream: runtime.Stream | None = None) -> None:
        """Reads `nbytes` of a buffer once (the attainable read bandwidth)."""
        nbytes = src.size if nbytes is None else nbytes
        if nbytes > src.size or nbytes % 16 or src.ptr % 16:
            raise LaunchError("fk_stream_read: a read past the buffer or not in 16-byte words")
        if out.size < groups * 4 * 4:
            raise LaunchError("fk_stream_read: the output holds a word per wavefront")
        self.launch("fk_stream_read", groups, 256, {"src": src.ptr, "out": out.ptr}, StreamReadParams(nbytes // 16),
                    stream)

    def softmax(self, x: runtime.Buffer, y: runtime.Buffer, rows: int, n: int, threads: int = 256,
                stream: runtime.Stream | None = None) -> None:
        """The softmax of each row in the order of `threads` threads; of 256,
        four make what one of them would where the rows are few and long, bit
        for bit."""
        entry = "fk_softmax_f32"
        if rows <= 0 or n <= 0 or n % 4:
            raise LaunchError(f"{entry}: rows of {n} are not packs of 4")
        if threads % WAVE or not 0 < threads <= 1024:
            raise LaunchError(f"{entry}: {threads} threads is not 1 to 16 wavefronts")
        _need(x, rows * n * 4, "x", entry)
        _need(y, rows * n * 4, "y", entry)
        if threads == 256 and SOFTMAX_WIDE_FROM < n <= SOFTMAX_WIDE and rows <= SOFTMAX_WIDE_ROWS:
            entry, threads = "fk_softmax_f32_wide", 1024
        self.launch(entry, rows, threads, {"x": x.ptr, "y": y.ptr}, SoftmaxParams(rows, n), stream)


# What each launch reads and writes: the buffers its kernel dereferences for
# its entry and parameters.  A buffer outside this set may be unbound (passed
# as address 0); one inside it never may.

_GEMV_SUFFIX = re.compile(r"^(fk_step_gemv_(f16|bf16|f32)_k(\d+)_r(\d+))_p(\d)_e(\d)$")
PRO_STORED, PRO_RMSNORM, PRO_GATHER, PRO_GATHER_RMSNORM, PRO_SILU_MUL, PRO_COMBINE = range(6)
COMBINE_SPLITS = 8  # the combine prologue's splits at most
EPI_NONE, EPI_ADD_STORED, EPI_ADD_GATHER, EPI_SILU_MUL, EPI_ARGMAX, EPI_SOFTCAP = range(6)
ACT_SILU, ACT_GELU_TANH = 0, 1


def gemv_entry(entry: str) -> tuple[str, str, int, int, int, int]:
    """(shape, weight type, widest k, rows a block, prologue, epilogue) of a
    GEMV step entry: the kernel is specialised on the modes its name carries,
    whatever its parameter struct says."""
    m = _GEMV_SUFFIX.match(entry)
    if m is None:
        raise LaunchError(f"{entry} is not a GEMV step entry")
    return m.group(1), m.group(2), int(m.group(3)), int(m.group(4)), int(m.group(5)), int(m.group(6))


def gemv_reads(pro: int, epi: int, n_anchors: int, store_tile: bool, arg_slots: int = 0) -> set[str]:
    """The buffers a GEMV step kernel of prologue `pro` and epilogue `epi`
    dereferences (fk_step_gemv.h): the gathers read the token unconditionally,
    the norms their gains, and so on."""
    need = {f"w{j}" for j in range(n_anchors)}
    if store_tile:
        need |= {f"y{j}" for j in range(n_anchors)}
    if pro in (PRO_GATHER, PRO_GATHER_RMSNORM):
        need |= {"table", "token"}
    else:
        need.add("src")
    if pro == PRO_SILU_MUL:
        need.add("src2")
    if pro in (PRO_RMSNORM, PRO_GATHER_RMSNORM):
        need.add("gamma")
    if epi == EPI_ADD_STORED:
        need |= {"res", "epi_out"}
    elif epi == EPI_ADD_GATHER:
        need |= {"res_table", "res_token", "epi_out"}
    elif epi == EPI_SILU_MUL:
        need.add("epi_out")
    elif epi == EPI_ARGMAX:
        need.add("arg")
    elif epi == EPI_SOFTCAP:
        need.add("epi_out")
        if arg_slots:
            need.add("arg")
    return need


def launch_reads(entry: str, params: dict) -> set[str]:
    """The buffers a launch of `entry` with `params` dereferences."""
    abi = ABIS[entry]
    if entry.startswith("fk_step_gemv"):
        _, _, _, _, pro, epi = gemv_entry(entry)
        return gemv_reads(pro, epi, params["n_anchors"], bool(params.get("store_tile", 0)), params.get("arg_slots", 0))
    if entry in ("fk_step_attend", "fk_step_attend_wide", "fk_step_attend_paged"):
        paged = entry == "fk_step_attend_paged"
        need = {"q", "position", "partials"} | ({"kpool", "vpool", "table"} if paged else {"kc", "vc", "slot"})
        if params.get("store"):
            need |= {"knew", "vnew"}
        if params.get("rope") or params.get("krope"):
            need.add("rope")
        if params.get("has_reach"):
            need.add("reach")
        return need
    if entry == "fk_step_route":
        return {"x", "ids", "ws"} | ({"scale"} if params.get("has_scale") else set())
    if entry.startswith("fk_step_router_"):
        return set(abi.buffers) - (set() if params.get("has_gamma") else {"gamma"}) - \
            (set() if params.get("has_scale") else {"scale"})
    if entry.startswith("fk_gemv_routed_combine_"):
        return set(abi.buffers) - (set() if params.get("residual") else {"res"})
    if entry == "fk_step_combine_ranks":
        return {"w", "x", "y"} | ({"res"} if params.get("residual") else set())
    if entry == "fk_step_act_mul":
        return {"a", "y"} | (set() if params.get("half") else {"b"})
    if entry == "fk_step_elementwise":
        op = params.get("op", ELT_ADD)
        return {"a", "y"} | ({"b", "c"} if op == ELT_STANDARDIZE else {"b"})
    if entry == "fk_step_store_paged":
        need = {"x0", "p0", "position", "table"}
        if params.get("n_stores", 1) > 1:
            need |= {"x1", "p1"}
        if any(params.get("rope", (0, 0))):
            need.add("rope")
        return need
    if entry == "fk_step_store":
        need = {"x0", "c0", "position", "slot"}
        if params.get("n_stores", 1) > 1:
            need |= {"x1", "c1"}
        if any(params.get("rope", (0, 0))):
            need.add("rope")
        return need
    if entry == "fk_step_token":
        return {"arg", "out"} | ({"token", "position"} if params.get("advance") else set())
    if entry.startswith("fk_gemm_f16_"):
        n = params.get("n_anchors", 1)
        need = {"a"} | {f"b{j}" for j in range(n)} | {f"c{j}" for j in range(n)}
        if entry == "fk_gemm_f16_add":
            need.add("r0")
        if entry == "fk_gemm_f16_qkv_rope":
            need |= {"position", "slot", "rope"}
        if entry == "fk_gemm_f16_qkv_rope_paged":
            need |= {"position", "table", "rope"}
        if entry == "fk_gemm_f16_store_keys":
            need.add("keys")
        return need
    if entry.startswith("fk_rows_norm"):
        source = params.get("source", ROWS_STORED)
        need = {"y"} | ({"gamma"} if params.get("has_gamma") else set())
        if source != ROWS_STORED:
            need.add("xout")
        if source in (ROWS_GATHER_F16, ROWS_GATHER_F32):
            return need | {"table", "tokens"}
        return need | {"x"} | ({"partials"} if source == ROWS_PARTS else set())
    if entry.startswith("fk_rows_attend"):
        return set(abi.buffers) - (set() if params.get("parts", 1) > 1 else {"partials"})
    if entry.startswith("fk_skinny_"):
        mode, _ = skinny_entry(entry)
        n = params.get("n_anchors", 1)
        need = {"a"} | {f"b{j}" for j in range(n)} | {f"c{j}" for j in range(n)}
        if mode in ("qkv_rope", "qkv_rope_paged"):
            need |= {"position", "slot", "rope"}
        return need | {"add": {"r0"}, "store_keys": {"keys"}}.get(mode, set())
    if entry == "fk_rmsnorm_f32" or entry.startswith("fk_prefill_norm_pack"):
        return set(abi.buffers) - ({"gamma"} if not params.get("has_gamma") else set())
    if entry in ATTEND_FORMS and "_paged_" not in entry:
        return set(abi.buffers) - (set() if params.get("staged") else {"ks", "vs"})
    return set(abi.buffers)
