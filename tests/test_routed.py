"""The rule that joins a routed step's launches: which runs of launches it
takes, the joined launches through the engine's checks and the launch
table's, and runs that it must leave alone."""

import pytest

from furykernel_amd import kernels as K, runtime
from furykernel_amd.engine import Engine, check_launch, params_struct
from furykernel_amd.lower import routed_fusions
from moe_cases import ONE_B_MOE, lowered, moe_program
from routed_cases import CASES, case_id, lowered_case


@pytest.mark.parametrize("case", CASES, ids=case_id)
def test_joined_launches(case):
    hidden, experts, ffn, k, table, _, _ = case
    low = lowered_case(case)
    found = routed_fusions(low)
    packs = ffn // (4 if table == "f32" else 8)
    want = ([f"fk_step_router_{'f16' if table == 'f32' else table}"] if experts <= 32 else []) + \
        [f"fk_gemv_routed_act_{table}"] + \
        ([f"fk_gemv_routed_combine_{table}"] if packs <= (128 if k > 2 else 256) else [])
    assert [L.entry for _, _, L in found] == want
    at = 1 << 40
    addr = {}
    for name, spec in low.buffers.items():
        addr[name] = at
        at += (spec.nbytes + 4095) // 4096 * 4096
    for first, count, L in found:
        # every value that the replaced launches store, and no other
        stores = {n for M in low.launches[first:first + count] for b, n in M.bind.items()
                  if b in ("y", "y0", "ids", "ws") and not (b == "ids" and "route" not in M.step)}
        check_launch(L, low.buffers)
        bound = {n for n in L.bind.values() if n is not None}
        assert {n for n in stores if n.startswith("value:")} <= bound
        spans = [(0, 0) if L.bind.get(b) is None else (addr[L.bind[b]], low.buffers[L.bind[b]].nbytes)
                 for b in K.ABIS[L.entry].buffers]
        runtime.launch_check(L.entry, L.groups, L.threads, 0, spans, params_struct(L))
        with pytest.raises(Exception):  # a threadgroup missing or to spare
            runtime.launch_check(L.entry, 0, L.threads, 0, spans, params_struct(L))


def test_a_value_that_meets_another_is_left_alone():
    """Launches whose stored value is another's operand, whose segments are
    not the ranks' rows, or that have another between them."""
    def entries(change):
        low = lowered(moe_program(ONE_B_MOE))
        change(low.launches)
        return [L.entry for _, _, L in routed_fusions(low)]
    router, act, comb = "fk_step_router_f16", "fk_gemv_routed_act_f16", "fk_gemv_routed_combine_f16"
    assert entries(lambda ls: None) == [router, act, comb]
    assert act not in entries(lambda ls: ls[4].bind.update(y=ls[3].bind["x"]))
    assert comb not in entries(lambda ls: ls[6].bind.update(y=ls[5].bind["x"]))
    assert comb not in entries(lambda ls: ls[6].bind.update(x="value:x"))
    assert act not in entries(lambda ls: ls[4].params.update(half=512, n=2048))
    assert router not in entries(lambda ls: ls[0].params.update(seg=1024))
    assert router not in entries(lambda ls: ls[1].params.update(store_tile=0))
    assert router not in entries(lambda ls: ls[2].bind.update(x="value:moe_in"))
    assert router not in entries(lambda ls: ls.insert(2, ls[4]))


def test_picks_of_some_launches_run_them_apart():
    eng = Engine.__new__(Engine)
    eng._fused = {0: (3, 7), 3: (2, 8)}
    assert eng._with_fused([0, 1, 2, 3, 4, 5, 6]) == [7, 8, 5, 6]
    assert eng._with_fused([0, 1, 3, 4]) == [0, 1, 8]
    assert eng._with_fused([2, 3]) == [2, 3]
    assert eng._with_fused([1, 2, 3, 4, 6]) == [1, 2, 8, 6]
