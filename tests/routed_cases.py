"""Routed-experts steps of one row for the tests of their joined launches."""

from __future__ import annotations

import numpy as np

from furykernel_amd.lower import lower_plan
from furykernel_amd.program.build import program
from furykernel_amd.program.check import check_program
from furykernel_amd.program.graph import BF16, F16, F32, whole_row
from furykernel_amd.program.plan import PlanOptions, plan
from oracle.cpu_target import CpuTarget

# hidden, experts, expert ffn, k, table type, expert scale, residual
CASES = [(64, 1, 8, 1, F16, False, True), (2048, 32, 1024, 4, F16, True, True), (520, 17, 264, 3, F16, True, False),
         (1032, 16, 1536, 2, F16, False, True), (512, 9, 136, 2, BF16, True, True), (256, 8, 516, 4, F32, False, True),
         (2048, 33, 128, 2, F16, True, True), (256, 8, 1032, 3, F16, True, True)]


def case_id(c) -> str:
    return "h{}_e{}_f{}_k{}_{}_s{:d}_r{:d}".format(*c)


def routed_program(c):
    hidden, experts, ffn, k, table, scaled, residual = c

    def body(b):
        x = b.input("x", whole_row(hidden), F32)
        g = b.weight("moe_norm", [hidden], F32)
        router = b.weight("router", [experts, hidden], F16 if table == F32 else table)
        scale = b.weight("expert_scale", [experts], F32) if scaled else None
        gu = b.table("experts_gate_up", experts, [2 * ffn, hidden], table)
        dn = b.table("experts_down", experts, [hidden, ffn], table)
        cn = b.rmsnorm("moe_in", 1e-6, g, 1.0, x)
        ids, ws = b.route("route", k, scale, b.linear("router_logits", router, 0, cn))
        act = b.gated_gelu("experts_act", b.linear_routed("experts_gate_up_out", gu, ids, cn))
        s = b.combine_ranks("experts_sum", ws, b.linear_routed("experts_out", dn, ids, act))
        b.output("y", b.add("y", x, s) if residual else s)
    return check_program(program("routed", body))


def lowered_case(c):
    checked = routed_program(c)
    return lower_plan(checked, plan(PlanOptions(), checked))


def _typed(t, a):
    if t == F32:
        return a.astype(np.float32)
    if t == F16:
        return a.astype(np.float16)
    return (a.astype(np.float32).view(np.uint32) >> 16).astype(np.uint16)


def state_of(c, seed=5):
    hidden, experts, ffn, k, table, scaled, _ = c
    rng = np.random.default_rng(seed)
    w = {"moe_norm": (1 + 0.1 * rng.standard_normal(hidden)).astype(np.float32),
         "router": _typed(F16 if table == F32 else table, rng.standard_normal((experts, hidden)) * 0.2),
         "experts_gate_up": _typed(table, rng.standard_normal((experts, 2 * ffn, hidden)) * 0.05),
         "experts_down": _typed(table, rng.standard_normal((experts, hidden, ffn)) * 0.05)}
    if scaled:
        w["expert_scale"] = (1 + 0.2 * rng.standard_normal(experts)).astype(np.float32)
    return w, rng.standard_normal(hidden).astype(np.float32)


def cpu_values(low, c, weights, x) -> dict:
    """The values that the step's launches store, by the CPU target."""
    cpu = CpuTarget(low, 64)
    for name, v in weights.items():
        for kind in ("weight", "table"):
            if f"{kind}:{name}" in low.buffers:
                cpu.write(f"{kind}:{name}", v.ravel())
    cpu.write("value:x", x)
    cpu.run()
    return {n: np.array(cpu.read(n)) for n in low.buffers if n.startswith("value:") and n != "value:x"}
