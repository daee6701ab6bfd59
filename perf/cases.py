"""The work that programs give this framework, as cases to measure: each kind
of step and kernel call through its public entry points, over the sizes it
is used at.

Kinds of case:

- ``decode``: one token of one sequence (``DecodeSession``), its step
  captured once as a HIP graph and replayed; over a ring or a paged pool.
- ``batch``: one token of each of several sequences at their own positions
  (``DecodeRows``), its step captured once and replayed.
- ``prefill``: the prompts of one or more sequences (``PrefillSession``).
- ``attend``: causal attention alone, a chunk of a prompt over what the ring
  already holds (``Kernels.prefill_attend``).
- ``gemv``: a matvec alone (``Kernels.gemv``).
- ``rows``: RMSNorm or softmax of rows alone (``Kernels.rmsnorm``,
  ``Kernels.softmax``).
- ``moe``: a routed-experts step of one row (a planned program run by
  ``Engine``).

The models are the repository's 1B-class decoder (of which most cases run one
or two layers and the head) and its tiny f32 one.  Outputs are the device
buffers that hold them, viewed as tensors: nothing is copied.
"""

from __future__ import annotations

import dataclasses
import math

import numpy as np
import torch

from furykernel_amd import kernels as fk
from furykernel_amd import runtime
from furykernel_amd.decode import DecodeSession
from furykernel_amd.engine import Engine
from furykernel_amd.lower import lower_plan
from furykernel_amd.prefill import DecodeRows, PrefillSession, weight_image
from furykernel_amd.program.build import program
from furykernel_amd.program.check import check_program
from furykernel_amd.program.decoder import ONE_B, TINY_GQA
from furykernel_amd.program.graph import F16, F32, whole_row
from furykernel_amd.program.plan import PlanOptions, plan

HEAD = 64                      # the 1B model's heads
LAYER_WEIGHTS = ("q_proj", "k_proj", "v_proj", "o_proj", "gate_proj", "up_proj", "down_proj")


# The cases ------------------------------------------------------------------------


def listed():
    return [
        # A token of a long conversation with the whole 1B model: the ring
        # full, every weight read once.
        {"name": "decode-1b-4096", "kind": "decode", "model": "1b", "layers": 16, "position": 4095, "block": 0},
        # A token early in a conversation, the cache a paged pool.
        {"name": "decode-paged-300", "kind": "decode", "model": "1b", "layers": 2, "position": 300, "block": 64},
        # A few conversations decoded together.
        {"name": "batch-8", "kind": "batch", "rows": 8, "layers": 2, "longest": 4095},
        # Many short conversations decoded together, an odd number of them.
        {"name": "batch-41", "kind": "batch", "rows": 41, "layers": 2, "longest": 700},
        # A short prompt: the time to the first token of a chat turn.
        {"name": "prefill-1x100", "kind": "prefill", "seqs": 1, "seq_rows": 100, "layers": 2, "cache": "f16",
         "block": 0},
        # Two ordinary prompts together, bf16 caches.
        {"name": "prefill-2x700-bf16", "kind": "prefill", "seqs": 2, "seq_rows": 700, "layers": 2, "cache": "bf16",
         "block": 0},
        # Long prompts through the whole 1B model.
        {"name": "prefill-4x2048", "kind": "prefill", "seqs": 4, "seq_rows": 2048, "layers": 16, "cache": "f16",
         "block": 0},
        # The attention of a prompt's next 512 rows over the 3072 before them.
        {"name": "attend-chunk-512", "kind": "attend", "seqs": 1, "seq_rows": 512, "start": 3072, "heads": 32,
         "kv_heads": 8, "cache": "f16", "window": 0},
        # A large int8 weight-only layer for one token.
        {"name": "gemv-i8-8192", "kind": "gemv", "wtype": "i8", "n": 8192, "k": 8192},
        # An f16 layer of ragged size for one token.
        {"name": "gemv-f16-5000x3080", "kind": "gemv", "wtype": "f16", "n": 5000, "k": 3080},
        # The probabilities of a few rows: the smallest call, launch and
        # latency.
        {"name": "softmax-64x4096", "kind": "rows", "op": "softmax", "rows": 64, "width": 4096},
        # A token through a mixture of experts, two of sixteen taken.
        {"name": "moe-2-of-16", "kind": "moe", "hidden": 2048, "experts": 16, "ffn": 1024, "k": 2},
    ]


def _log(rng, lo, hi):
    """A whole number of lo .. hi, spread over its logarithm."""
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(["decode", "batch", "batch", "prefill", "prefill", "attend", "gemv", "rows", "moe"])
    if kind == "decode":
        if rng.random() < 0.2:
            return {"kind": kind, "model": "tiny", "layers": rng.randint(1, 2), "position": _log(rng, 1, 255),
                    "block": 0}
        return {"kind": kind, "model": "1b", "layers": rng.randint(1, 3), "position": _log(rng, 1, 4095),
                "block": rng.choice([0, 0, 16, 64])}
    if kind == "batch":
        return {"kind": kind, "rows": _log(rng, 1, 64), "layers": 1, "longest": _log(rng, 16, 4095)}
    if kind == "prefill":
        cache = rng.choice(["f16", "f16", "bf16"])
        return {"kind": kind, "seqs": rng.choice([1, 1, 2, 3, 4]), "seq_rows": _log(rng, 8, 1500), "layers": 1,
                "cache": cache, "block": rng.choice([0, 0, 64]) if cache == "f16" else 0}
    if kind == "attend":
        seqs = rng.choice([1, 1, 2, 4])
        rows = 256 * _log(rng, 1, 8)
        kv_heads = rng.choice([4, 8])
        return {"kind": kind, "seqs": seqs, "seq_rows": rows, "start": 64 * rng.randint(0, 32),
                "heads": kv_heads * rng.choice([1, 2, 4, 4]), "kv_heads": kv_heads,
                "cache": rng.choice(["f16", "bf16"]), "window": rng.choice([0, 0, _log(rng, 64, 2048)])}
    if kind == "gemv":
        wtype = rng.choice(["f32", "f16", "i8"])
        pack = fk.GEMV_PACK[wtype]
        return {"kind": kind, "wtype": wtype, "n": _log(rng, 256, 16384),
                "k": pack * _log(rng, 256 // pack, 8192 // pack)}
    if kind == "rows":
        return {"kind": kind, "op": rng.choice(["rmsnorm", "softmax"]), "rows": _log(rng, 1, 4096),
                "width": 4 * _log(rng, 16, 4096)}
    return {"kind": kind, "hidden": 64 * rng.randint(8, 32), "experts": rng.choice([8, 16, 32]),
            "ffn": 64 * rng.randint(4, 16), "k": rng.randint(1, 4)}


# What a program has in hand --------------------------------------------------------


class _Framework:
    """The device and its kernels, opened once a process."""

    device = None
    kernels = None


def _framework():
    if _Framework.device is None:
        torch.cuda.init()
        _Framework.device = runtime.Device(0)
        _Framework.kernels = fk.Kernels(_Framework.device)
    return _Framework.device, _Framework.kernels


class _Owner:
    """Gives back what a state holds, once neither the state nor any view of
    its buffers is left."""

    def __init__(self):
        self.closing = []

    def __del__(self):
        if self.closing:
            torch.cuda.synchronize()
        for close in self.closing:
            close()


class _Span:
    """Device memory as torch takes it; a tensor over it keeps its owner."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": typestr, "data": (int(ptr), False),
                                         "strides": None, "version": 2}


_VIEWS = {"f32": ("<f4", None), "f16": ("<f2", None), "bf16": ("<i2", torch.bfloat16), "u32": ("<i4", None)}


def _view(owner, buf, dtype, shape):
    """A buffer of the framework's as a tensor over the same memory."""
    typestr, as_type = _VIEWS[dtype]
    t = torch.as_tensor(_Span(owner, buf.ptr, shape, typestr), device="cuda")
    return t if as_type is None else t.view(as_type)


class _State:
    """A pass (`go`), the outputs it leaves, and what holds its memory."""

    def __init__(self, go, outputs, owner):
        self.go, self.outputs, self.owner = go, outputs, owner


def run(state):
    state.go()
    return state.outputs


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 2 + 1)


def _normal(gen, dims, std, dtype):
    return (torch.randn(dims, generator=gen, device="cuda") * std).to(dtype)


def _host(t):
    return t.cpu().numpy()


def prepare(case, seed):
    return _PREPARE[case["kind"]](case, int(seed))


def exact(case, seed):
    """What `run` returns, computed in binary64 from the same inputs."""
    make = _EXACT[case["kind"]]
    return make(case, int(seed))


# A decoder's weights, tokens and caches, made from the seed ---------------------------


def _dims(case):
    if case["kind"] == "decode":
        return TINY_GQA if case["model"] == "tiny" else ONE_B
    if case["kind"] == "batch":
        return dataclasses.replace(ONE_B, slots=case["rows"])
    return dataclasses.replace(ONE_B, slots=case["seqs"], cache_elem=case["cache"])


def _weights(dims, layers, gen):
    """Gains about 1, projections of normals that keep a row's size, the
    unembedding tied to the embedding."""
    wt = torch.float32 if dims.weight_type == F32 else torch.float16
    shapes = {"q_proj": (dims.q_width, dims.d_model), "k_proj": (dims.kv_width, dims.d_model),
              "v_proj": (dims.kv_width, dims.d_model), "o_proj": (dims.d_model, dims.q_width),
              "gate_proj": (dims.ffn, dims.d_model), "up_proj": (dims.ffn, dims.d_model),
              "down_proj": (dims.d_model, dims.ffn)}
    std = 0.02 if dims.d_model >= 1024 else 0.1
    out = {}
    for i in range(layers):
        for norm in ("attn_norm", "mlp_norm"):
            out[f"l{i}_{norm}"] = 1 + _normal(gen, (dims.d_model,), 0.1, torch.float32)
        for name in LAYER_WEIGHTS:
            out[f"l{i}_{name}"] = _normal(gen, shapes[name], std, wt)
    out["final_norm"] = 1 + _normal(gen, (dims.d_model,), 0.1, torch.float32)
    embed = _normal(gen, (dims.vocab, dims.d_model), 0.5, torch.float32)
    out["embed"] = embed.to(wt)
    out["lm_head"] = (embed * 0.04).to(wt)
    return out


def _tokens(dims, count, gen):
    return torch.randint(0, dims.vocab, (count,), generator=gen, device="cuda")


def _caches(dims, layers, gen):
    """[slots][kv heads][positions][head dimension] f16, one a layer and side."""
    shape = (dims.slots, dims.kv_heads, dims.context, dims.head_dim)
    return [[_normal(gen, shape, 1.0, torch.float16) for _ in range(layers)] for _ in range(2)]


def _session(owner, session):
    """The session, closed with its owner."""
    owner.closing.append(session.close)
    return session


def _graph(owner, graph):
    owner.closing.insert(0, graph.destroy)
    return graph


def _buffers(owner, *buffers):
    owner.closing += [b.free for b in buffers if b is not None]


# decode: a token of one sequence --------------------------------------------------------


def _paging(case, dims):
    return (case["block"], dims.context // case["block"] + 16) if case["block"] else None


def _table(case, dims, seed):
    block, blocks = _paging(case, dims)
    return np.random.default_rng(seed).permutation(blocks)[:dims.context // block].astype(np.uint32)


def _prepare_decode(case, seed):
    dev, ks = _framework()
    own = _Owner()
    dims, layers, pos = _dims(case), case["layers"], case["position"]
    gen = _generator(seed)
    weights = _weights(dims, layers, gen)
    token = int(_tokens(dims, 1, gen))
    caches = _caches(dims, layers, gen)
    paging = _paging(case, dims)
    s = _session(own, DecodeSession(dev, ks, dims, PlanOptions(store_gelus=True), layers=layers, tuned=True,
                                    paging=paging))
    s.engine.write_weights({name: _host(w) for name, w in weights.items()})
    rows = {}
    for side, per_layer in zip("kv", caches):
        rows[side] = []
        for i, c in enumerate(per_layer):
            buf = s.engine.buffers[f"cache:l{i}_{side}_cache"]
            if paging is None:
                held = _view(own, buf, "f16", c.shape)
                held.copy_(c)
                rows[side].append(held[0, :, pos])
            else:
                block, blocks = paging
                table = _table(case, dims, seed)
                held = _view(own, buf, "f16", (blocks, dims.kv_heads, block, dims.head_dim))
                held.zero_()
                held[torch.from_numpy(table.astype(np.int64)).cuda()] = \
                    c[0].view(dims.kv_heads, -1, block, dims.head_dim).transpose(0, 1)
                rows[side].append(held[int(table[pos // block]), :, pos % block])
    torch.cuda.synchronize()
    s.set_position(pos, token=token, table=None if paging is None else _table(case, dims, seed))
    graph = _graph(own, s.engine.capture())
    outputs = {"logits": _view(own, s.engine.buffers["value:logits"], "f32", (dims.vocab,)),
               "token": _view(own, s.engine.buffers["value:token"], "u32", (1,)), **rows}
    return _State(graph.replay, outputs, own)


def _exact_decode(case, seed):
    dims, layers, pos = _dims(case), case["layers"], case["position"]
    gen = _generator(seed)
    weights = _weights(dims, layers, gen)
    token = _tokens(dims, 1, gen)
    caches = _caches(dims, layers, gen)
    logits, ks, vs = _decoder(dims, layers, weights, token, [(0, 1, pos, 0)], caches)
    return {"logits": logits[0], "token": None, "k": [k[0] for k in ks], "v": [v[0] for v in vs]}


# batch: a token of each of several sequences -----------------------------------------------


def _batch_positions(case):
    """Positions spread over the logarithm up to the longest, the longest
    among them."""
    m, longest = case["rows"], case["longest"]
    low = max(1, longest // 16)
    return [round(low * (longest / low) ** ((i + 1) / m)) for i in range(m)]


def _prepare_batch(case, seed):
    dev, ks = _framework()
    own = _Owner()
    dims, layers, m = _dims(case), case["layers"], case["rows"]
    gen = _generator(seed)
    weights = _weights(dims, layers, gen)
    tokens = _tokens(dims, m, gen)
    caches = _caches(dims, layers, gen)
    pos = _batch_positions(case)
    s = _session(own, DecodeRows(dev, ks, dims, pos, list(range(m)), layers=layers))
    s.write_weights({name: _host(w) for name, w in weights.items()})
    rows = {}
    for side, per_layer in zip("kv", caches):
        rows[side] = []
        for i, c in enumerate(per_layer):
            held = _view(own, s.engine.buffers[f"cache:l{i}_{side}_cache"], "f16", (dims.slots + 1, *c.shape[1:]))
            held[:m].copy_(c)
            held[m].zero_()
            rows[side].append([held[r, :, p] for r, p in enumerate(pos)])
    torch.cuda.synchronize()
    s.set_tokens(_host(tokens))
    graph = _graph(own, s.graph())
    # Row r of the batch is row real[r] of the step; the rows are evenly
    # apart, so the batch is a strided view.
    apart = int(s.real[1] - s.real[0]) if m > 1 else 1
    logits = _view(own, s.engine.buffers["value:logits"], "f32", (s.rows, dims.vocab))[::apart][:m]
    token = _view(own, s.engine.buffers["value:token"], "u32", (s.rows,))[::apart][:m]
    # the rows that the longest sequence stored: every layer's
    stored = {side: [per_row[-1] for per_row in rows[side]] for side in rows}
    stored.update({side + "_first": [per_row[0] for per_row in rows[side]] for side in rows})
    return _State(graph.replay, {"logits": logits, "token": token, **stored}, own)


def _exact_batch(case, seed):
    dims, layers, m = _dims(case), case["layers"], case["rows"]
    gen = _generator(seed)
    weights = _weights(dims, layers, gen)
    tokens = _tokens(dims, m, gen)
    caches = _caches(dims, layers, gen)
    runs = [(r, 1, p, r) for r, p in enumerate(_batch_positions(case))]
    logits, ks, vs = _decoder(dims, layers, weights, tokens, runs, caches)
    return {"logits": logits, "token": None, "k": [k[-1] for k in ks], "v": [v[-1] for v in vs],
            "k_first": [k[0] for k in ks], "v_first": [v[0] for v in vs]}


# prefill: the prompts of one or more sequences -----------------------------------------------


def _synthetic(case):
    """The whole model's prefill takes weights made on the device: packing
    2 GB of host weights for each state would take longer than all its runs."""
    return case["layers"] > 4


def _prepare_prefill(case, seed):
    dev, ks = _framework()
    own = _Owner()
    dims, layers, seqs, n = _dims(case), case["layers"], case["seqs"], case["seq_rows"]
    gen = _generator(seed)
    block = case["block"]
    paging = (block, seqs * dims.context // block) if block else None
    s = _session(own, PrefillSession(dev, ks, dims, seqs, n, layers=layers, paging=paging))
    if _synthetic(case):
        s.init_synthetic(seed=seed)
        ends = _weights(dims, 0, gen)
        for name, src in (("weight:embed", "embed"), ("tiled:lm_head", "lm_head")):
            s.engine.write(name, weight_image(s.lowered, name, {src: _host(ends[src])}))
    else:
        s.write_weights({name: _host(w) for name, w in _weights(dims, layers, gen).items()})
    rows = {}
    for side in "kv":
        rows[side] = []
        for i in range(layers):
            buf = s.engine.buffers[f"cache:l{i}_{side}_cache"]
            per = dims.kv_heads * HEAD * (block or dims.context)
            units = buf.size // (2 * per)
            held = _view(own, buf, case["cache"], (units, dims.kv_heads, block or dims.context, HEAD))
            held.zero_()
            rows[side].append(held[:paging[1]] if block else held[:seqs, :, :n])
    torch.cuda.synchronize()
    s.set_tokens(_host(_tokens(dims, seqs * n, gen)))
    graph = _graph(own, s.graph())
    runs = s.rows // s.run_rows
    logits = _view(own, s.engine.buffers["value:logits"], "f32", (runs, s.run_rows, dims.vocab))[:seqs, :n]
    token = _view(own, s.engine.buffers["value:token"], "u32", (runs, s.run_rows))[:seqs, :n]
    return _State(graph.replay, {"logits": logits, "token": token, **rows}, own)


def _exact_prefill(case, seed):
    if _synthetic(case):
        return None
    dims, layers, seqs, n = _dims(case), case["layers"], case["seqs"], case["seq_rows"]
    gen = _generator(seed)
    weights = _weights(dims, layers, gen)
    tokens = _tokens(dims, seqs * n, gen)
    runs = [(i * n, n, 0, i) for i in range(seqs)]
    logits, ks, vs = _decoder(dims, layers, weights, tokens, runs, None,
                              torch.bfloat16 if case["cache"] == "bf16" else torch.float16)
    out = {"logits": logits.view(seqs, n, -1), "token": None}
    for side, got in (("k", ks), ("v", vs)):
        if case["block"]:
            out[side] = None   # a pool's blocks are in the session's own order
        else:
            out[side] = [t.view(seqs, n, dims.kv_heads, HEAD).transpose(1, 2).contiguous() for t in got]
    return out


# The decoder in binary64 ----------------------------------------------------------------


def _norm(x, gain, eps):
    return x * (x.square().mean(-1, keepdim=True) + eps).rsqrt() * gain.double()


def _rope(x, pos, theta):
    """NeoX halves turned by binary32 angles (the program's definition: the
    position times the frequency, rounded to binary32)."""
    half = x.shape[-1] // 2
    freq = torch.tensor([math.pow(theta, -i / half) for i in range(half)], dtype=torch.float32, device="cuda")
    angle = (pos.float()[:, None] * freq).double()[:, None]
    c, s = angle.cos(), angle.sin()
    a, b = x[..., :half], x[..., half:]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _attention(q, k, v, pos, scale, window=0):
    """q [n, heads, d] at positions pos over k, v [kv heads, keys, d] of
    positions 0 .. keys - 1, causal, in binary64."""
    n, heads, d = q.shape
    keys = k.shape[1]
    at = torch.arange(keys, device="cuda")
    dead = at[None] > pos[:, None]
    if window:
        dead |= at[None] <= pos[:, None] - window
    out = torch.empty_like(q)
    group = heads // k.shape[0]
    for h in range(heads):
        score = (q[:, h] @ k[h // group].t()).mul_(scale).masked_fill_(dead, -math.inf)
        out[:, h] = torch.softmax(score, -1) @ v[h // group]
    return out


def _decoder(dims, layers, weights, tokens, runs, caches, cache_type=torch.float16):
    """The step's logits and each layer's new k and v rows (as its cache
    holds them).  `runs`: (first row, rows, first position, slot)."""
    d = dims.head_dim
    pos = torch.cat([torch.arange(p, p + n, device="cuda") for _, n, p, _ in runs])
    x = weights["embed"][tokens].double()
    rows = x.shape[0]
    new_k, new_v = [], []
    for i in range(layers):
        def w(name):
            return weights[f"l{i}_{name}"]

        def linear(a, name):
            return a @ w(name).double().t()

        a = _norm(x, w("attn_norm"), dims.eps)
        q = _rope(linear(a, "q_proj").view(rows, dims.heads, d), pos, dims.rope_theta)
        k = _rope(linear(a, "k_proj").view(rows, dims.kv_heads, d), pos, dims.rope_theta).to(cache_type).double()
        v = linear(a, "v_proj").view(rows, dims.kv_heads, d).to(cache_type).double()
        new_k.append(k)
        new_v.append(v)
        o = torch.empty_like(q)
        for first, n, p, slot in runs:
            at = slice(first, first + n)
            kk, vv = k[at].transpose(0, 1), v[at].transpose(0, 1)
            if caches is not None:
                kk = torch.cat([caches[0][i][slot, :, :p].double(), kk], 1)
                vv = torch.cat([caches[1][i][slot, :, :p].double(), vv], 1)
            o[at] = _attention(q[at], kk, vv, pos[at], 1 / math.sqrt(d))
        x = x + linear(o.reshape(rows, -1), "o_proj")
        m = _norm(x, w("mlp_norm"), dims.eps)
        gate = linear(m, "gate_proj")
        x = x + linear(torch.nn.functional.silu(gate) * linear(m, "up_proj"), "down_proj")
    logits = _norm(x, weights["final_norm"], dims.eps) @ weights["lm_head"].double().t()
    return logits, new_k, new_v


# attend: a chunk of a prompt over what the ring holds --------------------------------------


def _attend_length(case):
    return -(-(case["start"] + case["seq_rows"]) // 1024) * 1024


def _attend_inputs(case, seed):
    gen = _generator(seed)
    seqs, rows = case["seqs"], case["seqs"] * case["seq_rows"]
    ct = torch.bfloat16 if case["cache"] == "bf16" else torch.float16
    q = _normal(gen, (rows, case["heads"] * HEAD), 1.0, torch.float16)
    kc, vc = (_normal(gen, (seqs, case["kv_heads"], _attend_length(case), HEAD), 1.0, ct) for _ in range(2))
    return q, kc, vc


def _prepare_attend(case, seed):
    dev, ks = _framework()
    own = _Owner()
    q, kc, vc = _attend_inputs(case, seed)
    seqs, n = case["seqs"], case["seq_rows"]
    positions = np.tile(np.arange(case["start"], case["start"] + n, dtype=np.uint32), seqs)
    slots = np.repeat(np.arange(seqs, dtype=np.uint32), n)
    held = [dev.upload(_host(t.view(torch.int16))) for t in (q, kc, vc)] + [dev.upload(positions), dev.upload(slots)]
    out = dev.alloc(q.numel() * 2)
    args = (*held, out, seqs * n, case["heads"], case["kv_heads"], _attend_length(case), seqs, 1 / math.sqrt(HEAD))
    options = {"window": case["window"], "cache_bf16": case["cache"] == "bf16"}
    _buffers(own, *held, out)
    return _State(lambda: ks.prefill_attend(*args, **options), _view(own, out, "f16", (q.numel(),)), own)


def _tiled(x):
    """[rows, columns] in the tile layout that the matrix-core kernels read:
    slabs of 256 rows, each a chunk of 16 rows x 32 columns after another,
    a chunk's 16-byte units swizzled by its row div 4."""
    r, k = x.shape
    t = x.view(r // 256, 16, 16, k // 32, 4, 8).permute(0, 3, 1, 2, 4, 5)
    row = torch.arange(16, device="cuda")
    unit = torch.arange(4, device="cuda")[None] ^ ((row // 4) % 4)[:, None]
    return t[:, :, :, row[:, None], unit].reshape(-1)


def _exact_attend(case, seed):
    q, kc, vc = _attend_inputs(case, seed)
    seqs, n = case["seqs"], case["seq_rows"]
    pos = torch.arange(case["start"], case["start"] + n, device="cuda")
    out = torch.empty(q.shape, dtype=torch.float64, device="cuda")
    for i in range(seqs):
        at = slice(i * n, (i + 1) * n)
        keys = case["start"] + n
        out[at] = _attention(q[at].double().view(n, case["heads"], HEAD), kc[i, :, :keys].double(),
                             vc[i, :, :keys].double(), pos, 1 / math.sqrt(HEAD), case["window"]).view(n, -1)
    return _tiled(out)


# gemv ---------------------------------------------------------------------------------


def _gemv_inputs(case, seed):
    gen = _generator(seed)
    n, k, wtype = case["n"], case["k"], case["wtype"]
    if wtype == "i8":
        w = torch.randint(-127, 128, (n, k), generator=gen, device="cuda", dtype=torch.int8)
        scale = 1e-3 * (1 + torch.rand((n,), generator=gen, device="cuda"))
        return w, _normal(gen, (k,), 1.0, torch.float16), scale
    w = _normal(gen, (n, k), 0.02, torch.float32 if wtype == "f32" else torch.float16)
    return w, _normal(gen, (k,), 1.0, torch.float32), None


def _prepare_gemv(case, seed):
    dev, ks = _framework()
    own = _Owner()
    n, k = case["n"], case["k"]
    held = [None if t is None else dev.upload(_host(t)) for t in _gemv_inputs(case, seed)]
    w, x, scale = held
    y = dev.alloc(n * 4)
    _buffers(own, *held, y)
    return _State(lambda: ks.gemv(w, x, y, n, k, wtype=case["wtype"], scale=scale), _view(own, y, "f32", (n,)), own)


def _exact_gemv(case, seed):
    w, x, scale = _gemv_inputs(case, seed)
    y = w.double() @ x.double()
    return y if scale is None else y * scale.double()


# rows: RMSNorm and softmax ------------------------------------------------------------------


def _rows_inputs(case, seed):
    gen = _generator(seed)
    x = _normal(gen, (case["rows"], case["width"]), 2.0, torch.float32)
    return x, 1 + _normal(gen, (case["width"],), 0.1, torch.float32)


def _prepare_rows(case, seed):
    dev, ks = _framework()
    own = _Owner()
    x, gain = _rows_inputs(case, seed)
    bx, bg, by = dev.upload(_host(x)), dev.upload(_host(gain)), dev.alloc(x.numel() * 4)
    rows, width = case["rows"], case["width"]
    if case["op"] == "softmax":
        def go():
            ks.softmax(bx, by, rows, width)
    else:
        def go():
            ks.rmsnorm(bx, bg, by, rows, width)
    _buffers(own, bx, bg, by)
    return _State(go, _view(own, by, "f32", (rows, width)), own)


def _exact_rows(case, seed):
    x, gain = _rows_inputs(case, seed)
    return torch.softmax(x.double(), -1) if case["op"] == "softmax" else _norm(x.double(), gain, 1e-6)


# moe: a routed-experts step ----------------------------------------------------------------


def _moe_program(case):
    hidden, experts, ffn, k = case["hidden"], case["experts"], case["ffn"], case["k"]

    def body(b):
        x = b.input("x", whole_row(hidden), F32)
        g = b.weight("moe_norm", [hidden], F32)
        router = b.weight("router", [experts, hidden], F16)
        scale = b.weight("expert_scale", [experts], F32)
        gu = b.table("experts_gate_up", experts, [2 * ffn, hidden], F16)
        dn = b.table("experts_down", experts, [hidden, ffn], F16)
        cn = b.rmsnorm("moe_in", 1e-6, g, 1.0, x)
        ids, ws = b.route("route", k, scale, b.linear("router_logits", router, 0, cn))
        act = b.gated_gelu("experts_act", b.linear_routed("experts_gate_up_out", gu, ids, cn))
        s = b.combine_ranks("experts_sum", ws, b.linear_routed("experts_out", dn, ids, act))
        b.output("y", b.add("y", x, s))
    return check_program(program("moe", body))


def _moe_inputs(case, seed):
    hidden, experts, ffn = case["hidden"], case["experts"], case["ffn"]
    gen = _generator(seed)
    weights = {"moe_norm": 1 + _normal(gen, (hidden,), 0.1, torch.float32),
               "router": _normal(gen, (experts, hidden), 0.05, torch.float16),
               "expert_scale": 1 + _normal(gen, (experts,), 0.1, torch.float32),
               "experts_gate_up": _normal(gen, (experts, 2 * ffn, hidden), 0.02, torch.float16),
               "experts_down": _normal(gen, (experts, hidden, ffn), 0.02, torch.float16)}
    return weights, _normal(gen, (hidden,), 1.0, torch.float32)


def _prepare_moe(case, seed):
    dev, ks = _framework()
    own = _Owner()
    weights, x = _moe_inputs(case, seed)
    checked = _moe_program(case)
    engine = _session(own, Engine(dev, ks, lower_plan(checked, plan(PlanOptions(), checked))))
    engine.write_weights({name: _host(w) for name, w in weights.items()})
    engine.write("value:x", _host(x))
    graph = _graph(own, engine.capture())
    return _State(graph.replay, _view(own, engine.buffers["value:y"], "f32", (case["hidden"],)), own)


def _exact_moe(case, seed):
    weights, x = _moe_inputs(case, seed)
    w = {name: t.double() for name, t in weights.items()}
    x = x.double()
    a = _norm(x, w["moe_norm"], 1e-6)
    top, ids = torch.topk(w["router"] @ a, case["k"])
    share = torch.softmax(top, -1) * w["expert_scale"][ids]
    y = x.clone()
    for p, e in zip(share, ids.tolist()):
        h = w["experts_gate_up"][e] @ a
        gate, up = h[:case["ffn"]], h[case["ffn"]:]
        y += p * (w["experts_down"][e] @ (torch.nn.functional.gelu(gate, approximate="tanh") * up))
    return y


_PREPARE = {"decode": _prepare_decode, "batch": _prepare_batch, "prefill": _prepare_prefill,
            "attend": _prepare_attend, "gemv": _prepare_gemv, "rows": _prepare_rows, "moe": _prepare_moe}
_EXACT = {"decode": _exact_decode, "batch": _exact_batch, "prefill": _exact_prefill, "attend": _exact_attend,
          "gemv": _exact_gemv, "rows": _exact_rows, "moe": _exact_moe}


# What a pass cannot do without ---------------------------------------------------------------


def _keys_read(first, n, window=0):
    """Keys read by n rows from position `first`, each its own (causal)."""
    total = 0
    for p in range(first, first + n):
        total += min(p + 1, window) if window else p + 1
    return total


def _decoder_work(case, rows, contexts, pairs):
    """`rows` rows; `contexts`: cached and new positions whose k and v are
    read or written; `pairs`: (row, key) pairs of the attention."""
    dims, layers = _dims(case), case["layers"]
    elem = 4 if dims.weight_type == F32 else 2
    layer = dims.layer_params() - 2 * dims.d_model
    head = dims.vocab * dims.d_model
    return {"bytes": elem * (layers * layer + head + rows * dims.d_model) + 4 * rows * dims.vocab
            + layers * contexts * dims.kv_width * 2 * 2,
            "flops": 2 * rows * (layers * layer + head) + layers * pairs * dims.q_width * 4}


def work(case):
    kind = case["kind"]
    if kind == "decode":
        return _decoder_work(case, 1, case["position"] + 1, case["position"] + 1)
    if kind == "batch":
        held = sum(p + 1 for p in _batch_positions(case))
        return _decoder_work(case, case["rows"], held, held)
    if kind == "prefill":
        rows = case["seqs"] * case["seq_rows"]
        return _decoder_work(case, rows, rows, case["seqs"] * _keys_read(0, case["seq_rows"]))
    if kind == "attend":
        rows, keys = case["seqs"] * case["seq_rows"], case["start"] + case["seq_rows"]
        if case["window"]:
            keys = min(keys, case["seq_rows"] + case["window"])
        pairs = case["seqs"] * _keys_read(case["start"], case["seq_rows"], case["window"])
        return {"bytes": 2 * rows * case["heads"] * HEAD * 2 + 2 * case["seqs"] * keys * case["kv_heads"] * HEAD * 2,
                "flops": pairs * case["heads"] * HEAD * 4}
    if kind == "gemv":
        elem, x = {"f32": (4, 4), "f16": (2, 4), "i8": (1, 2)}[case["wtype"]]
        n, k = case["n"], case["k"]
        return {"bytes": n * k * elem + k * x + n * 4 * (2 if case["wtype"] == "i8" else 1), "flops": 2 * n * k}
    if kind == "rows":
        count = case["rows"] * case["width"]
        return {"bytes": 8 * count, "flops": 4 * count}
    hidden, ffn, k, experts = case["hidden"], case["ffn"], case["k"], case["experts"]
    params = experts * hidden + 3 * k * ffn * hidden
    return {"bytes": 2 * params + 12 * hidden, "flops": 2 * params}


def tolerance(case):
    """About four times what the path differs from binary64 by (measured at
    the listed sizes, given here), or what the data types give."""
    kind = case["kind"]
    if kind == "decode":
        # binary32 throughout but for the new k and v rows' rounding to f16,
        # where a sum in another order may round the other way (2.5e-5 at 16
        # layers; the logits 3e-7)
        return {"rel": 1e-4, "max": 4e-3}
    if kind in ("batch", "prefill"):
        # f16 operands of the matrix products, f16 probabilities (5.8e-4 at
        # two layers); bf16 caches round k and v to 8 bits (1.3e-3)
        deep = 4 if case["layers"] > 4 else 1
        return {"rel": deep * (5e-3 if case.get("cache") == "bf16" else 2.5e-3), "max": deep * 0.05, "differ": 0.01}
    if kind == "attend":
        return {"rel": 1.2e-3, "max": 2e-2}   # 2.9e-4: f16 probabilities and outputs
    return {"rel": 2e-6, "max": 2e-5}         # binary32 sums (1e-7)
