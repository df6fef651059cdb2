"""The workloads whose speed matters to a user of this framework, as data and four functions.

Every case is one pass through the public operators exactly as a training (or evaluation) program calls them:

  attention   attention_func / MLA on one device, forward or forward + backward
  ring        ring_attention_local, one GPU's share of context-parallel attention, forward + backward
  combine     the log2 merge of two partial attention results
  gqa_prologue  per-head RMSNorm + rotary embedding of q and k, forward + backward
  mla_prologue  rotary embedding + assembly of query / key / value states, forward + backward

`listed()` is a fixed selection over the whole range of sizes, `draw(rng)` takes further cases from the same ranges,
`prepare` makes what the program has in hand before the call, `run` is the pass, `work` what the pass cannot do
without (inputs read once, outputs written once; matrix products counted as the algorithm needs them, without
recomputation) and `tolerance` how far another correct implementation at the same precision may be off.

Imported with the root of the tree under measurement as the working folder.
"""

import math
import os
import sys

import torch

_PACKAGE = os.path.join(os.getcwd(), "pith-train_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

from pithtrain_amd.operators.mla import MLA, attention_func  # noqa: E402
from pithtrain_amd.operators.mla_assemble import mla_assemble_qkv  # noqa: E402
from pithtrain_amd.operators.norm_rope import qk_norm_rope  # noqa: E402
from pithtrain_amd.operators.ring_attention.local import ring_attention_local, ring_schedule  # noqa: E402
from pithtrain_amd.operators.ring_attention.mla import _online_softmax_combine_log2  # noqa: E402

VALUE_DIM = {64: 64, 128: 128, 192: 128}  # value features that go with a key dim
ROPE_DIM = 64  # rotary features of the MLA key


def _attention(name, b, s, hq, hkv, d, causal=True, backward=True):
    return {"name": name, "kind": "attention", "b": b, "s": s, "hq": hq, "hkv": hkv, "d": d, "causal": causal, "backward": backward}


def _ring(name, b, s, hq, hkv, d, cp, rank, layout, split_key=False):
    return {"name": name, "kind": "ring", "b": b, "s": s, "hq": hq, "hkv": hkv, "d": d, "cp": cp, "rank": rank,
            "layout": layout, "split_key": split_key}  # fmt: skip


def listed():
    return [
        # The smallest call: one layer of a toy model (8 q / 2 kv heads, 256 tokens) as in unit tests and debugging runs;
        # all launches and host work.
        _attention("attention_small", 1, 256, 8, 2, 128),
        # A small dense model with 64-feature heads and a micro-batch of two: an ordinary pretraining step.
        _attention("attention_head64", 2, 2048, 16, 4, 64),
        # A Qwen3-30B-A3B layer (32 q / 4 kv heads) without context parallelism at the usual pretraining length.
        _attention("gqa_layer_4k", 1, 4096, 32, 4, 128),
        # Validation of the same layer on a batch whose length is nobody's multiple: forward only.
        _attention("gqa_eval_ragged", 3, 1999, 32, 4, 128, backward=False),
        # A DeepSeek-V2-Lite layer (16 heads, 192/128) without context parallelism, forward and backward.
        _attention("mla_layer_4k", 1, 4096, 16, 16, 192),
        # One rank's share of Qwen3-30B-A3B at 32K tokens over 4 ranks: the headline workload.
        _ring("ring_gqa_32k", 1, 8192, 32, 4, 128, 4, 1, "zigzag"),
        # One rank's share of the MLA layer at 16K tokens over 4 ranks.
        _ring("ring_mla_16k", 1, 4096, 16, 16, 192, 4, 1, "zigzag"),
        # The largest: long-context GQA (64 q / 4 kv heads) at 131K tokens over 8 ranks.
        _ring("ring_gqa_131k", 1, 16384, 64, 4, 128, 8, 3, "zigzag"),
        # A short MLA ring in the default (contiguous) layout, with the key in two parts, odd chunk length: fine-tuning on
        # short documents.
        _ring("ring_mla_split_key_short", 1, 1021, 16, 16, 192, 4, 2, "contiguous", split_key=True),
        # The merge of two partial results at the size of a ring step (4096 positions x 32 heads).
        {"name": "combine_4k", "kind": "combine", "b": 1, "s": 4096, "h": 32, "d": 128, "partial": "bf16"},
        # What runs before the attention of a Qwen3 layer at the 32K share.
        {"name": "gqa_prologue_8k", "kind": "gqa_prologue", "b": 1, "s": 8192, "hq": 32, "hkv": 4, "d": 128, "weight": "bf16"},
        # What runs before the attention of an MLA layer at the 16K share.
        {"name": "mla_prologue_4k", "kind": "mla_prologue", "b": 1, "s": 4096, "h": 16},
    ]


def _log_size(rng, lo, hi):
    """A length spread evenly over its logarithm; half of them are multiples of 128 (of 16 when short), the others anything."""
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if rng.random() < 0.5:
        step = 128 if n >= 512 else 16
        n = max(step, n // step * step)
    return min(max(n, lo), hi)


def _draw_any(rng):
    kind = rng.choice(["attention", "attention", "attention", "ring", "ring", "combine", "gqa_prologue", "mla_prologue"])
    if kind == "attention":
        d = rng.choice([64, 128, 128, 192])
        heads = {64: [(4, 4), (16, 4), (16, 16), (32, 8)], 128: [(8, 2), (16, 16), (32, 4), (64, 4)], 192: [(4, 4), (16, 16), (128, 128)]}[d]
        hq, hkv = rng.choice(heads)
        s = _log_size(rng, 64, 32768)
        b = rng.choice([n for n in (1, 2, 3, 4, 8) if n * s <= 32768])
        case = _attention("", b, s, hq, hkv, d, causal=d == 192 or rng.random() < 0.75, backward=rng.random() < 0.7)
    elif kind == "ring":
        d = rng.choice([128, 128, 192])
        hq, hkv = rng.choice([(8, 2), (32, 4), (64, 4)] if d == 128 else [(4, 4), (16, 16)])
        layout = rng.choice(["zigzag", "contiguous"])
        s = _log_size(rng, 128, 16384)
        s += s % 2 if layout == "zigzag" else 0  # a zigzag chunk is two blocks
        cp = rng.choice([2, 4, 8])
        case = _ring("", 1 if s > 4096 else rng.choice([1, 2]), s, hq, hkv, d, cp, rng.randrange(cp), layout, d == 192 and rng.random() < 0.5)
    elif kind == "combine":
        case = {"kind": kind, "b": rng.choice([1, 2]), "s": _log_size(rng, 64, 16384), "h": rng.choice([8, 16, 32]), "d": 128,
                "partial": rng.choice(["bf16", "fp32"])}  # fmt: skip
    elif kind == "gqa_prologue":
        hq, hkv = rng.choice([(8, 2), (32, 4), (64, 4)])
        case = {"kind": kind, "b": rng.choice([1, 2]), "s": _log_size(rng, 64, 16384), "hq": hq, "hkv": hkv, "d": 128,
                "weight": rng.choice(["bf16", "fp32"])}  # fmt: skip
    else:
        case = {"kind": kind, "b": rng.choice([1, 2]), "s": _log_size(rng, 64, 16384), "h": rng.choice([4, 16, 32])}
    case.pop("name", None)
    return case


def draw(rng):
    """One more case of these ranges; none costs more than the largest listed one."""
    most = {m: max(work(c)[m] for c in listed()) for m in ("bytes", "flops")}
    while True:
        case = _draw_any(rng)
        w = work(case)
        if all(w[m] <= most[m] for m in most):
            return case


class _Maker:
    """Normally distributed tensors from one seed, on the GPU. q and k have unit variance, as after a per-head norm: their
    scores are then N(0, 1) after the softmax scale."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, *shape, dtype=torch.bfloat16, grad=False, std=1.0):
        x = (torch.randn(*shape, generator=self.g, device="cuda", dtype=torch.float32) * std).to(dtype)
        return x.requires_grad_(grad)


def _rotary_tables(positions, dim):
    """cos and sin [positions, dim] in bf16, the two halves alike, as the rotary modules of both model families keep them."""
    freq = 10000.0 ** (-torch.arange(0, dim, 2, device="cuda", dtype=torch.float32) / dim)
    angle = torch.arange(positions, device="cuda", dtype=torch.float32)[:, None] * freq[None, :]
    angle = torch.cat([angle, angle], dim=-1)
    return angle.cos().to(torch.bfloat16), angle.sin().to(torch.bfloat16)


def _visited(case):
    return sorted({st.kv_rank for st in ring_schedule(case["rank"], case["cp"], case["s"], case["layout"])})


def prepare(case, seed):
    m = _Maker(seed)
    kind, b, s = case["kind"], case["b"], case["s"]
    state = {"kind": kind}
    if kind == "attention":
        d, dv, bwd = case["d"], VALUE_DIM[case["d"]], case["backward"]
        q = m.normal(b, s, case["hq"], d, grad=bwd)
        k = m.normal(b, s, case["hkv"], d, grad=bwd)
        v = m.normal(b, s, case["hkv"], dv, grad=bwd)
        scale = d**-0.5
        if d == 192:
            call = MLA(case["hq"], d, dv, scale)
        else:
            causal = case["causal"]
            call = lambda q, k, v: attention_func(q, k, v, scale, causal=causal)  # noqa: E731
        state.update(q=q, k=k, v=v, call=call, dout=m.normal(b, s, case["hq"], dv) if bwd else None)
    elif kind == "ring":
        d, dv, visited = case["d"], VALUE_DIM[case["d"]], _visited(case)
        kd = d - ROPE_DIM if case["split_key"] else d
        chunks = lambda *shape: [m.normal(*shape, grad=True) if j in visited else None for j in range(case["cp"])]  # noqa: E731
        state.update(
            q=m.normal(b, s, case["hq"], d, grad=True), ks=chunks(b, s, case["hkv"], kd), vs=chunks(b, s, case["hkv"], dv),
            pes=chunks(b, s, ROPE_DIM) if case["split_key"] else None, dout=m.normal(b, s, case["hq"], dv),
            scale=d**-0.5, rank=case["rank"], cp=case["cp"], layout=case["layout"])  # fmt: skip
        state["inputs"] = [state["q"]] + [state[n][j] for n in ("ks", "vs", "pes") if state[n] is not None for j in visited]
    elif kind == "combine":
        dtype = torch.bfloat16 if case["partial"] == "bf16" else torch.float32
        h, d = case["h"], case["d"]
        state["args"] = []
        for _ in range(2):  # log2-sum-exp of a few thousand N(0, 1) scores: about 11 to 13
            state["args"] += [m.normal(b, s, h, d, dtype=dtype, std=0.1), m.normal(b, h, s, dtype=torch.float32) + 12.0]
    elif kind == "gqa_prologue":
        hq, hkv, d = case["hq"], case["hkv"], case["d"]
        wdtype = torch.bfloat16 if case["weight"] == "bf16" else torch.float32
        cos, sin = _rotary_tables(s, d)
        state.update(
            x=[m.normal(b, s, hq, d, grad=True), m.normal(b, s, hkv, d, grad=True)],
            w=[(1.0 + m.normal(d, dtype=torch.float32, std=0.1)).to(wdtype).requires_grad_(True) for _ in range(2)],
            cos=cos[None], sin=sin[None], dout=[m.normal(b, s, hq, d), m.normal(b, s, hkv, d)])  # fmt: skip
    else:
        h, nope, dv = case["h"], 128, 128
        cos, sin = _rotary_tables(s, ROPE_DIM)
        state.update(
            x=[m.normal(b, s, h, nope + ROPE_DIM, grad=True), m.normal(b, s, h, nope + dv, grad=True), m.normal(b, s, 1, ROPE_DIM, grad=True)],
            cos=cos, sin=sin, pos=torch.arange(s, device="cuda")[None].expand(b, s).contiguous(),
            dout=[m.normal(b, s, h, nope + ROPE_DIM), m.normal(b, s, h, nope + ROPE_DIM), m.normal(b, s, h, dv)])  # fmt: skip
    return state


def run(state):
    kind = state["kind"]
    if kind == "attention":
        q, k, v = state["q"], state["k"], state["v"]
        if state["dout"] is None:
            with torch.no_grad():
                return state["call"](q, k, v)
        out = state["call"](q, k, v)
        return [out.detach(), *torch.autograd.grad(out, (q, k, v), state["dout"])]
    if kind == "ring":
        out = ring_attention_local(state["q"], state["ks"], state["vs"], state["scale"], state["rank"], state["cp"], state["layout"], state["pes"])
        return [out.detach(), *torch.autograd.grad(out, state["inputs"], state["dout"])]
    if kind == "combine":
        return _online_softmax_combine_log2(*state["args"])
    if kind == "gqa_prologue":
        outs = qk_norm_rope(*state["x"], *state["w"], state["cos"], state["sin"], 1e-6)
        return [*(o.detach() for o in outs), *torch.autograd.grad(outs, (*state["x"], *state["w"]), state["dout"])]
    outs = mla_assemble_qkv(*state["x"], state["cos"], state["sin"], state["pos"])
    return [*(o.detach() for o in outs), *torch.autograd.grad(outs, state["x"], state["dout"])]


def work(case):
    kind, b, s = case["kind"], case["b"], case["s"]
    if kind in ("attention", "ring"):
        hq, hkv, d, dv = case["hq"], case["hkv"], case["d"], VALUE_DIM[case["d"]]
        if kind == "attention":
            backward, chunks = case["backward"], 1
            entries = s * (s + 1) // 2 if case["causal"] else s * s
            key_values = hkv * (d + dv)  # features per position
        else:
            backward, chunks, entries = True, len(_visited(case)), 0
            for st in ring_schedule(case["rank"], case["cp"], s, case["layout"]):
                rows, keys = st.q_rows[1] - st.q_rows[0], st.kv_rows[1] - st.kv_rows[0]
                entries += rows * (rows + 1) // 2 if st.causal else rows * keys
            key_values = hkv * (d - ROPE_DIM + dv) + ROPE_DIM if case["split_key"] else hkv * (d + dv)
        inputs = b * s * (hq * d + chunks * key_values)
        outputs = b * s * hq * dv
        # forward: S and O; backward: S, dP, dV, dK and dQ, each once
        flops = 2 * (d + dv) * entries * hq * b
        if not backward:
            return {"bytes": 2 * (inputs + outputs), "flops": flops}
        flops += 2 * (3 * d + 2 * dv) * entries * hq * b
        return {"bytes": 2 * (2 * inputs + 2 * outputs), "flops": flops}  # gradients are as large as what they belong to
    if kind == "combine":
        n, rows = b * s * case["h"] * case["d"], b * s * case["h"]
        return {"bytes": n * (2 * (2 if case["partial"] == "bf16" else 4) + 4) + 12 * rows, "flops": 4 * n}
    if kind == "gqa_prologue":
        n = b * s * (case["hq"] + case["hkv"]) * case["d"]
        tables = 2 * s * case["d"] * 2
        weights = 2 * case["d"] * (2 if case["weight"] == "bf16" else 4)
        return {"bytes": 2 * 4 * n + tables + 2 * weights, "flops": 30 * n}
    h = case["h"]
    ins, outs = h * (192 + 256) + ROPE_DIM, h * (192 + 192 + 128)
    return {"bytes": b * s * (2 * (2 * ins + 2 * outs) + 8) + 2 * s * ROPE_DIM * 2, "flops": 12 * b * s * (h + 1) * ROPE_DIM}


def tolerance(case):
    if case["kind"] == "combine":
        return {"rel": 1e-5}  # fp32 results of fp32 arithmetic
    if case["kind"] in ("gqa_prologue", "mla_prologue"):
        return {"rel": 4e-3}  # fp32 arithmetic, bf16 results: one rounding (2^-9) on either side
    return {"rel": 1e-2}  # P and dS are rounded to bf16 between the products, and so are the results
