"""dS hand-over between the two backward kernels of one chunk pair (head dims 128/128 and 192/128): with a `ds`
buffer the dK/dV kernel stores the dS tiles it forms and the dQ kernel computes dQ = scale * dS K from
them instead of recomputing S and dP (pithtrain/operators/mla/triton.py:205-266 recomputes). Expected
values come from the fp64 oracle; the recomputing dQ kernel is compared as well (the same bf16 dS values
summed in another order), and dK/dV must not change by a bit when the tiles are also stored."""

import pytest
import torch

from helpers import check_bf16_result, norm_max_err
from oracle import ring_oracle as R
from pithtrain_amd.operators.mla.hip import (
    _mla_bwd_preprocess,
    _mla_fwd,
    attn_bwd_dkdv_into,
    attn_bwd_dq_into,
    attn_bwd_ds_bytes,
    ds_buffer,
)
from pithtrain_amd.operators.ring_attention.local import ring_attention_local

pytestmark = pytest.mark.gpu

SHAPES = [
    # B, Sq, Skv, Hq, Hkv
    (1, 256, 256, 4, 4),
    (1, 512, 512, 8, 2),
    (2, 384, 384, 4, 1),
    (1, 333, 333, 4, 2),      # ragged last query tile and key block
    (1, 1000, 1000, 2, 1),
    (1, 2048, 2048, 16, 2),   # head split of the dK/dV kernel
    (1, 65, 65, 2, 2),        # one row beyond a query tile: two tiles, one key block
    (1, 129, 129, 4, 1),      # one row beyond a key block
    (2, 777, 777, 8, 2),
]
NONCAUSAL_SHAPES = SHAPES + [(1, 512, 256, 8, 2), (1, 256, 768, 4, 4), (1, 200, 450, 4, 2), (1, 65, 129, 2, 2)]


def _inputs(B, Sq, Skv, Hq, Hkv, seed=42, dqk=128):
    g = torch.Generator().manual_seed(seed)
    scale = dqk**-0.5
    q = (torch.randn(B, Sq, Hq, dqk, generator=g) * scale).to(torch.bfloat16)
    k = (torch.randn(B, Skv, Hkv, dqk, generator=g) * scale).to(torch.bfloat16)
    v = (torch.randn(B, Skv, Hkv, 128, generator=g) * scale).to(torch.bfloat16)
    dout = torch.randn(B, Sq, Hq, 128, generator=g).to(torch.bfloat16)
    return q, k, v, dout, scale


def _run(gpu, causal, shape, dq_dtype, dqk=128):
    q, k, v, dout, scale = _inputs(*shape, dqk=dqk)
    qd, kd, vd, dod = (t.to(gpu) for t in (q, k, v, dout))
    o, lse = _mla_fwd(qd, kd, vd, scale, causal)
    delta = _mla_bwd_preprocess(o, dod)
    o_ref, lse_ref = R.chunk_fwd(q, k, v, scale, causal)
    dq_ref, dk_ref, dv_ref = R.chunk_bwd(q, k, v, dout, lse_ref, R.bwd_delta(o_ref, dout), scale, causal)

    dk0, dv0 = torch.empty_like(kd), torch.empty_like(vd)
    dq0 = torch.empty(qd.shape, dtype=dq_dtype, device=gpu)
    attn_bwd_dkdv_into(qd, kd, vd, dod, lse, delta, dk0, dv0, scale, causal)
    attn_bwd_dq_into(qd, kd, vd, dod, lse, delta, dq0, scale, causal)

    need = attn_bwd_ds_bytes(qd, kd, vd, causal)
    n_qt, n_kb = (shape[1] + 63) // 64, (shape[2] + 127) // 128
    # 16 KB per (64-row query tile, 128-key block); under the mask tile t keeps its first t // 2 + 1 key blocks
    blocks = sum(t // 2 + 1 for t in range(n_qt)) if causal else n_qt * n_kb
    assert need == shape[0] * shape[3] * blocks * 16384
    # poisoned buffer: whatever the dQ kernel reads must have been written by the dK/dV kernel
    ds = torch.full((need,), 0x7F, dtype=torch.uint8, device=gpu)
    dk1, dv1 = torch.empty_like(kd), torch.empty_like(vd)
    dq1 = torch.empty(qd.shape, dtype=dq_dtype, device=gpu)
    attn_bwd_dkdv_into(qd, kd, vd, dod, lse, delta, dk1, dv1, scale, causal, ds=ds)
    attn_bwd_dq_into(qd, kd, vd, dod, lse, delta, dq1, scale, causal, ds=ds)
    torch.cuda.synchronize()
    assert torch.equal(dk0, dk1) and torch.equal(dv0, dv1), "storing dS changed dK/dV"
    check_bf16_result(dq1, dq_ref, "dQ from dS", otol=1e-3)
    # two bf16 results of the same sums in different orders: up to one bf16 step (2^-8) of the largest element
    assert norm_max_err(dq1.float().cpu(), dq0.float().cpu()) < 6e-3, "dQ from dS vs recomputing kernel"
    return qd, kd, vd, dod, lse, delta, dq1, ds, scale


@pytest.mark.parametrize("shape", SHAPES)
def test_causal_dq_from_ds(gpu, shape):
    _run(gpu, True, shape, torch.bfloat16)


SHAPES_192 = [(1, 129, 129, 4, 1), (1, 256, 256, 4, 4), (1, 257, 257, 2, 1), (2, 333, 333, 4, 2), (2, 777, 777, 8, 2), (1, 1025, 1025, 2, 2),
              (1, 2048, 2048, 4, 4), (17, 255, 255, 16, 16)]  # fmt: skip


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("causal,shape", [(True, s) for s in SHAPES_192] + [(False, s) for s in [*SHAPES_192[:4], (1, 512, 256, 8, 2), (1, 200, 450, 4, 2), (1, 257, 129, 2, 2)]])
def test_dq_from_ds_192(gpu, causal, shape, dtype):
    """(192, 128): 256 rows per dQ workgroup, two waves to 64 of them with half of the features each (the last quarter from the tile of
    trailing features); pairs of 128-row blocks under the mask, consecutive rows where the grid exceeds a round."""
    _run(gpu, causal, shape, dtype, dqk=192)


@pytest.mark.parametrize("dqk", [128, 192])
@pytest.mark.parametrize("keys", [2, 32, 33, 65])  # (of a single key P is 1 and dS = dP - delta nothing but rounding)
def test_dq_from_ds_of_few_key_steps(gpu, keys, dqk):
    """Walks of one, two and three 32-key steps: shorter than the rings, and than what is read ahead of the products."""
    _run(gpu, False, (1, 321, keys, 4, 2), torch.bfloat16, dqk=dqk)


@pytest.mark.parametrize("layout", ["contiguous", "zigzag"])
def test_ring_share_of_192_with_and_without_handover(gpu, layout, monkeypatch):
    """Steps that hand dS over (fp32 dQ added to and finished by their kernels) against one launch that recomputes: the same bf16 dS
    values summed in other orders, up to one bf16 step (2^-8) of the largest element; and two heads against the oracle."""
    from pithtrain_amd.operators.mla import hip as H
    from pithtrain_amd.operators.ring_attention import local as L

    g = torch.Generator(device=gpu).manual_seed(5)
    t = lambda h, d: torch.randn(1, 2050, h, d, generator=g, device=gpu).to(torch.bfloat16)  # noqa: E731
    q, dout, ks, vs = t(16, 192), t(16, 128), [t(16, 192) for _ in range(3)], [t(16, 128) for _ in range(3)]
    visited = len(L.ring_schedule(1, 3, 2050, layout))
    ks, vs = (ks, vs) if layout == "zigzag" else ([*ks[:2], None], [*vs[:2], None])
    out, lse = L.ring_forward_local(q, ks, vs, 0.07, 1, 3, layout)
    monkeypatch.setattr(L, "_handover_pays", lambda *a: True)
    monkeypatch.setattr(H, "ds_plan", lambda q, k, v, causal=False: (16, attn_bwd_ds_bytes(q, k, v, causal)))
    used, pair = [], H.attn_bwd_pair_into
    monkeypatch.setattr(L, "attn_bwd_pair_into", lambda *a, **kw: used.append(pair(*a, **kw)) or used[-1])
    steps = L.ring_backward_local(dout, q, out, lse, ks, vs, 0.07, 1, 3, layout)
    assert len(used) == visited and all(used), "every step hands its dS over"
    monkeypatch.setattr(L, "_handover_pays", lambda *a: False)
    one = L.ring_backward_local(dout, q, out, lse, ks, vs, 0.07, 1, 3, layout)
    assert len(used) == visited and not torch.equal(steps[0], one[0])
    flat = lambda r: [r[0], *(x for l in r[1:3] for x in l if x is not None)]  # noqa: E731
    for a, b in zip(flat(steps), flat(one), strict=True):
        assert norm_max_err(a.float(), b.float()) < 6e-3
    two = lambda x: None if x is None else x[:, :, 6:8].cpu()  # noqa: E731
    host = two(q), [two(x) for x in ks], [two(x) for x in vs]
    o_ref, lse_ref = R.ring_forward(*host, 0.07, 1, 3, layout)
    want = R.ring_backward(two(dout), host[0], o_ref, lse_ref, *host[1:], 0.07, 1, 3, layout)
    for name, a, b in zip(["dQ", *[f"{n}{j}" for n in ("dK", "dV") for j in range(visited)]], flat(steps), flat(want), strict=True):
        check_bf16_result(a[:, :, 6:8], b, f"ring {name}", otol=1e-3)


@pytest.mark.parametrize("b,s,h,cp,rank,layout,two_parts", [
    (1, 256, 2, 2, 0, "zigzag", False), (2, 640, 2, 3, 1, "zigzag", True), (1, 333, 2, 3, 2, "contiguous", False), (1, 1021, 4, 4, 2, "contiguous", True),
    (3, 1100, 48, 2, 1, "contiguous", False), (5, 1024, 16, 4, 2, "zigzag", False), (1, 1152, 3, 4, 1, "zigzag", True),
])  # fmt: skip
def test_share_of_192_in_two_launches(gpu, b, s, h, cp, rank, layout, two_parts):
    """All chunks' images in one buffer (poisoned), one dK/dV and one dQ launch: dK and dV bit for bit as without, dQ of the same bf16 dS
    values summed in another order (one bf16 step, 2^-8, of the largest element). Half and whole chunks, an empty middle block of
    rows, both orders of workgroups, ragged rows and keys."""
    from pithtrain_amd._ext import native
    from pithtrain_amd.operators.ring_attention import local as L

    g = torch.Generator(device=gpu).manual_seed(s)
    t = lambda *n: torch.randn(*n, generator=g, device=gpu).to(torch.bfloat16)  # noqa: E731
    of = lambda *n: [t(b, s, *n) if layout == "zigzag" or j <= rank else None for j in range(cp)]  # noqa: E731
    q, dout, ks, vs, pes = t(b, s, h, 192), t(b, s, h, 128), of(h, 128 if two_parts else 192), of(h, 128), of(64) if two_parts else None
    out, lse = L.ring_forward_local(q, ks, vs, 0.07, rank, cp, layout, pes)
    blocks = 0
    for st in L.ring_schedule(rank, cp, s, layout):
        qt, kb = -((st.q_rows[0] - st.q_rows[1]) // 64), -((st.kv_rows[0] - st.kv_rows[1]) // 128)
        blocks += sum(i // 2 + 1 for i in range(qt)) if st.causal else qt * kb
    ds = torch.full((b * h * blocks * 16384,), 0x7F, dtype=torch.uint8, device=gpu)
    args = (dout, q, out, lse, ks, vs, pes, 0.07, rank, cp, layout == "zigzag")
    want, got, small = native.ring_backward(*args), native.ring_backward(*args, ds), native.ring_backward(*args, ds[:-256])
    for a, x, y in zip((l for r in want[1:] for l in r), (l for r in got[1:] for l in r), (l for r in small[1:] for l in r), strict=True):
        assert a is None and x is None or torch.equal(a, x) and torch.equal(a, y)
    assert torch.equal(small[0], want[0]), "a buffer that is too small must not be used"
    assert not torch.equal(got[0], want[0]) and norm_max_err(got[0].float(), want[0].float()) < 6e-3


def test_share_of_192_hands_over_within_the_limits(gpu, monkeypatch):
    """Also in a captured graph, every replay; above the memory limit and where the allocation fails the share recomputes."""
    from pithtrain_amd._ext import native
    from pithtrain_amd.operators.mla import hip as H

    units = torch.cuda.get_device_properties(gpu).multi_processor_count
    t = lambda d, grad: torch.randn(1, 3072, 16, d, device=gpu).to(torch.bfloat16).requires_grad_(grad)  # noqa: E731
    q, ks, vs, dout = t(192, True), [t(192, True) for _ in range(2)], [t(128, True) for _ in range(2)], t(128, False)
    need = native.share_ds_bytes(q, ks, vs, None, 1, 2, True)
    assert (need > 0) == native.share_of_192_pays(1, 3072, 16, units)
    buffers, real = [], H._try_alloc
    monkeypatch.setattr(H, "_try_alloc", lambda *a: buffers.append(a[0]) or real(*a))

    def step():
        return torch.autograd.grad(ring_attention_local(q, ks, vs, 0.07, 1, 2, "zigzag"), [q, *ks, *vs], dout)

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        want = step()
    torch.cuda.current_stream().wait_stream(side)
    assert buffers == ([need] if need else [])
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = step()
    for replay in range(3):
        for x in captured:
            x.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(captured, want)), f"replay {replay}"
        assert all(torch.equal(a, b) for a, b in zip(step(), want))
    monkeypatch.setattr(H, "_try_alloc", lambda *a: None)
    failed = step()
    monkeypatch.setattr(H, "DS_BUFFER_LIMIT_BYTES", 0)
    limited = step()
    assert all(torch.equal(a, b) for a, b in zip(failed, limited)) and norm_max_err(limited[0].float(), want[0].float()) < 6e-3


@pytest.mark.parametrize("S", [255, 257, 511, 513, 767, 769, 1025, 1281, 1537])
def test_causal_pairs_of_row_blocks(gpu, S):
    """Under the mask a workgroup takes 256-row blocks in pairs, one from either end: odd and even numbers of blocks, the last
    one full, of one row or one row short."""
    _run(gpu, True, (1, S, S, 2, 1), torch.bfloat16)


@pytest.mark.parametrize("B,S", [(17, 255), (9, 513), (9, 1024), (6, 1025), (5, 1537), (4, 2049), (4, 2303)])
def test_consecutive_rows_equal_pairs(gpu, B, S):
    """More than one round of workgroups takes consecutive rows, a batch element alone pairs of blocks: the same sums."""
    from pithtrain_amd import _C

    g = torch.Generator(device=gpu).manual_seed(S)
    t = lambda h: torch.randn(B, S, h, 128, generator=g, device=gpu).to(torch.bfloat16)  # noqa: E731
    q, k, v, dout = t(16), t(2), t(2), t(16)
    o, lse = _mla_fwd(q, k, v, 0.09, True)
    delta = _mla_bwd_preprocess(o, dout)

    def dq_of(*x):
        args, plan = _C.AttnBwdArgs(B=x[0].shape[0], Sq=S, Skv=S, Hq=16, Hkv=2, Dqk=128, Dv=128, causal=1), _C.AttnBwdPlan()
        _C.check(_C.lib().pith_attn_bwd_plan(_C.byref(args), _C.byref(plan)))
        ds = torch.full((attn_bwd_ds_bytes(*x[:3], True),), 0x7F, dtype=torch.uint8, device=gpu)
        dk, dv, dq = torch.empty_like(x[1]), torch.empty_like(x[2]), torch.full_like(x[0], float("nan"))
        attn_bwd_dkdv_into(*x, dk, dv, 0.09, True, ds=ds)
        attn_bwd_dq_into(*x, dq, 0.09, True, ds=ds)
        return dq, plan.dq_ds_pairs

    whole, pairs = dq_of(q, k, v, dout, lse, delta)
    if torch.cuda.get_device_properties(gpu).multi_processor_count == 256:
        assert not pairs
    for b in range(B):
        one, pairs = dq_of(*[x[b : b + 1] for x in (q, k, v, dout, lse, delta)])
        assert pairs and torch.equal(whole[b : b + 1], one), f"batch element {b}"


@pytest.mark.parametrize("heads", [1, 3])
@pytest.mark.parametrize("S", [129, 255, 513, 1024, 1100])
def test_consecutive_rows_equal_pairs_192(gpu, S, heads):
    """The same of 192 features, at either side of one round of this device's units (256-row workgroups, pairs of 128-row blocks)."""
    from pithtrain_amd import _C

    units = torch.cuda.get_device_properties(gpu).multi_processor_count
    B = units // (heads * -(-S // 256)) + 1
    g = torch.Generator(device=gpu).manual_seed(S)
    t = lambda d: torch.randn(B, S, heads, d, generator=g, device=gpu).to(torch.bfloat16)  # noqa: E731
    q, k, v, dout = t(192), t(192), t(128), t(128)
    o, lse = _mla_fwd(q, k, v, 0.07, True)
    delta = _mla_bwd_preprocess(o, dout)

    def dq_of(*x):
        args, plan = _C.AttnBwdArgs(B=x[0].shape[0], Sq=S, Skv=S, Hq=heads, Hkv=heads, Dqk=192, Dv=128, causal=1), _C.AttnBwdPlan()
        _C.check(_C.lib().pith_attn_bwd_plan(_C.byref(args), _C.byref(plan)))
        ds = torch.full((attn_bwd_ds_bytes(*x[:3], True),), 0x7F, dtype=torch.uint8, device=gpu)
        dk, dv, dq = torch.empty_like(x[1]), torch.empty_like(x[2]), torch.full_like(x[0], float("nan"))
        attn_bwd_dkdv_into(*x, dk, dv, 0.07, True, ds=ds)
        attn_bwd_dq_into(*x, dq, 0.07, True, ds=ds)
        return dq, plan.dq_ds_pairs

    whole, pairs = dq_of(q, k, v, dout, lse, delta)
    assert not pairs
    most, pairs = dq_of(*[x[1:] for x in (q, k, v, dout, lse, delta)])
    one, pairs_one = dq_of(*[x[:1] for x in (q, k, v, dout, lse, delta)])
    assert pairs and pairs_one and torch.equal(whole[1:], most) and torch.equal(whole[:1], one)


@pytest.mark.parametrize("shape", NONCAUSAL_SHAPES)
def test_noncausal_dq_from_ds(gpu, shape):
    _run(gpu, False, shape, torch.bfloat16)


@pytest.mark.parametrize("causal", [True, False])
def test_fp32_output_and_accumulation(gpu, causal):
    qd, kd, vd, dod, lse, delta, dq1, ds, scale = _run(gpu, causal, (1, 512, 512, 8, 2), torch.float32)
    acc = torch.full_like(dq1, 0.25)
    attn_bwd_dq_into(qd, kd, vd, dod, lse, delta, acc, scale, causal, accumulate=True, ds=ds)
    assert torch.equal(acc, dq1 + 0.25)


def test_small_buffer_falls_back_to_recomputation(gpu):
    q, k, v, dout, scale = _inputs(1, 256, 256, 4, 4)
    qd, kd, vd, dod = (t.to(gpu) for t in (q, k, v, dout))
    o, lse = _mla_fwd(qd, kd, vd, scale, True)
    delta = _mla_bwd_preprocess(o, dod)
    dq0, dq1 = torch.empty_like(qd), torch.empty_like(qd)
    attn_bwd_dq_into(qd, kd, vd, dod, lse, delta, dq0, scale, True)
    small = torch.zeros(attn_bwd_ds_bytes(qd, kd, vd, True) - 1024, dtype=torch.uint8, device=gpu)
    attn_bwd_dq_into(qd, kd, vd, dod, lse, delta, dq1, scale, True, ds=small)
    assert torch.equal(dq0, dq1)
    # head dims without a hand-over path, and rows that leave half of the 192-feature workgroups empty, report 0 bytes and get no buffer
    for d in (64, 192):
        qx = torch.empty(1, 128, 4, d, dtype=torch.bfloat16, device=gpu)
        vx = torch.empty(1, 128, 4, min(d, 128), dtype=torch.bfloat16, device=gpu)
        assert attn_bwd_ds_bytes(qx, qx, vx) == 0 and ds_buffer(qx, qx, vx) is None


@pytest.mark.parametrize("layout", ["contiguous", "zigzag"])
def test_ring_share_uses_the_handover(gpu, layout, monkeypatch):
    """The ring backward with the hand-over equals the ring backward without it (dK/dV bit for bit, dQ up to
    summation order) and the oracle's ring share."""
    from pithtrain_amd.operators.ring_attention import local as L

    B, S, Hq, Hkv, C, rank = 1, 2048, 8, 2, 4, 1
    q_full, k_full, v_full, dout_full, scale = _inputs(B, S, S, Hq, Hkv, seed=7)
    split = (lambda x: R.zigzag_split(x, C)) if layout == "zigzag" else (lambda x: list(x.chunk(C, 1)))
    qs, ks, vs, dos = (split(t) for t in (q_full, k_full, v_full, dout_full))

    def run():
        q = qs[rank].to(gpu).requires_grad_(True)
        kc = [t.to(gpu).requires_grad_(True) for t in ks]
        vc = [t.to(gpu).requires_grad_(True) for t in vs]
        out = ring_attention_local(q, kc, vc, scale, rank, C, layout)
        out.backward(dos[rank].to(gpu))
        return q.grad, [t.grad for t in kc], [t.grad for t in vc]

    from pithtrain_amd.operators.mla import hip as H

    used = []
    real_plan = H.ds_plan

    def always(q, k, v, causal=False):  # the default policy would decline a share this small
        used.append(1)
        return k.shape[2], attn_bwd_ds_bytes(q, k, v, causal)

    monkeypatch.setattr(H, "ds_plan", always)
    dq1, dk1, dv1 = run()
    assert used, "the ring backward did not ask for a hand-over plan"
    monkeypatch.setattr(H, "ds_plan", lambda *a: None)
    dq0, dk0, dv0 = run()
    monkeypatch.setattr(H, "ds_plan", real_plan)
    for a, b in zip(dk0 + dv0, dk1 + dv1):
        assert (a is None and b is None) or torch.equal(a, b)
    assert norm_max_err(dq1.float().cpu(), dq0.float().cpu()) < 6e-3
    o_ref, lse_ref = R.ring_forward(qs[rank], ks, vs, scale, rank, C, layout)
    dq_ref, _, _ = R.ring_backward(dos[rank], qs[rank], o_ref, lse_ref, ks, vs, scale, rank, C, layout)
    check_bf16_result(dq1, dq_ref, "ring dQ", otol=1e-3)


@pytest.mark.parametrize("layout", ["contiguous", "zigzag"])
def test_small_ring_share_step_by_step_uses_the_handover(gpu, layout, monkeypatch):
    """The same with the rule that would send a share this small out as one launch switched off."""
    from pithtrain_amd.operators.mla import hip as H
    from pithtrain_amd.operators.ring_attention import local as L

    buffers, real = [], H._try_alloc
    monkeypatch.setattr(L, "_steps_beat_one_launch", lambda *a: True)
    monkeypatch.setattr(H, "_try_alloc", lambda *a: buffers.append(real(*a)) or buffers[-1])
    test_ring_share_uses_the_handover(gpu, layout, monkeypatch)
    assert buffers, "no step handed dS over"


def _shaped(gpu, b, s, hq, hkv):
    q = torch.empty(b, s, hq, 128, dtype=torch.bfloat16, device=gpu)
    k = torch.empty(b, s, hkv, 128, dtype=torch.bfloat16, device=gpu)
    return q, k, k


def test_default_policy_of_the_buffer(gpu, monkeypatch):
    """ds_plan takes the hand-over only when the dS-reading dQ kernel would fill the device, keeps the buffer
    under the configured limit and under a fraction of the free memory by going through the kv heads in slabs,
    and gives up (both kernels recompute) when not even one kv head fits."""
    from pithtrain_amd.operators.mla import hip as H

    assert H.DS_BUFFER_LIMIT_BYTES <= 4 << 30, "the default limit must stay modest"
    assert H.ds_plan(*_shaped(gpu, 1, 512, 8, 2)) is None  # 1 x 8 workgroups: too few
    big = _shaped(gpu, 1, 4096, 32, 4)  # 8 x 32 workgroups, 1 GiB
    assert attn_bwd_ds_bytes(*big) == 1 << 30
    assert H.ds_plan(*big) == (4, 1 << 30)
    buf = ds_buffer(*big)
    assert buf is not None and buf.numel() == 1 << 30 and buf.data_ptr() % 256 == 0
    del buf
    monkeypatch.setattr(H, "DS_BUFFER_LIMIT_BYTES", (1 << 30) - 1)
    assert H.ds_plan(*big) is None and ds_buffer(*big) is None  # slabs of 2 kv heads: 8 x 16 workgroups, too few
    # 16384 x 16384 rows, 32 / 4 heads: 4 GiB per kv head, 32 x 8 workgroups of the dQ kernel per kv head
    q = torch.empty(1, dtype=torch.bfloat16, device=gpu).as_strided((1, 16384, 32, 128), (0, 0, 0, 0))
    k = torch.empty(1, dtype=torch.bfloat16, device=gpu).as_strided((1, 16384, 4, 128), (0, 0, 0, 0))
    monkeypatch.setattr(H, "DS_BUFFER_LIMIT_BYTES", 16 << 30)
    assert H.ds_plan(q, k, k) == (4, 16 << 30)
    monkeypatch.setattr(H, "DS_BUFFER_LIMIT_BYTES", (16 << 30) - 1)
    assert H.ds_plan(q, k, k) == (2, 8 << 30) and ds_buffer(q, k, k) is None  # two slabs of two kv heads
    monkeypatch.setattr(H, "DS_BUFFER_LIMIT_BYTES", (4 << 30) + 5)
    assert H.ds_plan(q, k, k) == (1, 4 << 30)
    monkeypatch.setattr(H, "DS_BUFFER_LIMIT_BYTES", (4 << 30) - 1)
    assert H.ds_plan(q, k, k) is None
    # the 131072-token configuration (64 / 4 heads, 16384 x 8192 rows per ring step): one kv head at a time
    monkeypatch.setattr(H, "DS_BUFFER_LIMIT_BYTES", 4 << 30)
    q64 = torch.empty(1, dtype=torch.bfloat16, device=gpu).as_strided((1, 16384, 64, 128), (0, 0, 0, 0))
    k8k = torch.empty(1, dtype=torch.bfloat16, device=gpu).as_strided((1, 8192, 4, 128), (0, 0, 0, 0))
    assert H.ds_plan(q64, k8k, k8k) == (1, 4 << 30)
    # little free memory: the budget follows it
    monkeypatch.setattr(H, "DS_BUFFER_LIMIT_BYTES", 16 << 30)
    monkeypatch.setattr(H.torch.cuda, "mem_get_info", lambda dev=None: (8 << 30, 1 << 38))
    monkeypatch.setattr(H.torch.cuda, "memory_reserved", lambda dev=None: 0)
    monkeypatch.setattr(H.torch.cuda, "memory_allocated", lambda dev=None: 0)
    assert H.ds_plan(q, k, k) == (1, 4 << 30)


@pytest.mark.parametrize("dqk", [128, 192])
@pytest.mark.parametrize("causal", [False, True])
def test_slabs_of_kv_heads_equal_the_whole_call(gpu, causal, dqk, monkeypatch):
    """attn_bwd_pair_into through a buffer that holds one or two kv heads at a time (head ranges of the full
    tensors, passed in place) gives dK/dV bit for bit and dQ bit for bit what the whole-pair hand-over gives."""
    from pithtrain_amd.operators.mla import hip as H

    B, Sq, Hq, Hkv = 2, 1024, 16, 4
    Skv = Sq if causal else 640
    q, k, v, dout, scale = _inputs(B, Sq, Skv, Hq, Hkv, seed=11, dqk=dqk)
    qd, kd, vd, dod = (t.to(gpu) for t in (q, k, v, dout))
    o, lse = _mla_fwd(qd, kd, vd, scale, causal)
    delta = _mla_bwd_preprocess(o, dod)
    need = attn_bwd_ds_bytes(qd, kd, vd, causal)
    results = []
    for heads in (4, 2, 1):
        monkeypatch.setattr(H, "ds_plan", lambda *a, heads=heads: (heads, need // Hkv * heads))
        dq = torch.full(qd.shape, 0.25, dtype=torch.float32, device=gpu)
        dk, dv = torch.empty_like(kd), torch.empty_like(vd)
        used = H.attn_bwd_pair_into(qd, kd, vd, dod, lse, delta, dq, dk, dv, scale, causal, accumulate_dq=True)
        assert used == need // Hkv * heads
        results.append((dq, dk, dv))
        # rows that are finished by the call go out as bf16, the others stay in fp32
        part, final = torch.full_like(dq, 0.25), torch.full_like(qd, 7.0)
        H.attn_bwd_pair_into(qd, kd, vd, dod, lse, delta, part, dk, dv, scale, causal, accumulate_dq=True, dq_final=final, dq_final_rows=(320, 992))
        assert torch.equal(final[:, 320:992], dq[:, 320:992].to(torch.bfloat16)) and (part[:, 320:992] == 0.25).all()
        for rows in (slice(0, 320), slice(992, Sq)):
            assert torch.equal(part[:, rows], dq[:, rows]) and (final[:, rows] == 7).all()
    for dq, dk, dv in results[1:]:
        assert torch.equal(dq, results[0][0]) and torch.equal(dk, results[0][1]) and torch.equal(dv, results[0][2])
    rdq, rdk, rdv = R.chunk_bwd(q, k, v, dout, lse.double().cpu(), delta.double().cpu(), scale, causal)
    check_bf16_result(results[2][0] - 0.25, rdq, "slab dQ", otol=1e-3)
    check_bf16_result(results[2][1], rdk, "slab dK", otol=1e-3)
    check_bf16_result(results[2][2], rdv, "slab dV", otol=1e-3)


def test_head_range_calls_without_handover(gpu):
    """The recomputing kernels accept a head range of wider tensors too (all three head-dim families)."""
    for d_q, d_v in ((128, 128), (192, 128), (64, 64)):
        B, S, Hq, Hkv = 1, 320, 8, 4
        g = torch.Generator().manual_seed(5)
        q = (torch.randn(B, S, Hq, d_q, generator=g) * d_q**-0.5).to(torch.bfloat16).to(gpu)
        k = (torch.randn(B, S, Hkv, d_q, generator=g) * d_q**-0.5).to(torch.bfloat16).to(gpu)
        v = torch.randn(B, S, Hkv, d_v, generator=g).to(torch.bfloat16).to(gpu)
        dout = torch.randn(B, S, Hq, d_v, generator=g).to(torch.bfloat16).to(gpu)
        scale = d_q**-0.5
        o, lse = _mla_fwd(q, k, v, scale, True)
        delta = _mla_bwd_preprocess(o, dout)
        dq0, dk0, dv0 = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
        from pithtrain_amd.operators.mla import hip as H_

        H_.attn_bwd_pair_into(q, k, v, dout, lse, delta, dq0, dk0, dv0, scale, True, handover=False)
        dq1, dk1, dv1 = torch.zeros_like(q), torch.zeros_like(k), torch.zeros_like(v)
        for h0 in range(0, Hkv, 2):
            kv_h, q_h = slice(h0, h0 + 2), slice(2 * h0, 2 * h0 + 4)
            H_.attn_bwd_pair_into(q[:, :, q_h], k[:, :, kv_h], v[:, :, kv_h], dout[:, :, q_h], lse[:, q_h], delta[:, q_h],
                                  dq1[:, :, q_h], dk1[:, :, kv_h], dv1[:, :, kv_h], scale, True, handover=False)  # fmt: skip
        assert torch.equal(dq0, dq1) and torch.equal(dk0, dk1) and torch.equal(dv0, dv1), (d_q, d_v)


def test_allocation_failure_falls_back_to_recomputation(gpu, monkeypatch):
    """When the hand-over buffer cannot be allocated the pair recomputes: dK/dV bit-identical to the hand-over
    path (the dK/dV kernel's arithmetic does not depend on the stores), dQ within oracle parity."""
    from pithtrain_amd.operators.mla import hip as H

    B, Sq, Skv, Hq, Hkv = 1, 1024, 768, 8, 2
    q, k, v, dout, scale = _inputs(B, Sq, Skv, Hq, Hkv, seed=3)
    qd, kd, vd, dod = (t.to(gpu) for t in (q, k, v, dout))
    o, lse = _mla_fwd(qd, kd, vd, scale, False)
    delta = _mla_bwd_preprocess(o, dod)
    monkeypatch.setattr(H, "ds_plan", lambda *a: (Hkv, attn_bwd_ds_bytes(qd, kd, vd, False)))
    need = attn_bwd_ds_bytes(qd, kd, vd, False)
    real_empty = torch.empty

    def failing_empty(*a, **kw):  # only the hand-over buffer's allocation fails
        if a and a[0] == need and kw.get("dtype") == torch.uint8:
            raise torch.cuda.OutOfMemoryError("forced by the test")
        return real_empty(*a, **kw)

    out = {}
    for name in ("handover", "oom"):
        with monkeypatch.context() as m:
            if name == "oom":
                m.setattr(torch, "empty", failing_empty)
            dq, dk, dv = torch.empty_like(qd), torch.empty_like(kd), torch.empty_like(vd)
            used = H.attn_bwd_pair_into(qd, kd, vd, dod, lse, delta, dq, dk, dv, scale, False)
        out[name] = (dq, dk, dv, used)
    assert out["handover"][3] > 0 and out["oom"][3] == 0
    assert torch.equal(out["handover"][1], out["oom"][1]) and torch.equal(out["handover"][2], out["oom"][2])
    rdq, _, _ = R.chunk_bwd(q, k, v, dout, lse.double().cpu(), delta.double().cpu(), scale, False)
    check_bf16_result(out["oom"][0], rdq, "recomputed dQ after allocation failure", otol=1e-3)
    check_bf16_result(out["handover"][0], rdq, "hand-over dQ", otol=1e-3)


def test_layer_of_one_round_under_capture(gpu):
    """A causal layer whose dS-reading dQ kernel just fills the device hands dS over, eagerly and in a captured graph."""
    import pithtrain_amd.operators.mla.hip as H

    g = torch.Generator(device=gpu).manual_seed(3)
    mk = lambda h: torch.randn(4, 1024, h, 128, generator=g, device=gpu).to(torch.bfloat16)  # noqa: E731
    q, k, v, dout, scale = mk(32), mk(4), mk(4), mk(32), 128**-0.5
    if H._device_compute_units(q.device) == 256:
        assert H.ds_plan(q, k, v, True) is not None  # 2 x 32 x 4 workgroups of 512 rows
    fwd, bwd = torch.ops.pithtrain_amd.attn_fwd, torch.ops.pithtrain_amd.attn_bwd

    def step():
        o, lse = fwd(q, k, v, scale, True)
        return [o, lse, *bwd(q, k, v, o, lse, dout, scale, True)]

    want = [t.clone() for t in step()]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = step()
    for replay in range(3):
        for t in captured:
            t.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(captured, want)), f"replay {replay}"
        assert all(torch.equal(a, b) for a, b in zip(step(), want))


@pytest.mark.parametrize("head_dim", [128, 192])
def test_chunk_call_leaves_the_ds_of_its_arguments_alone(gpu, head_dim):
    """pith_attn_bwd_chunks ignores args.ds, which may hold a chunk pair's tiles: nothing is written there, no result depends on it and
    an odd address is none of its business. The buffer of the hand-over is an argument of its own call."""
    from pithtrain_amd import _C

    S, H, scale = 256, 2, 0.07
    g = torch.Generator(device=gpu).manual_seed(3)
    t = lambda d: torch.randn(1, S, H, d, generator=g, device=gpu).to(torch.bfloat16)  # noqa: E731
    q, dout, out, ks, vs = t(head_dim), t(128), t(128), [t(head_dim) for _ in range(2)], [t(128) for _ in range(2)]
    lse, delta = torch.full((1, H, S), 12.0, device=gpu), _mla_bwd_preprocess(out, dout)
    grads = [torch.empty_like(q), *(torch.empty_like(x) for x in (*ks, *vs))]
    chunks = (_C.KeyChunk * 2)(*[_C.KeyChunk(k=ks[i].data_ptr(), v=vs[i].data_ptr(), rows=S, dk=grads[1 + i].data_ptr(), dv=grads[3 + i].data_ptr())
                                 for i in range(2)])  # fmt: skip

    def run(ds=None, offset=0, call="pith_attn_bwd_chunks", *more):
        for x in grads:
            x.fill_(float("nan"))
        a = _C.AttnBwdArgs(q=q.data_ptr(), dout=dout.data_ptr(), lse=lse.data_ptr(), delta=delta.data_ptr(), dq=grads[0].data_ptr(), B=1, Sq=S, Hq=H, Hkv=H,
                           Dqk=head_dim, Dv=128, q_bs=q.stride(0), k_bs=q.stride(0), v_bs=dout.stride(0), dout_bs=dout.stride(0), dq_bs=q.stride(0),
                           dk_bs=q.stride(0), dv_bs=dout.stride(0), lse_bs=H * S, lse_hs=S, scale=scale)  # fmt: skip
        if ds is not None and not more:
            a.ds, a.ds_bytes = ds.data_ptr() + offset, ds.numel() - offset
        _C.check(getattr(_C.lib(), call)(_C.byref(a), chunks, 2, *more, torch.cuda.current_stream().cuda_stream))
        return [x.clone() for x in grads]

    want = run()
    ds = torch.full((1 << 20,), 0x7F, dtype=torch.uint8, device=gpu)
    for offset in (0, 8):
        assert all(torch.equal(a, b) for a, b in zip(run(ds, offset), want))
        assert (ds == 0x7F).all(), "written through args.ds"
    handed = run(ds, 0, "pith_attn_bwd_chunks_handover", ds.data_ptr(), ds.numel())
    assert (ds == 0x7F).all() == (head_dim == 128) and torch.equal(handed[0], want[0]) == (head_dim == 128)
    assert all(torch.equal(a, b) for a, b in zip(handed[1:], want[1:])) and norm_max_err(handed[0].float(), want[0].float()) < 6e-3
    assert all(torch.equal(a, b) for a, b in zip(run(ds, 0, "pith_attn_bwd_chunks_handover", None, 0), want))


@pytest.mark.parametrize("head_dim", [128, 192])
def test_misaligned_buffer(gpu, head_dim):
    """A buffer off 256 bytes: refused at 128 features, where it always was; at 192, where the field used to be ignored, both calls
    recompute and leave it alone."""
    from pithtrain_amd import _C

    S, H, scale = 256, 2, 0.07
    g = torch.Generator(device=gpu).manual_seed(4)
    t = lambda d: torch.randn(1, S, H, d, generator=g, device=gpu).to(torch.bfloat16)  # noqa: E731
    q, k, v, dout = t(head_dim), t(head_dim), t(128), t(128)
    o, lse = _mla_fwd(q, k, v, scale, True)
    delta = _mla_bwd_preprocess(o, dout)
    dq, dk, dv = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
    a = _C.AttnBwdArgs(q=q.data_ptr(), k=k.data_ptr(), v=v.data_ptr(), dout=dout.data_ptr(), lse=lse.data_ptr(), delta=delta.data_ptr(), dq=dq.data_ptr(),
                       dk=dk.data_ptr(), dv=dv.data_ptr(), B=1, Sq=S, Skv=S, Hq=H, Hkv=H, Dqk=head_dim, Dv=128, q_bs=q.stride(0), k_bs=k.stride(0),
                       v_bs=v.stride(0), dout_bs=v.stride(0), dq_bs=q.stride(0), dk_bs=k.stride(0), dv_bs=v.stride(0), lse_bs=H * S, lse_hs=S,
                       scale=scale, causal=1)  # fmt: skip
    stream = torch.cuda.current_stream().cuda_stream

    def run(*calls):
        for x in (dq, dk, dv):
            x.fill_(float("nan"))
        codes = [getattr(_C.lib(), c)(_C.byref(a), stream) for c in calls]
        return codes, [x.clone() for x in (dq, dk, dv)]

    forms = [("pith_attn_bwd_dkdv", "pith_attn_bwd_dq"), ("pith_attn_bwd",)]
    want = [run(*calls)[1] for calls in forms]
    ds = torch.full((1 << 20,), 0x7F, dtype=torch.uint8, device=gpu)
    a.ds, a.ds_bytes = ds.data_ptr() + 16, ds.numel() - 16
    for calls, results in zip(forms, want):
        codes, got = run(*calls)
        if head_dim == 128:
            assert codes == [_C.PITH_ERR_MISALIGNED] * len(calls)
        else:
            assert codes == [_C.PITH_OK] * len(calls) and all(torch.equal(x, y) for x, y in zip(got, results))
    assert (ds == 0x7F).all()


@pytest.mark.parametrize("S", [1024, 1000])
@pytest.mark.parametrize("head_dim", [128, 192])
def test_infinity_reaches_the_rows_that_it_reaches_without_handover(gpu, head_dim, S):
    """An infinity in K or V of one key (LSE and delta are those of finite ones): rows before the key's 64-row tile do not see it, and dQ
    from dS is not finite exactly where the recomputing kernel's is not. dK and dV bit for bit."""
    q, k, v, dout, scale = (t.to(gpu) if torch.is_tensor(t) else t for t in _inputs(1, S, S, 2, 2, dqk=head_dim))
    o, lse = _mla_fwd(q, k, v, scale, True)
    delta = _mla_bwd_preprocess(o, dout)
    for which in (1, 2):
        for key in (0, 33, 64, 95, 127, 128, 300, 999):
            x = [q, k.clone(), v.clone(), dout, lse, delta]
            x[which][:, key, :, 5] = float("inf")
            runs = []
            for ds in (None, torch.full((attn_bwd_ds_bytes(*x[:3], True),), 0x7F, dtype=torch.uint8, device=gpu)):
                dk, dv, dq = torch.empty_like(k), torch.empty_like(v), torch.empty_like(q)
                attn_bwd_dkdv_into(*x, dk, dv, scale, True, ds=ds)
                attn_bwd_dq_into(*x, dq, scale, True, ds=ds)
                runs.append((dq, dk, dv))
            finite = [r[0].isfinite().all(-1) for r in runs]
            assert torch.equal(*finite) and finite[0][:, : key // 64 * 64].all() and not finite[0][:, key:].all(), (which, key)
            assert all(torch.equal(a.view(torch.int16), b.view(torch.int16)) for a, b in zip(runs[0][1:], runs[1][1:])), (which, key)


@pytest.mark.parametrize("magnitude", [1e4, 1e18])
def test_large_values_at_masked_keys(gpu, magnitude):
    """Rows of one 64-row tile see none of the next tile's keys, however large their scores and values are."""
    S = 512
    q, k, v, dout, scale = (t.to(gpu) if torch.is_tensor(t) else t for t in _inputs(1, S, S, 2, 2, dqk=192))
    dqs = []
    for factor in (1.0, magnitude):
        kx, vx = k.clone(), v.clone()
        kx[:, 320:] *= factor
        vx[:, 320:] *= factor
        o, lse = _mla_fwd(q, kx, vx, scale, True)
        delta = _mla_bwd_preprocess(o, dout)
        ds = torch.full((attn_bwd_ds_bytes(q, kx, vx, True),), 0x7F, dtype=torch.uint8, device=gpu)
        dk, dv, dq = torch.empty_like(k), torch.empty_like(v), torch.empty_like(q)
        attn_bwd_dkdv_into(q, kx, vx, dout, lse, delta, dk, dv, scale, True, ds=ds)
        attn_bwd_dq_into(q, kx, vx, dout, lse, delta, dq, scale, True, ds=ds)
        dqs.append(dq)
    assert torch.equal(dqs[0][:, :320], dqs[1][:, :320])
