"""A ring share as one launch over all of its chunks: every work split of the kernels, at row counts where a tile or a wave
straddles the first row that sees a chunk, the end of a chunk or the diagonal, against the float64 oracle."""

import ctypes

import pytest
import torch

from helpers import check_bf16_result, check_lse
from oracle import ring_oracle as R
from pithtrain_amd import _C
from pithtrain_amd.operators.mla import hip as H
from pithtrain_amd.operators.ring_attention import local as L

pytestmark = pytest.mark.gpu


CASES = [  # B, S_l, Hq, Hkv, D, C, rank, layout, keys in two parts
    (2, 2, 2, 1, 64, 2, 0, "zigzag", False), (1, 66, 4, 2, 64, 3, 1, "zigzag", False), (1, 257, 4, 4, 64, 2, 1, "contiguous", False),
    (1, 1, 2, 1, 128, 2, 1, "contiguous", False), (2, 130, 4, 2, 128, 3, 0, "zigzag", False), (1, 258, 4, 2, 128, 3, 2, "zigzag", False),
    (1, 1100, 32, 4, 128, 2, 1, "zigzag", False), (1, 1026, 30, 2, 128, 2, 0, "zigzag", False), (1, 96, 2, 2, 128, 16, 15, "contiguous", False),
    (1, 34, 2, 2, 192, 4, 1, "zigzag", True), (2, 129, 2, 2, 192, 3, 2, "contiguous", True), (1, 322, 4, 4, 192, 2, 0, "zigzag", False),
    (1, 1022, 36, 36, 192, 2, 1, "contiguous", True),
]  # fmt: skip


def _not_used(*args, **kwargs):
    raise AssertionError("the other path took the call")


# (step by step: what a ring does whose chunks arrive one after the other)
@pytest.mark.parametrize("one_launch,B,S,Hq,Hkv,D,C,rank,layout,two_part", [(True, *c) for c in CASES] + [(False, *c) for c in CASES[3:6] + CASES[9:12]])
def test_share(gpu, monkeypatch, one_launch, B, S, Hq, Hkv, D, C, rank, layout, two_part):
    monkeypatch.setattr(L, "FUSE_CHUNKS", one_launch)
    for name in ("RingForward", "RingBackward") if one_launch else ("native",):
        monkeypatch.setattr(L, name, _not_used)
    g = torch.Generator().manual_seed(5)
    mk = lambda h, d: torch.randn(B, S, h, d, generator=g).to(torch.bfloat16)  # noqa: E731
    scale, dv = D**-0.5, min(D, 128)
    q = mk(Hq, D)
    ks = [mk(Hkv, 128 if two_part else D) for _ in range(C)]
    vs = [mk(Hkv, dv) for _ in range(C)]
    pes = [mk(1, 64)[:, :, 0] for _ in range(C)] if two_part else None
    full_ks = [torch.cat([k, pe[:, :, None].expand(-1, -1, Hkv, -1)], -1) for k, pe in zip(ks, pes)] if two_part else ks
    ref_o, ref_lse = R.ring_forward(q, full_ks, vs, scale, rank, C, layout)
    on_gpu = lambda ts: None if ts is None else [t.to(gpu) for t in ts]  # noqa: E731
    out, lse = L.ring_forward_local(q.to(gpu), on_gpu(ks), on_gpu(vs), scale, rank, C, layout, on_gpu(pes))
    check_bf16_result(out, ref_o, "O")
    check_lse(lse, ref_lse, "LSE2")

    # Both sides take O as the operator has it, in bf16: delta = rowsum(dO * O) inherits its rounding (2^-9 of each |O dO|),
    # which a row with one or two keys and a saturated softmax does not average out.
    dout, o = mk(Hq, dv), ref_o.to(torch.bfloat16)
    ref_dq, ref_dk, ref_dv = R.ring_backward(dout, q, o, ref_lse, full_ks, vs, scale, rank, C, layout)
    dq, dk, dv_, *dpe = L.ring_backward_local(dout.to(gpu), q.to(gpu), o.to(gpu), ref_lse.to(gpu, torch.float32), on_gpu(ks),
                                              on_gpu(vs), scale, rank, C, layout, on_gpu(pes))  # fmt: skip
    check_bf16_result(dq, ref_dq, "dQ", otol=1e-3)
    for j in range(C):
        assert (dk[j] is None) == (ref_dk[j] is None)
        if ref_dk[j] is None:
            continue
        check_bf16_result(dk[j], ref_dk[j][..., : dk[j].shape[-1]], f"chunk {j} dK", otol=1e-3)
        check_bf16_result(dv_[j], ref_dv[j], f"chunk {j} dV", otol=1e-3)
        if two_part:
            check_bf16_result(dpe[0][j], ref_dk[j][..., 128:].sum(2), f"chunk {j} dk_pe", otol=1e-3)


@pytest.mark.parametrize("S,Hq,Hkv,D,C", [(1030, 2, 1, 128, 4), (1030, 2, 2, 192, 4), (1030, 2, 1, 64, 4), (650, 2, 2, 192, 8), (98, 4, 2, 128, 2), (130, 260, 130, 64, 2)])
def test_share_of_rows_that_see_nothing_at_first(gpu, monkeypatch, S, Hq, Hkv, D, C):
    """Rank 0, zigzag: the first half of the rows sees only its own chunk, which comes last; a workgroup across the halves walks all of them."""
    test_share(gpu, monkeypatch, True, 1, S, Hq, Hkv, D, C, 0, "zigzag", False)


@pytest.mark.parametrize("scale,size", [(4.0, 1.0), (1e-3, 1.0), (128**-0.5, 30.0), (30.0, 3.0)])
def test_share_of_rows_that_see_nothing_at_first_at_other_scales(gpu, scale, size):
    """Scores of up to some 10^4 either way; each row against all keys it sees."""
    g = torch.Generator(device=gpu).manual_seed(8)
    mk = lambda: (size * torch.randn(1, 1030, 2, 128, generator=g, device=gpu)).to(torch.bfloat16)  # noqa: E731
    q, ks, vs = mk(), [mk() for _ in range(3)], [mk() / size for _ in range(3)]
    out, lse = L.ring_forward_local(q, ks, vs, scale, 0, 3, "zigzag")
    at = lambda j: torch.cat([torch.arange(515) + 515 * j, torch.arange(515) + 515 * (5 - j)])  # noqa: E731
    hidden = (torch.cat([at(j) for j in range(3)])[None, :] > at(0)[:, None]).to(gpu)
    s = q[0].transpose(0, 1).double() @ torch.cat(ks, 1)[0].permute(1, 2, 0).double().contiguous() * scale
    s = s.masked_fill(hidden, float("-inf"))
    # fp32 scores and LSE of size x: 2^-23 x log2(e) each, over some dozen roundings
    bound = 1e-3 + 16 * 2**-23 * 1.4427 * s[s > -1e30].abs().max().item()
    check_lse(lse, torch.logsumexp(s, -1)[None] / 0.6931471805599453, "LSE2", tol=bound)
    if scale * size**2 <= 128:  # (beyond, scores close to each other are rounded apart: P is another function)
        check_bf16_result(out, (torch.softmax(s, -1) @ torch.cat(vs, 1)[0].transpose(0, 1).double().contiguous()).transpose(0, 1)[None], "O")


def test_share_of_unequal_rows_64_features(gpu, monkeypatch):
    """The two-team forward over several chunks."""
    test_share(gpu, monkeypatch, True, 1, 1026, 36, 36, 64, 2, 0, "zigzag", False)


# Backward of shares with more 128-row query workgroups than one grid of dK/dV and dQ takes (attn_bwd_dkdv.hip, one_grid: two per
# compute unit at 192 features, four at 128, eight against more than two chunks' keys): two launches, the dQ one with two workgroups per
# compute unit; and the last of the single grids (64 features: all of these). Chunk ends, half chunks and half rows fall into tiles in all of them. Keys in two parts
# with 16 and 33 MiB of per-head gradients of the shared part, written through and not.
@pytest.mark.parametrize("one_grid,S,Hq,Hkv,D,C,rank,layout,two_part", [
    (1, 130, 516, 258, 64, 3, 1, "zigzag", False), (1, 130, 516, 516, 128, 3, 1, "zigzag", False), (0, 258, 344, 86, 128, 2, 1, "contiguous", False),
    (1, 130, 260, 130, 128, 3, 1, "zigzag", False), (0, 130, 516, 258, 128, 2, 0, "zigzag", False), (0, 130, 516, 516, 128, 2, 1, "zigzag", False),
    (0, 130, 1028, 514, 128, 3, 1, "zigzag", False), (0, 130, 260, 260, 192, 3, 1, "zigzag", False), (0, 258, 172, 172, 192, 2, 1, "contiguous", True),
    (0, 130, 260, 260, 192, 2, 0, "zigzag", True), (0, 130, 516, 516, 192, 2, 1, "contiguous", True)])  # fmt: skip
def test_share_with_many_workgroups(gpu, monkeypatch, one_grid, S, Hq, Hkv, D, C, rank, layout, two_part):
    monkeypatch.setattr(H, "DS_BUFFER_LIMIT_BYTES", 0)  # no dS hand-over: every kernel recomputes
    steps = sorted(L.ring_schedule(rank, C, S, layout), key=lambda st: (st.kv_rank == rank, st.q_rows[0]))
    chunks = (_C.KeyChunk * len(steps))(*(_C.KeyChunk(rows=st.kv_rows[1] - st.kv_rows[0], q_row0=st.q_rows[0]) for st in steps))
    args, plan = _C.AttnBwdArgs(B=1, Sq=S, Skv=S, Hq=Hq, Hkv=Hkv, Dqk=D, Dv=min(D, 128)), _C.AttnBwdPlan()
    _C.check(_C.lib().pith_attn_bwd_chunks_plan(_C.byref(args), chunks, len(steps), _C.byref(plan)))
    assert plan.one_grid == one_grid
    test_share(gpu, monkeypatch, True, 1, S, Hq, Hkv, D, C, rank, layout, two_part)


@pytest.mark.parametrize("full,S,Hq,Hkv,rank", [(0, 1100, 56, 2, 1), (1, 1100, 58, 2, 1), (0, 1100, 120, 4, 0), (1, 1090, 58, 2, 2), (1, 1278, 52, 2, 2), (1, 2100, 62, 2, 0), (0, 1400, 48, 2, 0)])
def test_forward_a_little_above_whole_rounds(gpu, monkeypatch, full, S, Hq, Hkv, rank):
    """On 256 compute units 128-row workgroups for just below and above two rounds (256-row ones there, up to 1.15 per unit and an odd number to a head; rank 2, whose rows are nearly equal, in any case) and above four,
    against float32 and against a launch per ring step; either rounds P and the result to bf16, and a merge rounds once more: two steps (2^-8
    each) of the largest element."""
    steps = sorted(L.ring_schedule(rank, 3, S, "zigzag"), key=lambda st: (st.kv_rank == rank, st.q_rows[0]))
    chunks = (_C.KeyChunk * len(steps))(*(_C.KeyChunk(rows=st.kv_rows[1] - st.kv_rows[0], q_row0=st.q_rows[0]) for st in steps))
    split = ctypes.c_int32(-1)
    _C.check(_C.lib().pith_attn_fwd_split(_C.byref(_C.AttnFwdArgs(B=1, Sq=S, Hq=Hq, Hkv=Hkv, Dqk=128, Dv=128)), chunks, len(steps), _C.byref(split)))
    assert (split.value == 0) == bool(full)
    g = torch.Generator(device=gpu).manual_seed(7)
    mk = lambda h: torch.randn(1, S, h, 128, generator=g, device=gpu).to(torch.bfloat16)  # noqa: E731
    q, ks, vs = mk(Hq), [mk(Hkv) for _ in range(3)], [mk(Hkv) for _ in range(3)]
    out, lse = L.ring_forward_local(q, ks, vs, 128**-0.5, rank, 3, "zigzag")
    at = lambda j: torch.cat([torch.arange(S // 2) + S // 2 * j, torch.arange(S // 2) + S // 2 * (5 - j)])  # noqa: E731
    hidden = (torch.cat([at(j) for j in range(3)])[None, :] > at(rank)[:, None]).to(gpu)
    k, v = torch.cat(ks, 1)[0].float(), torch.cat(vs, 1)[0].float()
    for h in range(0, Hq, 7):  # (heads of every group)
        s = (q[0, :, h].float() @ k[:, h * Hkv // Hq].t().contiguous()) * 128**-0.5
        s = s.masked_fill(hidden, float("-inf"))
        check_bf16_result(out[0, :, h], torch.softmax(s, -1) @ v[:, h * Hkv // Hq], f"O, head {h}")
        check_lse(lse[0, h], torch.logsumexp(s, -1) / 0.6931471805599453, f"LSE2, head {h}")
    monkeypatch.setattr(L, "FUSE_CHUNKS", False)
    stepwise, lse_steps = L.ring_forward_local(q, ks, vs, 128**-0.5, rank, 3, "zigzag")
    assert (out.float() - stepwise.float()).abs().max() <= 2**-7 * stepwise.float().abs().max()
    assert (lse - lse_steps).abs().max() < 1e-3
