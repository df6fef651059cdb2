"""The backward's kernels at the edges of their tiles and on both sides of the lines between them, against plain fp32 PyTorch."""

import pytest
import torch

from helpers import check_bf16_result
from pithtrain_amd import _C
from pithtrain_amd.operators.mla import hip
from pithtrain_amd.operators.mla.hip import _mla_bwd_dk_dv, _mla_bwd_dq, _mla_bwd_preprocess, _mla_fwd, attn_bwd_pair_into

pytestmark = pytest.mark.gpu


def _reference(q, k, v, dout, scale, causal):
    """dQ, dK, dV in fp32, one query head at a time."""
    b, sq, hq, _ = q.shape
    group = hq // k.shape[2]
    dq, dk, dv = (torch.zeros(t.shape, device=t.device) for t in (q, k, v))
    mask = torch.ones(sq, k.shape[1], dtype=torch.bool, device=q.device).triu(1) if causal else None
    for bi in range(b):
        for h in range(hq):
            qh, kh, vh, do = q[bi, :, h].float(), k[bi, :, h // group].float(), v[bi, :, h // group].float(), dout[bi, :, h].float()
            s = (qh @ kh.t().contiguous()) * scale
            if causal:
                s.masked_fill_(mask, float("-inf"))
            p = torch.softmax(s, -1)
            dp = do @ vh.t().contiguous()
            ds = p * (dp - (dp * p).sum(-1, keepdim=True)) * scale
            dq[bi, :, h] = ds @ kh
            dk[bi, :, h // group] += ds.t().contiguous() @ qh
            dv[bi, :, h // group] += p.t().contiguous() @ do
    return dq, dk, dv


CASES = [
    # one row; 32-row tiles and 128-row workgroups minus / plus one; ragged keys against ragged queries
    (1, 1, 1, 2, 1, 64, True), (1, 33, 33, 2, 2, 64, True), (2, 129, 129, 4, 2, 64, True), (1, 70, 200, 4, 1, 64, False),
    (1, 200, 70, 4, 2, 64, False), (1, 640, 640, 8, 4, 64, True), (1, 127, 127, 2, 1, 128, True), (1, 65, 257, 4, 2, 128, False),
    (1, 31, 256, 3, 3, 192, False), (1, 256, 256, 2, 2, 192, True), (1, 97, 33, 2, 2, 192, False),
    # 256 / 257 and 512 / 513 workgroups of 128 query rows, streams of 1535 / 1536 keys
    (1, 512, 512, 16, 4, 128, False), (1, 257, 300, 86, 86, 192, False), (1, 896, 300, 37, 37, 192, False), (1, 1535, 1535, 42, 2, 128, True),
    (1, 1536, 1536, 42, 42, 192, True), (1, 1664, 1664, 42, 2, 128, True),
]  # fmt: skip


@pytest.mark.parametrize("B,Sq,Skv,Hq,Hkv,D,causal", CASES)
def test_backward_splits(gpu, B, Sq, Skv, Hq, Hkv, D, causal):
    g = torch.Generator(device=gpu).manual_seed(13)
    mk = lambda s, h, d: torch.randn(B, s, h, d, generator=g, device=gpu).to(torch.bfloat16)  # noqa: E731
    dv_dim, scale = min(D, 128), D**-0.5
    q, k, v, dout = mk(Sq, Hq, D), mk(Skv, Hkv, D), mk(Skv, Hkv, dv_dim), mk(Sq, Hq, dv_dim)
    o, lse = _mla_fwd(q, k, v, scale, causal)
    delta = _mla_bwd_preprocess(o, dout)
    dq = _mla_bwd_dq(q, k, v, dout, lse, delta, scale, causal)
    dk, dv = _mla_bwd_dk_dv(q, k, v, dout, lse, delta, scale, causal)
    refs = _reference(q, k, v, dout, scale, causal)
    for name, got, want in zip(("dQ", "dK", "dV"), (dq, dk, dv), refs):
        check_bf16_result(got, want, name, otol=1e-3)
    pair = [torch.empty_like(t) for t in (q, k, v)]
    attn_bwd_pair_into(q, k, v, dout, lse, delta, *pair, scale, causal)
    for name, got, want in zip(("dQ", "dK", "dV"), pair, refs):
        check_bf16_result(got, want, name + " of the pair", otol=1e-3)


@pytest.mark.parametrize("B,Sq,Skv,Hq,Hkv,D,causal", [
    # both sides of 1.5 and of 2.5 workgroups per compute unit, above 2 of them, streams of 1023 / 1024 and 1535 / 1536 keys
    (1, 1536, 1536, 32, 4, 128, False), (1, 1537, 1537, 32, 4, 128, False), (1, 2177, 2177, 30, 2, 128, False), (1, 2100, 700, 32, 4, 128, False),
    (1, 2560, 2560, 32, 4, 128, True), (1, 2561, 2561, 32, 4, 128, True), (1, 1024, 1024, 64, 8, 128, True), (1, 1023, 1023, 64, 8, 128, True),
    (1, 1536, 1536, 32, 32, 192, True), (1, 1535, 1535, 32, 32, 192, True), (1, 1500, 1600, 32, 32, 192, False),
])  # fmt: skip
def test_backward_pairs_of_a_few_rounds(gpu, monkeypatch, B, Sq, Skv, Hq, Hkv, D, causal):
    monkeypatch.setattr(hip, "DS_BUFFER_LIMIT_BYTES", 0)  # (192 features would hand dS over)
    test_backward_splits(gpu, B, Sq, Skv, Hq, Hkv, D, causal)


@pytest.mark.parametrize("B,Sq,Skv,Hq,Hkv,D", [
    # eight head parts: 32 MiB of partial sums, written through, and a row of keys more, for which there are four; ragged keys, the last of 32 missing; four
    # parts of 64 features
    (1, 129, 1024, 32, 4, 128), (1, 129, 1025, 32, 4, 128), (1, 70, 95, 16, 2, 128), (2, 100, 1000, 16, 4, 64),
])  # fmt: skip
def test_backward_of_split_head_groups(gpu, B, Sq, Skv, Hq, Hkv, D):
    test_backward_splits(gpu, B, Sq, Skv, Hq, Hkv, D, False)


def test_partial_sums_beyond_the_caches(gpu):
    """64 MiB of them, stored plainly."""
    args, plan = _C.AttnBwdArgs(B=4, Sq=1024, Skv=1024, Hq=16, Hkv=4, Dqk=128, Dv=128, causal=1), _C.AttnBwdPlan()
    _C.check(_C.lib().pith_attn_bwd_plan(_C.byref(args), _C.byref(plan)))
    assert plan.dkdv_split == 4 and _C.lib().pith_attn_bwd_dkdv_workspace_bytes(_C.byref(args)) == 64 << 20
    test_backward_splits(gpu, 4, 1024, 1024, 16, 4, 128, True)


@pytest.mark.parametrize("B,Sq,Skv,H,D", [(2, 200, 300, 8, 64), (1, 130, 257, 16, 128), (3, 300, 130, 16, 192), (2, 64, 2, 8, 128), (1, 513, 513, 24, 128)])
def test_backward_in_chunks_of_heads(gpu, B, Sq, Skv, H, D):
    """Without a mask more than eight heads (over the batch), a multiple of eight, are taken eight at a time."""
    test_backward_splits(gpu, B, Sq, Skv, H, H, D, False)


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("B,S,Hq,Hkv,D", [
    # one, 32, 33, 64, 65 and 97 rows in the last workgroup of 128: three to no waves without any, as one grid and as two launches
    (1, 257, 4, 2, 128), (1, 288, 4, 4, 64), (2, 161, 6, 3, 64), (1, 192, 4, 2, 192), (2, 193, 2, 2, 192), (1, 225, 4, 1, 128),
    (6, 385, 40, 40, 192), (4, 1025, 32, 8, 128), (8, 643, 16, 4, 128),
])  # fmt: skip
def test_waves_without_rows(gpu, B, S, Hq, Hkv, D, causal):
    test_backward_splits(gpu, B, S, S, Hq, Hkv, D, causal)


@pytest.mark.parametrize("one_grid,B,S,H,D,causal", [
    # 3.32 and 3.34 dQ workgroups per compute unit under the mask, 383 and 384 keys; 3.09 and 3.11 without; 192 features from 256 keys on
    (1, 1, 640, 170, 128, True), (0, 1, 640, 171, 128, True), (0, 1, 383, 171, 128, True), (1, 1, 384, 171, 128, True), (1, 1, 513, 158, 128, False),
    (0, 1, 513, 159, 128, False), (0, 1, 255, 150, 192, True), (1, 1, 256, 150, 192, True), (1, 1, 300, 128, 192, True),
])  # fmt: skip
def test_backward_pairs_at_the_lines_of_one_grid(gpu, monkeypatch, one_grid, B, S, H, D, causal):
    monkeypatch.setattr(hip, "DS_BUFFER_LIMIT_BYTES", 0)  # (the first two would hand dS over)
    args, plan = _C.AttnBwdArgs(B=B, Sq=S, Skv=S, Hq=H, Hkv=H, Dqk=D, Dv=min(D, 128), causal=causal), _C.AttnBwdPlan()
    _C.check(_C.lib().pith_attn_bwd_plan(_C.byref(args), _C.byref(plan)))
    assert plan.one_grid == one_grid
    test_backward_splits(gpu, B, S, S, H, H, D, causal)
