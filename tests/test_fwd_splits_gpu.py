"""The forward's work splits on both sides of every line of its dispatch, and at the edges of the two-workgroup kernel's tiles,
against plain fp32 PyTorch."""

import pytest
import torch

from helpers import check_bf16_result, check_lse
from pithtrain_amd.operators.mla.hip import _mla_fwd

pytestmark = pytest.mark.gpu


def _reference(q, k, v, scale, causal):
    """O and base-2 LSE in fp32, one query head at a time."""
    b, sq, hq, _ = q.shape
    group = hq // k.shape[2]
    o = torch.empty(b, sq, hq, v.shape[-1], device=q.device)
    lse = torch.empty(b, hq, sq, device=q.device)
    mask = torch.ones(sq, k.shape[1], dtype=torch.bool, device=q.device).triu(1) if causal else None
    for bi in range(b):
        for h in range(hq):
            s = (q[bi, :, h].float() @ k[bi, :, h // group].float().t().contiguous()) * scale
            if causal:
                s.masked_fill_(mask, float("-inf"))
            lse[bi, h] = torch.logsumexp(s, -1) / 0.6931471805599453
            o[bi, :, h] = torch.softmax(s, -1) @ v[bi, :, h // group].float()
    return o, lse


@pytest.mark.parametrize("B,Sq,Skv,Hq,Hkv,D,causal", [
    # two-workgroup kernel: one row, tile and wave edges, ragged keys
    (1, 1, 1, 2, 1, 64, True), (1, 33, 33, 2, 2, 64, True), (2, 129, 129, 4, 2, 64, True), (1, 70, 200, 4, 1, 64, False),
    (1, 640, 640, 4, 4, 64, True), (1, 127, 127, 2, 1, 128, True), (1, 65, 257, 4, 2, 128, False), (1, 512, 512, 2, 2, 192, True),
    # 256 / 257 and 512 / 513 workgroups of 128 rows; streams of 512 / 513, 1024 / 1025, 1535 / 1536 keys
    (1, 512, 512, 16, 4, 128, False), (1, 513, 513, 16, 4, 128, False), (1, 520, 520, 52, 4, 128, True), (1, 896, 1025, 37, 37, 128, False),
    (1, 896, 1024, 37, 37, 128, False), (1, 1535, 1535, 42, 2, 192, True), (1, 1536, 1536, 42, 2, 192, True), (1, 3072, 3072, 22, 2, 128, True),
])  # fmt: skip
def test_forward_splits(gpu, B, Sq, Skv, Hq, Hkv, D, causal):
    g = torch.Generator(device=gpu).manual_seed(9)
    mk = lambda s, h, d: torch.randn(B, s, h, d, generator=g, device=gpu).to(torch.bfloat16)  # noqa: E731
    q, k, v = mk(Sq, Hq, D), mk(Skv, Hkv, D), mk(Skv, Hkv, min(D, 128))
    o, lse = _mla_fwd(q, k, v, D**-0.5, causal)
    ref_o, ref_lse = _reference(q, k, v, D**-0.5, causal)
    check_bf16_result(o, ref_o, "O")
    check_lse(lse, ref_lse, "LSE2")


@pytest.mark.parametrize("B,Sq,Skv,Hq,Hkv,D,causal", [
    # 64-row workgroups: stream of 256 / 257 and 320 / 321 keys, one tile for one team only, rows that see one key block
    (1, 256, 256, 4, 2, 64, True), (1, 257, 257, 4, 2, 64, True), (1, 320, 320, 2, 2, 128, False), (1, 1, 321, 2, 1, 128, False),
    (1, 33, 1025, 4, 4, 192, False), (2, 449, 449, 2, 1, 192, True), (1, 95, 350, 2, 2, 64, False), (1, 700, 700, 4, 1, 128, True),
    # 256 / 257 of them; under the mask 384 / 385 from 2048 keys and 512 / 513 from 6144 keys on
    (1, 512, 512, 32, 4, 128, True), (1, 2047, 2047, 12, 4, 128, True), (1, 2048, 2048, 12, 4, 128, True), (1, 2049, 2049, 12, 4, 192, True),
    (1, 6143, 6143, 5, 1, 128, True), (1, 6144, 6144, 5, 5, 192, True),
    # 128-row workgroups of two teams: 1024 / 1025 keys, 2048 / 2049 under the mask, ragged, one and two per compute unit
    (1, 900, 1025, 32, 8, 64, False), (1, 900, 1024, 32, 8, 64, False), (1, 2048, 2048, 32, 4, 64, True), (1, 2049, 2049, 30, 3, 64, True),
    (1, 4096, 4096, 16, 2, 64, True), (1, 2111, 2111, 11, 11, 64, True),
])  # fmt: skip
def test_forward_key_splits(gpu, B, Sq, Skv, Hq, Hkv, D, causal):
    test_forward_splits(gpu, B, Sq, Skv, Hq, Hkv, D, causal)


@pytest.mark.parametrize("B,Sq,Skv,Hq,Hkv,D,causal", [
    # 64-row workgroups whose teams take turns: 7 / 8 / 9 intervals, an odd tile, one ragged key, waves that end before their workgroup
    (1, 64, 896, 2, 1, 128, False), (1, 64, 897, 2, 1, 128, False), (1, 70, 1024, 2, 2, 192, False), (2, 33, 1025, 4, 2, 192, False),
    (1, 961, 961, 2, 2, 192, True), (1, 1023, 1023, 4, 1, 128, True), (1, 1089, 1089, 2, 1, 128, True),
    # as many of them as one and a quarter, one and a half or two per unit, from 1024, 1536 and 2048 (128 features: 3072) keys on
    (1, 1023, 1023, 20, 20, 192, True), (1, 1024, 1024, 20, 4, 128, True), (1, 1535, 1535, 16, 4, 128, True), (1, 1536, 1536, 16, 16, 192, True),
    (1, 2048, 2048, 16, 16, 192, True), (1, 2050, 2050, 16, 16, 192, True), (1, 3072, 3072, 10, 2, 128, True),
])  # fmt: skip
def test_forward_teams_in_turns(gpu, B, Sq, Skv, Hq, Hkv, D, causal):
    test_forward_splits(gpu, B, Sq, Skv, Hq, Hkv, D, causal)


@pytest.mark.parametrize("layout", ["contiguous", "zigzag"])
@pytest.mark.parametrize("rows,D", [(510, 192), (514, 128), (258, 192)])
def test_shares_of_teams_in_turns(gpu, rows, D, layout):
    """Streams over several chunks, whose tiles the teams take in turns: each row against all keys it sees."""
    from pithtrain_amd.operators.ring_attention.local import ring_forward_local

    rank, cp, h = 1, 4, 2
    g = torch.Generator(device=gpu).manual_seed(4)
    mk = lambda s, d: torch.randn(1, s, h, d, generator=g, device=gpu).to(torch.bfloat16)  # noqa: E731
    half = rows // 2
    # positions of a chunk's rows in the sequence
    at = lambda j: torch.cat([torch.arange(half) + half * j, torch.arange(half) + half * (2 * cp - 1 - j)]) if layout == "zigzag" else torch.arange(rows) + rows * j  # noqa: E731
    seen = range(cp) if layout == "zigzag" else range(rank + 1)
    q, ks, vs = mk(rows, D), [mk(rows, D) if j in seen else None for j in range(cp)], [mk(rows, min(D, 128)) if j in seen else None for j in range(cp)]
    o, lse = ring_forward_local(q, ks, vs, D**-0.5, rank, cp, layout)
    k, v = (torch.cat([x for x in t if x is not None], 1) for t in (ks, vs))
    hidden = torch.cat([at(j) for j in seen])[None, :] > at(rank)[:, None]
    s = (q[0].transpose(0, 1).float() @ k[0].permute(1, 2, 0).float().contiguous()) * D**-0.5
    s = s.masked_fill(hidden.to(gpu), float("-inf"))
    check_lse(lse, torch.logsumexp(s, -1)[None] / 0.6931471805599453, "LSE2")
    check_bf16_result(o, (torch.softmax(s, -1) @ v[0].transpose(0, 1).float().contiguous()).transpose(0, 1)[None], "O")


@pytest.mark.parametrize("B,Sq,Skv,Hq,Hkv,D,causal", [
    # 64-row workgroups of 4 waves: one ragged row, key halves that do not exist or end early, 64 / 65 and 512 / 513 keys
    *[(1, sq, skv, 2, 1, d, sq == skv) for d in (64, 128, 192) for sq, skv in ((65, 65), (1, 65), (64, 96), (33, 97), (127, 128), (95, 350), (300, 300), (512, 512))],
    (1, 70, 513, 2, 1, 64, False), (2, 257, 257, 3, 3, 192, True),
    # one and two of them per unit (from 129 keys on), at 64 features three and four, five from 1536 keys on; and on the other side of these lines
    (2, 512, 512, 16, 4, 128, True), (4, 320, 320, 25, 25, 128, True), (8, 128, 128, 32, 32, 192, True), (8, 129, 129, 21, 21, 192, True),
    (4, 192, 192, 43, 43, 64, False), (4, 576, 576, 32, 8, 64, True), (4, 577, 577, 32, 8, 64, True), (2, 1535, 1535, 26, 13, 64, True), (2, 1536, 1536, 26, 13, 64, True),
    (4, 512, 512, 32, 8, 64, True), (5, 512, 512, 27, 9, 64, True), (2, 2048, 2048, 18, 6, 64, True), (1, 2561, 2561, 16, 4, 64, True), (1, 2049, 2049, 12, 4, 64, False), (4, 129, 129, 32, 8, 128, True),
    # wave pairs of 128-row workgroups from 257 (192 features: 384) keys on
    (2, 255, 300, 70, 70, 128, False), (4, 256, 256, 32, 8, 128, False), (4, 256, 257, 32, 8, 128, False), (2, 384, 384, 33, 33, 192, False), (2, 1024, 1024, 20, 20, 192, True),
])  # fmt: skip
def test_forward_small_workgroups(gpu, B, Sq, Skv, Hq, Hkv, D, causal):
    test_forward_splits(gpu, B, Sq, Skv, Hq, Hkv, D, causal)


@pytest.mark.parametrize("layout", ["contiguous", "zigzag"])
@pytest.mark.parametrize("rows,D", [(66, 64), (100, 128), (130, 192)])
def test_shares_of_small_workgroups(gpu, rows, D, layout):
    test_shares_of_teams_in_turns(gpu, rows, D, layout)


@pytest.mark.parametrize("B,S,Hq,Hkv,D,causal", [
    # a row above one and two whole rounds of 128-row workgroups on 256 compute units, and on both sides of the lines above them
    (1, 8193, 4, 1, 128, True), (1, 9473, 4, 1, 128, True), (1, 4097, 16, 2, 128, True), (1, 5121, 16, 2, 128, True), (1, 4097, 8, 8, 192, True),
    (1, 4609, 8, 8, 192, True), (1, 2113, 16, 16, 192, True), (1, 2599, 16, 16, 192, True), (1, 4097, 16, 16, 192, True), (1, 4353, 16, 16, 192, True),
    (1, 4097, 8, 2, 64, True), (1, 4353, 8, 2, 64, True), (1, 8193, 8, 2, 64, True), (2, 6145, 8, 2, 64, True), (1, 2049, 32, 4, 128, False),
    (1, 2817, 32, 4, 128, False), (1, 1408, 24, 3, 128, False), (1, 1409, 24, 3, 128, False),
])  # fmt: skip
def test_forward_above_whole_rounds(gpu, B, S, Hq, Hkv, D, causal):
    test_forward_splits(gpu, B, S, S, Hq, Hkv, D, causal)
