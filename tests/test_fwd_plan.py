"""Which work split a forward takes, asked on a machine without a GPU (256 compute units are assumed there)."""

import ctypes

import pytest

from pithtrain_amd import _C
from pithtrain_amd.operators.ring_attention.local import ring_schedule

FULL, DUO, HALF, TEAMS, QUARTER, SMALL = range(6)


def _split(b, s, hq, hkv, d, causal=1, skv=None):
    args, split = _C.AttnFwdArgs(B=b, Sq=s, Skv=skv or s, Hq=hq, Hkv=hkv, Dqk=d, Dv=min(d, 128), causal=causal), ctypes.c_int32(-1)
    _C.check(_C.lib().pith_attn_fwd_split(_C.byref(args), None, 0, _C.byref(split)))
    return split.value


def _share_split(b, s, hq, hkv, d, cp, rank, layout):
    steps = sorted(ring_schedule(rank, cp, s, layout), key=lambda st: (st.kv_rank == rank, st.q_rows[0]))
    chunks = (_C.KeyChunk * len(steps))(*(_C.KeyChunk(rows=st.kv_rows[1] - st.kv_rows[0], q_row0=st.q_rows[0]) for st in steps))
    args, split = _C.AttnFwdArgs(B=b, Sq=s, Hq=hq, Hkv=hkv, Dqk=d, Dv=min(d, 128)), ctypes.c_int32(-1)
    _C.check(_C.lib().pith_attn_fwd_split(_C.byref(args), chunks, len(steps), _C.byref(split)))
    return split.value


def test_split_query():
    assert (_split(1, 4096, 32, 4, 128, 0), _split(3, 1999, 32, 4, 128), _split(1, 2048, 8, 8, 128)) == (FULL, DUO, QUARTER)
    out = _C.byref(ctypes.c_int32())
    for bad in (dict(B=1, Sq=0, Skv=1, Hq=3, Hkv=2), dict(B=0, Sq=1, Skv=1, Hq=1, Hkv=1)):
        assert _C.lib().pith_attn_fwd_split(_C.byref(_C.AttnFwdArgs(**bad)), None, 0, out) == -2
    assert _C.lib().pith_attn_fwd_split(_C.byref(_C.AttnFwdArgs(B=1, Sq=1, Skv=1, Hq=1, Hkv=1)), (_C.KeyChunk * 1)(), 17, out) == -2
    assert _C.lib().pith_attn_fwd_split(None, None, 0, out) == -1


@pytest.mark.parametrize("small,b,s,h,d,causal", [
    # 64 features, unequal rows, more than two 64-row workgroups per unit: all at once and rows that pad 128, many tiles, whole rounds
    (1, 12, 128, 32, 64, 1), (0, 14, 128, 32, 64, 1), (0, 16, 128, 32, 64, 1), (1, 10, 192, 32, 64, 1), (0, 12, 192, 32, 64, 1), (0, 8, 256, 32, 64, 1),
    (1, 6, 320, 32, 64, 1), (0, 7, 320, 29, 64, 1), (0, 3, 370, 64, 64, 1), (1, 3, 512, 32, 64, 1), (0, 5, 512, 27, 64, 1), (0, 5, 448, 27, 64, 1),
    (1, 2, 768, 32, 64, 1), (1, 3, 768, 28, 64, 1), (0, 3, 768, 27, 64, 1), (1, 2, 900, 30, 64, 1), (0, 3, 900, 24, 64, 1), (1, 4, 512, 32, 64, 1), (0, 7, 256, 30, 64, 1), (0, 3, 768, 32, 64, 1), (1, 2, 1000, 32, 64, 1), (0, 3, 1024, 23, 64, 1), (1, 1, 1088, 64, 64, 1), (1, 2, 1200, 29, 64, 1),
    (1, 2, 2048, 18, 64, 1), (1, 2, 2048, 16, 64, 1), (1, 1, 2560, 20, 64, 1), (0, 4, 2855, 4, 64, 1), (0, 1, 2914, 16, 64, 1), (0, 1, 6144, 8, 64, 1),
    (1, 1, 4096, 16, 64, 1), (1, 1, 4404, 16, 64, 1),
    # without a mask, up to two per unit
    (0, 3, 192, 30, 64, 0), (1, 6, 192, 28, 64, 0), (0, 3, 256, 29, 64, 0), (0, 3, 320, 26, 64, 0), (0, 3, 384, 25, 64, 0), (1, 2, 384, 26, 64, 0), (1, 1, 1024, 32, 64, 0),
    (1, 1, 2048, 12, 64, 0), (0, 1, 2304, 14, 64, 0), (0, 1, 6144, 5, 64, 0),
    # 128 and 192 features
    (0, 5, 128, 27, 128, 1), (0, 8, 128, 32, 128, 1), (0, 3, 129, 30, 128, 1), (1, 4, 129, 32, 128, 1), (0, 3, 192, 30, 192, 1), (1, 4, 192, 26, 192, 1), (1, 3, 256, 22, 192, 1),
    (1, 2, 512, 32, 128, 1), (0, 4, 256, 27, 128, 0),
])  # fmt: skip
def test_calls_of_small_workgroups(small, b, s, h, d, causal):
    """As measured (table at small_workgroups)."""
    assert (_split(b, s, h, h, d, causal) == SMALL) == bool(small)


def test_few_rows():
    """Up to one 64-row workgroup per unit: two teams from 385 keys on at 64 features, 513 at the others."""
    assert [_split(1, s, 20, 20, 64) for s in (64, 384, 385, 512)] == [DUO, SMALL, QUARTER, QUARTER]
    assert [_split(1, s, 20, 20, d) for d in (128, 192) for s in (512, 513)] == [SMALL, QUARTER] * 2
    assert [_split(4, s, 20, 20, 128, 0) for s in (256, 257)] == [DUO, HALF]


def test_short_rows_against_several_chunks():
    """Key halves from 1024 keys on for one chunk and in rank 0, from 1536 in others, as measured."""
    assert [_split(1, s, 44, 44, 192) for s in (1023, 1024)] == [DUO, HALF] and _share_split(2, 640, 32, 32, 192, 2, 0, "zigzag") == HALF
    assert _share_split(1, 2048, 40, 10, 64, 4, 2, "zigzag") == DUO and _split(1, 2048, 40, 10, 64) == SMALL
    assert _share_split(2, 582, 64, 16, 64, 4, 0, "zigzag") == SMALL and _share_split(2, 756, 48, 12, 64, 2, 1, "zigzag") == DUO
    assert [_share_split(2, s, 40, 8, 128, 4, 2, "zigzag") for s in (396, 510, 512)] == [DUO, DUO, HALF]


def test_shares_of_64_features_of_long_streams():
    """Nearly equal rows, two teams above 2048 keys."""
    assert _share_split(2, 2240, 4, 4, 64, 4, 3, "contiguous") == TEAMS and _share_split(1, 500, 40, 40, 64, 4, 3, "contiguous") == SMALL
    assert _share_split(1, 1152, 32, 8, 64, 4, 0, "zigzag") == SMALL  # (unequal ones stay at four waves)


@pytest.mark.parametrize("full,b,s,hq,hkv,cp,rank", [
    (1, 1, 2100, 32, 4, 4, 2), (1, 2, 2100, 16, 4, 4, 1), (1, 1, 2176, 32, 4, 4, 0), (1, 1, 2200, 32, 8, 4, 2), (1, 1, 1664, 40, 8, 4, 2), (1, 1, 2100, 32, 4, 2, 0),
    (0, 1, 2944, 24, 3, 4, 2), (0, 1, 1920, 40, 8, 4, 2), (0, 1, 2862, 24, 3, 4, 0), (0, 1, 1364, 48, 8, 4, 0), (0, 1, 1588, 40, 5, 2, 1),
    (0, 1, 1100, 64, 4, 4, 2), (1, 1, 1100, 58, 2, 4, 2), (0, 1, 1100, 56, 2, 4, 2), (0, 1, 2400, 32, 4, 4, 1), (1, 1, 2300, 64, 4, 4, 0), (1, 1, 2200, 64, 4, 4, 2),
    (0, 2, 2944, 24, 3, 2, 0), (0, 2, 1408, 48, 8, 4, 1), (0, 2, 1100, 64, 4, 4, 2), (0, 2, 2100, 16, 16, 4, 1),
])  # fmt: skip
def test_zigzag_shares_of_256_row_workgroups(full, b, s, hq, hkv, cp, rank):
    """As measured (comment at pick_split)."""
    assert (_share_split(b, s, hq, hkv, 128, cp, rank, "zigzag") == FULL) == bool(full)


@pytest.mark.parametrize("quarter,b,s,hq,hkv,d,cp,rank", [
    # the longer half in up to 256 workgroups of 64 rows or in more
    (1, 1, 896, 32, 4, 128, 8, 0), (1, 1, 960, 32, 4, 128, 8, 2), (1, 2, 1024, 16, 4, 128, 8, 0), (1, 3, 1204, 8, 2, 128, 8, 2), (1, 1, 896, 32, 4, 128, 4, 0), (1, 1, 960, 32, 32, 192, 8, 0),
    (1, 3, 1280, 8, 8, 192, 8, 0), (0, 1, 1022, 32, 4, 128, 8, 2), (0, 1, 1530, 20, 5, 128, 8, 0), (0, 3, 1270, 8, 2, 128, 8, 2), (0, 1, 1300, 24, 3, 128, 8, 0), (0, 1, 1022, 32, 32, 192, 8, 0),
    (0, 1, 768, 40, 8, 128, 2, 0), (1, 1, 1850, 16, 4, 64, 4, 0), (1, 2, 788, 16, 16, 64, 2, 0), (1, 1, 1062, 16, 16, 128, 4, 2), (0, 3, 2510, 4, 4, 192, 2, 1), (1, 3, 2074, 4, 4, 192, 4, 2), (0, 1, 678, 32, 32, 192, 4, 2), (1, 1, 2370, 8, 8, 192, 2, 1), (1, 1, 1782, 16, 16, 192, 8, 3),
    (1, 1, 1240, 16, 16, 192, 4, 2), (1, 2, 636, 16, 4, 128, 8, 4), (0, 3, 552, 16, 4, 64, 4, 2), (0, 1, 1280, 24, 6, 64, 2, 1), (0, 3, 256, 32, 8, 64, 8, 4), (0, 1, 1024, 20, 20, 192, 2, 1), (1, 1, 1290, 16, 4, 64, 2, 1), (1, 3, 2152, 4, 4, 64, 2, 1),
])  # fmt: skip
def test_zigzag_shares_of_64_row_workgroups_in_teams(quarter, b, s, hq, hkv, d, cp, rank):
    """As measured (in front of Split)."""
    assert (_share_split(b, s, hq, hkv, d, cp, rank, "zigzag") == QUARTER) == bool(quarter)
