"""How the backward is cut, asked on a machine without a GPU (256 compute units are assumed there)."""

import heapq

import pytest
import torch

from pithtrain_amd import _C
from pithtrain_amd._ext import native
from pithtrain_amd.operators.mla import hip as H
from pithtrain_amd.operators.ring_attention.local import ring_schedule

UNITS = 256


def _plan(b, sq, skv, hq, hkv, causal, d=128):
    args, plan = _C.AttnBwdArgs(B=b, Sq=sq, Skv=skv, Hq=hq, Hkv=hkv, Dqk=d, Dv=min(d, 128), causal=causal), _C.AttnBwdPlan()
    _C.check(_C.lib().pith_attn_bwd_plan(_C.byref(args), _C.byref(plan)))
    return plan


def _share_plan(b, s, hq, hkv, cp, rank, layout, d=64):
    steps = sorted(ring_schedule(rank, cp, s, layout), key=lambda st: (st.kv_rank == rank, st.q_rows[0]))
    chunks = (_C.KeyChunk * len(steps))(*(_C.KeyChunk(rows=st.kv_rows[1] - st.kv_rows[0], q_row0=st.q_rows[0]) for st in steps))
    args, plan = _C.AttnBwdArgs(B=b, Sq=s, Skv=s, Hq=hq, Hkv=hkv, Dqk=d, Dv=min(d, 128)), _C.AttnBwdPlan()
    _C.check(_C.lib().pith_attn_bwd_chunks_plan(_C.byref(args), chunks, len(steps), _C.byref(plan)))
    return plan


def test_plan_query():
    assert (_plan(1, 8192, 4096, 32, 4, 0).dkdv_rows, _plan(1, 256, 256, 8, 2, 1).dkdv_rows, _plan(1, 8192, 8192, 16, 16, 1, 192).dkdv_rows) == (256, 128, 128)
    assert _plan(1, 256, 256, 8, 2, 1).dkdv_split == 4
    assert not _plan(1, 4096, 4096, 32, 4, 0).dq_ds_pairs and _plan(1, 4096, 4096, 16, 16, 1, 192).dq_ds_pairs
    for bad in (dict(B=1, Sq=1, Skv=1, Hq=3, Hkv=2), dict(B=0, Sq=1, Skv=1, Hq=1, Hkv=1)):
        assert _C.lib().pith_attn_bwd_plan(_C.byref(_C.AttnBwdArgs(**bad)), _C.byref(_C.AttnBwdPlan())) == -2
    assert _C.lib().pith_attn_bwd_plan(None, None) == -1


@pytest.mark.parametrize("b,s,hq,hkv", [(65535, 1, 130, 130), (65535, 129, 120, 8), (60000, 1, 270, 30), (65535, 1, 256, 1)])
def test_one_grid_is_one_that_can_be_launched(b, s, hq, hkv):
    """64 features: two grids of fewer than 2^32 threads each may make a grid of more, which the runtime refuses."""
    dq, dkdv = -(-s // 128) * b * hq, -(-s // 128) * b * hkv
    assert _plan(b, s, s, hq, hkv, 0, 64).one_grid == ((dq + dkdv) * 256 < 2**32)
    assert _plan(64, s, s, hq, hkv, 0, 64).one_grid


@pytest.mark.parametrize("one,b,s,hq,hkv,cp,rank,layout", [
    (0, 1, 12288, 16, 4, 4, 0, "zigzag"), (0, 1, 16384, 16, 4, 4, 0, "zigzag"), (0, 1, 24576, 8, 2, 4, 0, "zigzag"), (0, 1, 16384, 16, 4, 4, 2, "contiguous"),
    (0, 1, 12288, 16, 4, 4, 3, "contiguous"),
    (1, 1, 12288, 16, 4, 4, 1, "zigzag"), (1, 1, 4096, 64, 8, 4, 0, "zigzag"), (1, 1, 8192, 32, 8, 4, 1, "zigzag"), (1, 1, 5120, 32, 8, 4, 0, "zigzag"),
    (1, 1, 32768, 8, 2, 2, 0, "zigzag"), (1, 1, 16384, 16, 16, 4, 0, "zigzag"), (1, 3, 3001, 16, 4, 2, 1, "contiguous"), (1, 2, 8192, 16, 16, 4, 2, "zigzag"),
    (1, 1, 16384, 32, 8, 4, 0, "zigzag"), (1, 1, 10240, 32, 8, 4, 0, "zigzag"), (1, 1, 12288, 32, 8, 4, 0, "zigzag"), (1, 3, 4096, 16, 4, 4, 0, "zigzag"),
])  # fmt: skip
def test_shares_of_64_features(one, b, s, hq, hkv, cp, rank, layout):
    """Both gradients in one grid unless either kernel alone is whole rounds of long walks, as measured (table at one_grid)."""
    assert _share_plan(b, s, hq, hkv, cp, rank, layout).one_grid == one


def _makespan(jobs):
    """Jobs handed out in order, each to the compute unit that is free first."""
    free = [0.0] * UNITS
    for j in jobs:
        heapq.heappush(free, heapq.heappop(free) + j)
    return max(free)


@pytest.mark.parametrize("tiles,heads", [(1, 256), (2, 128), (8, 32), (16, 16), (32, 8), (9, 32), (18, 16), (3, 96), (10, 32), (5, 64), (12, 32),
                                         (2, 192), (14, 32), (16, 32), (4, 128), (18, 32), (20, 32), (24, 32), (32, 32), (3, 86), (33, 8)])  # fmt: skip
def test_dq_from_ds_goes_out_in_the_order_that_ends_first(tiles, heads):
    """512-row tiles under the mask: tile t reads t + 1/2 units of dS. Either consecutive rows, the heaviest workgroups first, or
    pairs of 256-row blocks from both ends."""
    consecutive = _makespan([t + 0.5 for t in reversed(range(tiles)) for _ in range(heads)])
    pairs = _makespan([tiles / 2] * (tiles * heads))
    chosen = pairs if _plan(1, 512 * tiles, 512 * tiles, heads, heads, 1).dq_ds_pairs else consecutive
    # 10 %: busy units take over the memory rate that idle ones leave (24 tiles x 32 heads: 39.5 against 36, measured 2 % apart)
    assert chosen <= 1.1 * min(consecutive, pairs)
    if tiles * heads <= UNITS:
        assert chosen == pairs


@pytest.mark.parametrize("pairs,b,s,h", [(1, 1, 4096, 16), (1, 1, 3072, 16), (1, 4, 1024, 16), (1, 1, 16384, 4), (1, 1, 129, 1), (0, 1, 4097, 16), (0, 1, 4608, 16),
                                         (0, 3, 1999, 16), (0, 1, 8192, 16), (0, 17, 255, 16), (0, 1, 128, 16)])  # fmt: skip
def test_order_of_dq_from_ds_at_192(pairs, b, s, h):
    """256-row workgroups, one round of which takes pairs of 128-row blocks; 128 rows have no hand-over. A share orders its rows alike."""
    assert _plan(b, s, s, h, h, 1, 192).dq_ds_pairs == pairs and not _plan(b, s, s, h, h, 0, 192).dq_ds_pairs
    assert _share_plan(b, s, h, h, 4, 2, "contiguous", 192).dq_ds_pairs == pairs and not _share_plan(b, s, h, h, 4, 2, "contiguous").dq_ds_pairs


@pytest.mark.parametrize("b,s,hq", [(1, 4096, 32), (2, 2048, 32), (8, 512, 32), (1, 8192, 16), (1, 9216, 16), (3, 1536, 32), (2, 2560, 32), (1, 5120, 32),
                                    (6, 1024, 32), (3, 1999, 32), (2, 3072, 32), (1, 7168, 32), (1, 9216, 32), (1, 10240, 32)])  # fmt: skip
def test_layers_that_gain_hand_ds_over(b, s, hq):
    """Causal layers measured faster with the hand-over than without (table at ds_handover_pays)."""
    assert native.ds_handover_pays(b, s, s, hq, 16 if hq == 16 else 4, True, UNITS)


def test_grids_that_do_not_fill_the_device_recompute():
    assert not native.ds_handover_pays(1, 255 * 512, 255 * 512, 1, 1, True, UNITS) and native.ds_handover_pays(1, 256 * 512, 256 * 512, 1, 1, True, UNITS)
    assert not native.ds_handover_pays(1, 8192, 8192, 32, 4, True, 0) and not native.ds_handover_pays(1, 8192, 8192, 32, 3, True, UNITS)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("pays,b,sq,skv,hq,hkv", [
    (False, 2, 1536, 1536, 44, 4), (False, 8, 512, 512, 33, 3), (False, 1, 12288, 12288, 11, 1), (False, 2, 2048, 2048, 36, 4), (False, 1, 8192, 4096, 44, 4),
    (True, 4, 1536, 1536, 44, 4), (True, 2, 1536, 1536, 48, 4), (True, 2, 2048, 2048, 33, 11), (True, 1, 4096, 4096, 40, 8), (True, 1, 12288, 12288, 12, 1),
])  # fmt: skip
def test_grids_of_unsplit_groups(pays, b, sq, skv, hq, hkv, causal):
    """Groups of an odd number of heads are not split: too few dK/dV workgroups to hand dS over, as measured."""
    assert native.ds_handover_pays(b, sq, skv, hq, hkv, causal, UNITS) == pays


@pytest.mark.parametrize("pays,b,s,hq,hkv", [
    ("no", 8, 64, 64, 4), ("no", 8, 128, 32, 4), ("no", 64, 64, 32, 4), ("no", 8, 256, 32, 4), ("yes", 8, 257, 32, 4), ("yes", 32, 320, 8, 8), ("yes", 8, 512, 32, 4),
    ("causal", 4, 513, 32, 4), ("causal", 8, 600, 32, 4), ("causal", 16, 639, 32, 4), ("yes", 8, 640, 32, 8), ("yes", 8, 720, 16, 16), ("yes", 2, 1100, 64, 4),
    ("yes", 1, 4095, 32, 4), ("yes", 1, 2100, 64, 4), ("yes", 1, 3600, 32, 4),
])  # fmt: skip
def test_rows_that_fill_their_workgroups(pays, b, s, hq, hkv):
    """512-row workgroups that are mostly empty do not fill the device, as measured."""
    assert [native.ds_handover_pays(b, s, s, hq, hkv, c, UNITS) for c in (True, False)] == {"no": [False] * 2, "yes": [True] * 2, "causal": [True, False]}[pays]


@pytest.mark.parametrize("causal,b,sq,skv,h,pays", [
    (True, 1, 4096, 4096, 16, True), (True, 4, 1024, 1024, 16, True), (True, 1, 4608, 4608, 16, True), (True, 1, 16384, 16384, 4, True),
    (True, 1, 3072, 3072, 16, True), (True, 1, 2048, 2048, 16, False), (True, 1, 12288, 12288, 4, True), (True, 1, 8192, 8192, 4, False), (True, 8, 512, 512, 16, False), (True, 16, 512, 512, 16, True), (True, 16, 256, 256, 16, False),
    (False, 1, 4096, 2048, 16, True), (False, 1, 2048, 4096, 16, True), (False, 1, 2048, 1024, 16, False), (False, 1, 1024, 2048, 16, False),
    (False, 1, 8192, 4096, 4, False), (False, 1, 4096, 8192, 4, False),
])  # fmt: skip
def test_calls_of_192_that_hand_over(causal, b, sq, skv, h, pays):
    """As measured (table at ds_handover_pays_192)."""
    assert native.ds_handover_pays_192(b, sq, skv, h, h, causal, UNITS) == pays and not native.ds_handover_pays_192(b, sq, skv, h, h, causal, 0)


@pytest.mark.parametrize("b,s,h,pays", [(1, 1024, 16, 0), (1, 2048, 16, 0), (1, 8192, 4, 0), (4, 512, 16, 0), (8, 256, 32, 0), (1, 3072, 16, 1), (1, 12032, 4, 1),
                                        (2, 1536, 16, 1), (1, 4096, 16, 1), (4, 1024, 16, 1), (1, 16384, 4, 1), (1, 6144, 16, 1)])  # fmt: skip
def test_shares_of_192_that_hand_over(b, s, h, pays):
    """As measured (table at share_of_192_pays)."""
    assert native.share_of_192_pays(b, s, h, UNITS) == bool(pays) and not native.share_of_192_pays(b, s, h, 0)


@pytest.mark.parametrize("layout", ["zigzag", "contiguous"])
@pytest.mark.parametrize("b,s,h", [(1, 2048, 16), (1, 2176, 16), (1, 2560, 16), (1, 4096, 16), (1, 4098, 16), (1, 8194, 16), (1, 1024, 16), (1, 8192, 4), (4, 512, 16), (2, 2050, 64)])
def test_share_of_192_is_looked_at_in_python_where_one_of_its_steps_hands_over(b, s, h, layout):
    """2048 and 2176 rows x 16 heads: whole chunks would, the half chunks of a zigzag share do not."""
    for cp in (1, 2, 4):
        for rank in range(cp):
            sizes = [(st.q_rows[1] - st.q_rows[0], st.kv_rows[1] - st.kv_rows[0], st.causal) for st in ring_schedule(rank, cp, s, layout)]
            want = any(native.ds_handover_pays_192(b, m, n, h, h, c, UNITS) for m, n, c in sizes)
            assert native.step_of_192_hands_over(b, s, h, h, rank, cp, layout == "zigzag", UNITS) == want, (cp, rank)
            if s in (2048, 2176):
                assert want == (layout == "contiguous" and rank > 0)


def test_bytes_of_a_share_that_hands_over():
    """All chunks, a query tile of one lying within its images: 128 rows and keys of a half, their own chunk under the mask last."""
    def need(sq, chunks, dqk=192):
        args = _C.AttnBwdArgs(B=2, Sq=sq, Hq=4, Hkv=4, Dqk=dqk, Dv=128)
        given = (_C.KeyChunk * len(chunks))(*[_C.KeyChunk(rows=rows, q_row0=row0) for rows, row0 in chunks])
        return _C.lib().pith_attn_bwd_chunks_ds_bytes(_C.byref(args), given, len(chunks))

    assert need(256, [(128, 0), (256, 128), (256, 0)]) == 2 * 4 * 16384 * (4 * 1 + 2 * 2 + 6)
    assert need(258, [(129, 0), (258, 0)]) == 2 * 4 * 16384 * (5 * 2 + 1 + 1 + 2 + 2 + 3)
    assert need(258, [(129, 0), (258, 129), (258, 0)]) == 0 and need(128, [(128, 0), (128, 0)]) == 0
    assert need(256, [(256, 0)]) == 0 and need(256, [(128, 0), (256, 0)], 128) == 0


@pytest.mark.parametrize("causal", [False, True])
def test_slabs_are_asked_for_by_the_rule_of_whole_calls(monkeypatch, causal):
    """A budget for one of two halves of the kv heads: the grid of a slab has to pass the same rule as that of the whole pair."""
    q = torch.empty(1, 10240, 32, 128, dtype=torch.bfloat16, device="meta")
    k = torch.empty(1, 10240, 4, 128, dtype=torch.bfloat16, device="meta")
    monkeypatch.setattr(H, "_device_compute_units", lambda device: UNITS)
    monkeypatch.setattr(H, "attn_bwd_ds_bytes", lambda *a: 4 << 20)
    monkeypatch.setattr(H, "_ds_budget_bytes", lambda device, enough: 2 << 20)
    real, asked = native.ds_handover_pays, []

    def rule(*call, refuse=None):
        asked.append(call)
        return real(*call) and call[3] != refuse

    monkeypatch.setattr(native, "ds_handover_pays", rule)
    assert H.ds_plan(q, k, k, causal) == (2, 2 << 20)
    assert asked == [(1, 10240, 10240, heads, heads // 8, causal, UNITS) for heads in (32, 16)]
    monkeypatch.setattr(native, "ds_handover_pays", lambda *a: rule(*a, refuse=16))
    assert H.ds_plan(q, k, k, causal) is None


def test_slabs_that_leave_units_idle_recompute(monkeypatch):
    """8192 x 4096 rows, 88/8 heads: 256 dK/dV workgroups as a whole, 128 in either of two slabs (measured 27 % slower)."""
    q = torch.empty(1, 8192, 88, 128, dtype=torch.bfloat16, device="meta")
    k = torch.empty(1, 4096, 8, 128, dtype=torch.bfloat16, device="meta")
    monkeypatch.setattr(H, "_device_compute_units", lambda device: UNITS)
    monkeypatch.setattr(H, "attn_bwd_ds_bytes", lambda *a: 8 << 20)
    monkeypatch.setattr(H, "_ds_budget_bytes", lambda device, enough: 8 << 20)
    assert H.ds_plan(q, k, k) == (8, 8 << 20)
    monkeypatch.setattr(H, "_ds_budget_bytes", lambda device, enough: 4 << 20)
    assert H.ds_plan(q, k, k) is None


@pytest.mark.parametrize("steps,b,s,hq,hkv,cp,rank,layout", [
    (1, 1, 8192, 32, 4, 4, 1, "zigzag"), (1, 1, 4096, 32, 4, 2, 1, "zigzag"), (1, 1, 8192, 16, 16, 4, 2, "contiguous"), (1, 1, 7168, 32, 4, 4, 2, "zigzag"),
    (1, 1, 7680, 32, 4, 4, 2, "contiguous"), (1, 2, 2048, 64, 4, 2, 1, "contiguous"), (1, 1, 4352, 32, 4, 2, 0, "zigzag"), (1, 1, 20480, 8, 2, 2, 0, "zigzag"),
    (1, 2, 1536, 64, 4, 4, 0, "contiguous"), (1, 1, 4608, 32, 4, 2, 0, "contiguous"),
    (1, 1, 2560, 64, 4, 2, 0, "zigzag"), (1, 1, 2304, 64, 4, 4, 0, "zigzag"), (1, 1, 5120, 32, 4, 4, 0, "zigzag"), (0, 1, 3072, 64, 4, 4, 0, "zigzag"),
    (0, 1, 9216, 32, 4, 4, 2, "zigzag"), (0, 1, 4608, 32, 4, 4, 2, "contiguous"), (0, 1, 5120, 64, 4, 4, 2, "zigzag"), (0, 1, 10240, 16, 4, 4, 2, "zigzag"),
    (0, 2, 1536, 64, 4, 4, 2, "zigzag"), (0, 16, 512, 32, 4, 4, 2, "zigzag"), (0, 4, 1100, 64, 4, 2, 1, "contiguous"), (0, 4, 3000, 32, 4, 4, 2, "zigzag"),
    (0, 1, 1792, 64, 4, 4, 0, "zigzag"), (0, 1, 1792, 64, 4, 4, 3, "zigzag"), (0, 1, 2048, 64, 4, 2, 0, "zigzag"), (0, 1, 1024, 8, 2, 4, 2, "zigzag"),
])  # fmt: skip
def test_shares_that_hand_over_go_out_step_by_step_where_that_is_faster(steps, b, s, hq, hkv, cp, rank, layout):
    """As measured (table at share_hands_over), with the steps that hand over by the rule of calls."""
    sizes = [(st.q_rows[1] - st.q_rows[0], st.kv_rows[1] - st.kv_rows[0], st.causal) for st in ring_schedule(rank, cp, s, layout)]
    sizes = [(m, n, c, hkv if native.ds_handover_pays(b, m, n, hq, hkv, c, UNITS) else 0) for m, n, c in sizes]
    assert native.share_hands_over(b, s, hq, hkv, sizes, UNITS) == bool(steps)


@pytest.mark.parametrize("steps,b,s,h,cp,rank,layout", [
    (1, 1, 8192, 16, 4, 2, "zigzag"), (1, 1, 10240, 16, 4, 2, "zigzag"), (1, 1, 9216, 16, 4, 2, "contiguous"), (1, 1, 12288, 16, 2, 0, "zigzag"),
    (1, 1, 7170, 16, 4, 1, "zigzag"), (1, 2, 4098, 32, 4, 3, "zigzag"), (1, 16, 2048, 16, 4, 1, "zigzag"), (1, 16, 2050, 16, 4, 1, "zigzag"),
    (1, 8, 3072, 16, 4, 2, "contiguous"), (1, 8, 2306, 16, 4, 2, "zigzag"), (1, 4, 4096, 16, 4, 3, "contiguous"), (1, 1, 16384, 8, 4, 2, "zigzag"),
    (0, 1, 4098, 16, 4, 2, "zigzag"), (0, 1, 3074, 16, 4, 2, "zigzag"), (0, 1, 3074, 16, 2, 0, "zigzag"), (0, 64, 1024, 16, 4, 2, "zigzag"), (0, 1, 2560, 32, 4, 2, "zigzag"),
    (0, 1, 8194, 16, 4, 2, "zigzag"), (0, 1, 9216, 16, 4, 2, "zigzag"), (0, 1, 5122, 16, 4, 1, "zigzag"),
])  # fmt: skip
def test_shares_of_192_that_go_out_step_by_step(steps, b, s, h, cp, rank, layout):
    """The same at 192 features (asked where the share as a whole does not hand over): step by step only where that measured faster."""
    sizes = [(st.q_rows[1] - st.q_rows[0], st.kv_rows[1] - st.kv_rows[0], st.causal) for st in ring_schedule(rank, cp, s, layout)]
    sizes = [(m, n, c, h if native.ds_handover_pays_192(b, m, n, h, h, c, UNITS) else 0) for m, n, c in sizes]
    assert native.share_hands_over(b, s, h, h, sizes, UNITS, 192) == bool(steps)


def test_share_of_one_step_hands_over_as_the_call_it_is():
    """Also where its rows are less than a full device's."""
    for s, pays in ((3200, True), (2816, False), (4096, True)):
        assert native.ds_handover_pays(1, s, s, 32, 4, True, UNITS) == pays
        assert native.share_hands_over(1, s, 32, 4, [(s, s, True, 4 if pays else 0)], UNITS) == pays


def test_share_of_slabs_counts_their_grids():
    """131072 tokens, 64/4 heads: a slab of one kv head at a time fills the device; a quarter of its heads would not."""
    sizes = lambda heads: [(16384, 8192, False, heads)] * 3 + [(8192, 16384, False, heads)] * 4 + [(16384, 16384, True, 0)]  # noqa: E731
    assert native.share_hands_over(1, 16384, 64, 4, sizes(1), UNITS) and native.share_hands_over(1, 16384, 64, 4, sizes(4), UNITS)
    small = [(16384, 8192, False, 1)] * 3
    assert not native.share_hands_over(1, 16384, 16, 4, small, UNITS) and not native.share_hands_over(1, 16384, 64, 4, [], UNITS)


@pytest.mark.gpu
def test_more_workgroups_than_one_launch_takes(gpu):
    """One row attends to itself: O = V, dV = dO, dQ = dK = 0. 8.5 M workgroups of either kernel."""
    b, h, d = 65535, 130, 64
    assert not _plan(b, 1, 1, h, h, 0, d).one_grid
    g = torch.Generator(device=gpu).manual_seed(1)
    q, k, v, dout = (torch.randn(b, 1, h, d, generator=g, device=gpu, dtype=torch.bfloat16) for _ in range(4))
    o, lse = torch.ops.pithtrain_amd.attn_fwd(q, k, v, d**-0.5, False)
    assert torch.equal(o, v)
    dq, dk, dv = torch.ops.pithtrain_amd.attn_bwd(q, k, v, o, lse, dout, d**-0.5, False)
    assert torch.equal(dv, dout)
    # dS is the difference of two fp32 sums of 64 products |x y| < 36 in two orders: below 64 * 2^-24 * 64 * 36 = 0.0088; times |k| < 6, scale 1/8
    assert dq.abs().max() < 0.0067 and dk.abs().max() < 0.0067


@pytest.mark.gpu
def test_share_of_64_features_in_two_launches(gpu):
    """Whole rounds of workgroups go out as two launches, those of one kv head as one: equal bit for bit."""
    s, hq, hkv, cp = 16384, 12, 4, 4
    assert not _share_plan(1, s, hq, hkv, cp, 0, "zigzag").one_grid and _share_plan(1, s, 3, 1, cp, 0, "zigzag").one_grid
    g = torch.Generator(device=gpu).manual_seed(1)
    mk = lambda h: torch.randn(1, s, h, 64, generator=g, device=gpu, dtype=torch.bfloat16)  # noqa: E731
    q, ks, vs, dout = mk(hq), [mk(hkv) for _ in range(cp)], [mk(hkv) for _ in range(cp)], mk(hq)
    out, lse = mk(hq), torch.randn(1, hq, s, generator=g, device=gpu) + 12.0
    whole = native.ring_backward(dout, q, out, lse, ks, vs, None, 0.125, 0, cp, True)
    for h in (0, 3):
        qh, kh = slice(3 * h, 3 * h + 3), slice(h, h + 1)
        dout_h, q_h, out_h, lse_h = dout[:, :, qh].contiguous(), q[:, :, qh].contiguous(), out[:, :, qh].contiguous(), lse[:, qh].contiguous()
        one = native.ring_backward(dout_h, q_h, out_h, lse_h, [k[:, :, kh].contiguous() for k in ks], [v[:, :, kh].contiguous() for v in vs], None, 0.125, 0, cp, True)
        assert torch.equal(whole[0][:, :, qh], one[0])
        for j in range(cp):
            assert torch.equal(whole[1][j][:, :, kh], one[1][j]) and torch.equal(whole[2][j][:, :, kh], one[2][j])


@pytest.mark.parametrize("causal,b,s,hq,hkv,d,split", [
    # wanted 512 workgroups under the mask and 256 without: half of what doubling leaves, on either side of the lines
    (1, 3, 768, 32, 4, 128, 4), (1, 2, 2304, 16, 4, 128, 2), (1, 1, 2304, 32, 4, 128, 4), (1, 1, 2305, 32, 4, 128, 8), (1, 3, 1200, 32, 4, 128, 4),
    (1, 3, 1500, 32, 4, 128, 4), (1, 1, 4096, 32, 4, 128, 4), (1, 1, 4097, 32, 4, 128, 4), (1, 1, 3900, 32, 4, 128, 4), (1, 9, 768, 32, 4, 128, 2),
    (1, 9, 769, 32, 4, 128, 2), (1, 24, 128, 32, 4, 128, 4), (0, 1, 1100, 32, 4, 128, 4), (0, 2, 1100, 64, 4, 128, 4), (0, 1, 2816, 32, 4, 128, 2),
    (0, 1, 2817, 32, 4, 128, 4), (1, 9, 1100, 32, 8, 64, 1), (1, 1, 5120, 32, 8, 64, 2), (1, 1, 5121, 32, 8, 64, 4), (0, 4, 1290, 32, 8, 64, 1), (1, 3, 768, 32, 4, 192, 8),
    # rows that do not hand dS over without a mask: up to 256, 513 to 639
    (0, 4, 520, 32, 4, 128, 2), (0, 4, 600, 64, 4, 128, 2), (0, 20, 160, 32, 4, 128, 1), (0, 33, 100, 32, 4, 128, 1), (0, 8, 640, 16, 4, 128, 2), (0, 10, 400, 32, 4, 128, 2),
    # handing over under the mask: rows x heads of a part up to 4096, 6144, 12288, 24576 at 1.125, 1.375, 1.5 workgroups per unit and more
    (1, 11, 768, 16, 4, 128, 1), (1, 13, 520, 32, 4, 128, 2), (1, 11, 768, 64, 4, 128, 2), (1, 9, 1024, 16, 4, 128, 1), (1, 9, 1025, 16, 4, 128, 1), (1, 12, 664, 64, 4, 128, 2),
    (1, 13, 768, 32, 4, 128, 1), (1, 13, 709, 64, 4, 128, 2), (1, 7, 1500, 16, 4, 128, 1), (1, 7, 1500, 32, 4, 128, 2), (1, 15, 768, 64, 4, 128, 1), (1, 5, 2304, 64, 4, 128, 2),
    (1, 8, 1368, 64, 4, 128, 2), (1, 11, 1152, 64, 4, 128, 1), (1, 7, 1800, 64, 4, 128, 2), (1, 3, 2048, 64, 4, 128, 4),
])  # fmt: skip
def test_head_split_is_halved_where_that_is_faster(causal, b, s, hq, hkv, d, split):
    """As measured (table at half_as_many)."""
    assert _plan(b, s, s, hq, hkv, causal, d).dkdv_split == split


@pytest.mark.parametrize("b,s,hq,hkv,cp,rank,layout,d,split", [
    # more than 512 workgroups of all chunks; dQ workgroups of 128 rows: 257 to 1024 in the one grid, 256, more
    (1, 1100, 32, 4, 4, 3, "contiguous", 128, 2), (2, 2400, 8, 2, 4, 3, "zigzag", 128, 2), (1, 1024, 32, 4, 4, 3, "contiguous", 128, 4), (1, 900, 32, 4, 8, 4, "zigzag", 128, 4),
    (1, 2300, 64, 4, 4, 2, "contiguous", 128, 4), (1, 2048, 64, 4, 4, 2, "contiguous", 128, 2), (1, 4352, 16, 4, 4, 2, "contiguous", 64, 4),
])  # fmt: skip
def test_head_split_of_shares(b, s, hq, hkv, cp, rank, layout, d, split):
    assert _share_plan(b, s, hq, hkv, cp, rank, layout, d).dkdv_split == split


@pytest.mark.parametrize("two_part", [False, True])
@pytest.mark.parametrize("b,s,hq,hkv,d", [(1, 3200, 32, 4, 128), (1, 3600, 32, 4, 128), (2, 1700, 32, 4, 128), (1, 4300, 32, 8, 64), (1, 8192, 32, 4, 128), (3, 1100, 32, 4, 128),
                                          (1, 256, 8, 2, 128), (1, 2304, 64, 4, 128), (1, 2305, 64, 4, 128), (2, 1024, 16, 16, 192), (3, 768, 32, 4, 192)])  # fmt: skip
def test_share_of_one_chunk_asks_for_the_workspace_of_the_call_it_is(b, s, hq, hkv, d, two_part):
    if two_part and (d != 192 or hq != hkv):
        return
    dv, pe = min(d, 128), 256 if two_part else None
    share = _C.AttnBwdArgs(B=b, Sq=s, Hq=hq, Hkv=hkv, Dqk=d, Dv=dv)
    chunk = (_C.KeyChunk * 1)(_C.KeyChunk(rows=s, q_row0=0, k_pe=pe))
    call = _C.AttnBwdArgs(B=b, Sq=s, Skv=s, Hq=hq, Hkv=hkv, Dqk=d, Dv=dv, causal=1, k_pe=pe)
    assert _C.lib().pith_attn_bwd_chunks_workspace_bytes(_C.byref(share), chunk, 1) == _C.lib().pith_attn_bwd_dkdv_workspace_bytes(_C.byref(call))


@pytest.mark.parametrize("causal,b,s,hq,hkv,pays", [
    # 0.687 / 0.69 of the device filled with rows, to 16384 of them; enough dK/dV workgroups under the mask
    (True, 1, 2816, 32, 4, False), (True, 1, 2827, 32, 4, True), (False, 1, 2827, 32, 4, True), (True, 3, 768, 32, 4, False), (True, 1, 1450, 64, 4, True),
    (True, 1, 16384, 7, 7, True), (True, 1, 16385, 7, 7, False), (True, 1, 7900, 12, 4, False), (False, 1, 7900, 12, 4, True),
])  # fmt: skip
def test_handover_of_grids_that_two_thirds_fill_the_device(causal, b, s, hq, hkv, pays):
    """As measured (table at ds_handover_pays)."""
    assert native.ds_handover_pays(b, s, s, hq, hkv, causal, UNITS) == pays


@pytest.mark.parametrize("one,s,hq,cp,rank,layout", [(1, 2048, 64, 2, 1, "contiguous"), (0, 2176, 64, 2, 1, "contiguous"), (1, 4096, 64, 4, 1, "zigzag"), (0, 4224, 64, 4, 1, "zigzag")])
def test_shares_of_128_features_in_one_grid(one, s, hq, cp, rank, layout):
    """Up to four dQ workgroups per compute unit, up to eight against more than two chunks' keys, as measured (table at one_grid)."""
    assert _share_plan(1, s, hq, 4, cp, rank, layout, 128).one_grid == one
