"""dK/dV of 128 features with 256 key rows per workgroup against the 128-key kernel: both add up the rows in the same steps of 16,
so for the same head split the results are equal bit for bit. The large call takes the one, each of its batch elements or kv
heads alone, whose grid is too small for it, the other (asked of the plan each time). Sizes: keys and rows at, before and behind the edges of blocks (32, 64,
128, 256), two query walks, every output type and the dS images (through dQ)."""

import re

import pytest
import torch

from pithtrain_amd import _C
from pithtrain_amd.operators.mla.hip import attn_bwd_dkdv_into, attn_bwd_dq_into, attn_bwd_ds_bytes

gpu_only = pytest.mark.gpu


def _key_rows(q, k, causal):
    """Key rows per workgroup that dK/dV of such a call takes."""
    args, plan = _C.AttnBwdArgs(B=q.shape[0], Sq=q.shape[1], Skv=k.shape[1], Hq=q.shape[2], Hkv=k.shape[2], Dqk=128, Dv=128, causal=causal), _C.AttnBwdPlan()
    _C.check(_C.lib().pith_attn_bwd_plan(_C.byref(args), _C.byref(plan)))
    return plan.dkdv_rows


def _grads(q, k, v, dout, lse, delta, causal, handover, dtype, old, tail):
    b, sq = q.shape[:2]
    skv = k.shape[1]
    dk, dv = (torch.full((b, skv + tail, *t.shape[2:]), 7.0, dtype=dtype, device=q.device) for t in (k, v))
    if old is not None:
        dk[:, :skv], dv[:, :skv] = old, old
    ds = None
    if handover:  # poisoned: whatever dQ reads must have been written
        ds = torch.full((attn_bwd_ds_bytes(q, k, v, causal),), 0x7F, dtype=torch.uint8, device=q.device)
    attn_bwd_dkdv_into(q, k, v, dout, lse, delta, dk[:, :skv], dv[:, :skv], 0.1, causal, accumulate=old is not None, ds=ds, zero_tail=tail)
    dq = torch.empty_like(q)
    if handover:
        attn_bwd_dq_into(q, k, v, dout, lse, delta, dq, 0.1, causal, ds=ds)
    else:
        dq.zero_()
    return dk, dv, dq


@gpu_only
@pytest.mark.parametrize("dtype,accumulate,tail", [(torch.bfloat16, False, 33), (torch.float32, True, 0), (torch.bfloat16, True, 0)])
@pytest.mark.parametrize("handover", [True, False])
@pytest.mark.parametrize(
    "B,Sq,Skv,H,causal",
    [
        (8, 512, 257, 16, False), (16, 545, 385, 16, False), (16, 1023, 511, 8, False), (32, 600, 256, 16, False), (8, 577, 300, 16, False),
        (16, 1025, 1025, 8, True), (16, 1120, 1120, 8, True), (8, 1024, 1024, 16, True), (16, 1249, 1249, 8, True), (8, 1599, 1599, 16, True),
    ],
)  # fmt: skip
def test_equal_to_the_128_key_kernel(gpu, B, Sq, Skv, H, causal, handover, dtype, accumulate, tail):
    g = torch.Generator(device=gpu).manual_seed(Sq + Skv)
    t = lambda *s: torch.randn(*s, generator=g, device=gpu)  # noqa: E731
    q, k, v, dout = (t(B, s, H, 128).to(torch.bfloat16) for s in (Sq, Skv, Skv, Sq))
    lse, delta = t(B, H, Sq) + 8.0, t(B, H, Sq)
    old = t(B, Skv, H, 128).to(dtype) if accumulate else None
    assert _key_rows(q, k, causal) == 256 and _key_rows(q[:1], k[:1], causal) == 128
    got = _grads(q, k, v, dout, lse, delta, causal, handover, dtype, old, tail)
    for b in range(0, B, 5):
        one = [x[b : b + 1] for x in (q, k, v, dout, lse, delta)]
        want = _grads(*one, causal, handover, dtype, None if old is None else old[b : b + 1], tail)
        for name, x, y in zip(("dk", "dv", "dq"), got, want):
            assert torch.equal(x[b : b + 1], y), f"{name} of batch element {b}"
        if tail:
            assert not got[0][b, Skv:].any() and not got[1][b, Skv:].any()


def _heads(gpu, Sq, Skv, Hq, Hkv, causal, handover):
    """A grouped call against its first and last kv head, query head by query head, in fp32 (sums of sums in another order)."""
    g = torch.Generator(device=gpu).manual_seed(5)
    t = lambda *s: torch.randn(*s, generator=g, device=gpu)  # noqa: E731
    q, dout = (t(1, Sq, Hq, 128).to(torch.bfloat16) for _ in range(2))
    k, v = (t(1, Skv, Hkv, 128).to(torch.bfloat16) for _ in range(2))
    lse, delta = t(1, Hq, Sq) + 10.0, t(1, Hq, Sq)
    assert _key_rows(q, k, causal) == 256 and _key_rows(q[:, :, :1], k[:, :, :1], causal) == 128
    dk, dv, dq = _grads(q, k, v, dout, lse, delta, causal, handover, torch.float32, None, 0)
    group = Hq // Hkv
    for h in (0, Hkv - 1):
        want = [0.0, 0.0]
        for j in range(h * group, (h + 1) * group):
            part = _grads(q[:, :, j : j + 1].contiguous(), k[:, :, h : h + 1].contiguous(), v[:, :, h : h + 1].contiguous(),
                          dout[:, :, j : j + 1].contiguous(), lse[:, j : j + 1].contiguous(), delta[:, j : j + 1].contiguous(),
                          causal, handover, torch.float32, None, 0)  # fmt: skip
            want = [w + x.double() for w, x in zip(want, part)]
            if handover:
                assert torch.equal(dq[:, :, j : j + 1], part[2])  # dS has the same bits from either kernel
        for x, w in zip((dk, dv), want):
            # fp32 accumulation of up to group * Sq terms in two orders: 2^-24 a step, a random walk of them
            bound = 2.0**-24 * (group * Sq) ** 0.5 * 4
            assert (x[:, :, h : h + 1].double() - w).norm() <= bound * w.norm()


@gpu_only
@pytest.mark.parametrize("Sq,Skv,Hq,Hkv,causal", [(4096, 520, 64, 16, False), (4100, 4100, 64, 4, True), (16400, 16400, 24, 8, True)])
def test_head_parts_and_descending_walk(gpu, Sq, Skv, Hq, Hkv, causal):
    """Grouped heads: parts of a group in several workgroups. The last one walks the query tiles from the end
    (its Q and dO outgrow the last-level cache)."""
    _heads(gpu, Sq, Skv, Hq, Hkv, causal, False)


@gpu_only
def test_descending_walk_hands_ds_over(gpu):
    assert 2 * 16400 * 24 * 128 * 2 > 192 << 20  # bytes of Q and dO from which on the walk descends
    _heads(gpu, 16400, 16400, 24, 8, True, True)


def test_waits_for_its_tile_loads_only(tmp_path):
    """An interval ends with `s_waitcnt vmcnt(4)` where the wave has just stored four dS fragments: right only if they are its last
    vector-memory operations, so no register may be spilled."""
    import subprocess

    from pithtrain_amd import build as B

    out = tmp_path / "wide.s"
    subprocess.run([B._hipcc(), *B.HIPCC_FLAGS, "-I", B.INCLUDE_DIR, "-I", B.SRC_DIR, "--cuda-device-only", "-S",
                    B.SRC_DIR + "/attn_bwd_dkdv_wide.hip", "-o", str(out)], check=True, capture_output=True)  # fmt: skip
    lines = out.read_text().splitlines()
    assert not [l for l in lines if re.match(r"\s+scratch_", l)], "registers are spilled"
    # (the epilogue waits, too, far behind the last product)
    waits = [i for i, l in enumerate(lines) if re.search(r"s_waitcnt vmcnt\(4\)\s*$", l) and any("v_mfma" in x for x in lines[i - 40 : i])]
    assert len(waits) == 6, "one steady-state wait per instance"
    for w in waits:
        ops = [l.split()[0] for l in lines[w - 400 : w] if re.match(r"\s+(global_|buffer_|flat_)", l)]
        assert ops[-4:] == ["global_store_dwordx4"] * 4 and ops[-5].startswith("global_load_lds"), ops[-6:]
