"""The operators' native host path on a machine without a GPU."""

import sys
import threading

import pytest
import torch

from pithtrain_amd import _C
from pithtrain_amd._ext import native
from pithtrain_amd.operators.mla_assemble import mla_assemble_qkv
from pithtrain_amd.operators.norm_rope import norm_rope, qk_norm_rope
from pithtrain_amd.operators.ring_attention.local import ring_schedule


def _meta(*shape):
    return torch.empty(*shape, dtype=torch.bfloat16, device="meta")


TABLE_CALLS = {
    "norm_rope": (lambda c, s: norm_rope(_meta(1, 4, 2, 128), _meta(128), c, s, 1e-6), 128),
    "norm_rope_no_weight": (lambda c, s: norm_rope(_meta(1, 4, 2, 128), None, c, s, 1e-6), 128),
    "qk_norm_rope": (lambda c, s: qk_norm_rope(_meta(1, 4, 2, 128), _meta(1, 4, 1, 128), _meta(128), _meta(128), c, s, 1e-6), 128),
    "mla_assemble": (lambda c, s: mla_assemble_qkv(_meta(1, 4, 2, 192), _meta(1, 4, 2, 256), _meta(1, 4, 1, 64), c, s), 64),
}


@pytest.mark.parametrize("which", [0, 1])
@pytest.mark.parametrize("name", TABLE_CALLS)
def test_rotary_tables_that_require_grad(name, which):
    """The result requires grad when a rotary table does, and backward() runs without giving the table a gradient."""
    call, dim = TABLE_CALLS[name]
    tables = [_meta(4, dim), _meta(4, dim)]
    tables[which].requires_grad_()
    out = call(*tables)
    outs = [out] if torch.is_tensor(out) else [o for o in out if o.grad_fn is not None]
    assert outs and all(o.requires_grad for o in outs)
    torch.autograd.backward(outs, [torch.empty_like(o) for o in outs])
    assert tables[which].grad is None


def test_failed_launch_is_not_tried_again():
    """What the library rejects goes to the Python body; a failed launch, whose call may have written something, raises."""
    assert native.accepted(_C.PITH_OK) and not native.accepted(_C.PITH_ERR_BAD_SHAPE)
    with pytest.raises(_C.PithError) as e:
        native.accepted(_C.PITH_ERR_LAUNCH)
    assert e.value.code == _C.PITH_ERR_LAUNCH


def _declined_calls():
    """One call of every bound function that may launch kernels, on CPU tensors: declined without touching a device."""
    q, d = torch.empty(1, 2, 2, 128, dtype=torch.bfloat16), torch.empty(1, 2, 2)
    f = torch.empty(1, 2, 2, 128)
    n = native
    return {
        "attn_fwd_into": lambda: n.attn_fwd_into(q, q, q, q, d, 0.1, True, None, None, None, None, None),
        "attn_bwd_delta_into": lambda: n.attn_bwd_delta_into(q, q, d),
        "attn_bwd_dkdv_into": lambda: n.attn_bwd_dkdv_into(q, q, q, q, d, d, q, q, 0.1, True, False, None, None, None, 0),
        "attn_bwd_dq_into": lambda: n.attn_bwd_dq_into(q, q, q, q, d, d, q, 0.1, True, False, None, None, None, None),
        "attn_bwd_pair_into": lambda: n.attn_bwd_pair_into(q, q, q, q, d, d, q, q, q, 0.1, True, False, False, None, None, None, 0, None, None),
        "ring_forward": lambda: n.ring_forward(q, [q, q], [q, q], None, 0.1, 0, 2, True),
        "ring_backward": lambda: n.ring_backward(q, q, q, d, [q, q], [q, q], None, 0.1, 0, 2, True),
        "combine_into": lambda: n.combine_into(q, d, q, d, f, d, 0),
        "combine_new": lambda: n.combine_new(q, d, q, d, 0),
        "cast_f32_bf16_into": lambda: n.cast_f32_bf16_into(f, q),
    }


@pytest.mark.parametrize("name", _declined_calls())
def test_bound_functions_release_the_interpreter_lock(name):
    """A launch can block on a full queue; other Python threads must be able to run meanwhile. The interpreter is told not to
    take the lock away by itself, so the other thread gets it only from a call that gives it up."""
    call = _declined_calls()[name]
    go, ran = threading.Event(), threading.Event()
    other = threading.Thread(target=lambda: (go.wait(), ran.set()), daemon=True)
    other.start()
    before = sys.getswitchinterval()
    try:
        sys.setswitchinterval(1000.0)
        go.set()
        for _ in range(200000):
            assert not call()
            if ran.is_set():
                break
        else:
            raise AssertionError(f"{name} keeps the interpreter lock")
    finally:
        sys.setswitchinterval(before)
        other.join()


@pytest.mark.parametrize("in_one,dqk,rows,heads,cp,rank,layout", [
    (True, 128, 8192, 32, 4, 1, "zigzag"), (True, 192, 4096, 16, 4, 1, "zigzag"), (True, 192, 1021, 16, 4, 2, "contiguous"),
    (True, 128, 8192, 4, 4, 0, "zigzag"), (True, 128, 3072, 16, 4, 3, "contiguous"), (True, 64, 16384, 4, 4, 1, "contiguous"),
    (True, 192, 8192, 2, 2, 1, "contiguous"), (False, 128, 8192, 8, 2, 1, "zigzag"), (False, 128, 6144, 8, 4, 1, "contiguous"),
    (False, 128, 4096, 16, 2, 1, "contiguous"), (False, 192, 16384, 4, 8, 3, "zigzag"), (False, 192, 6144, 4, 4, 3, "contiguous"),
    (False, 192, 12288, 4, 4, 0, "zigzag"), (True, 128, 8192, 8, 4, 0, "contiguous"), (True, 192, 8192, 8, 8, 3, "zigzag"),
    (False, 128, 6144, 8, 2, 0, "zigzag"), (True, 128, 6144, 8, 4, 0, "zigzag")])  # fmt: skip
def test_share_forward_by_size(in_one, dqk, rows, heads, cp, rank, layout):
    """One launch over all chunks, or one per ring step: whichever measured faster (256 compute units)."""
    steps = ring_schedule(rank, cp, rows, layout)
    keys = sum(st.kv_rows[1] - st.kv_rows[0] for st in steps)
    seen = sum((st.q_rows[1] - st.q_rows[0]) * (st.kv_rows[1] - st.kv_rows[0]) // (2 if st.causal else 1) for st in steps)
    assert native.share_forward_in_one(dqk, rows, heads, len(steps), 100 * seen // (keys * rows), 256) == in_one


@pytest.mark.parametrize("in_one,dqk,rows,heads,cp,rank,layout", [
    (False, 128, 8192, 8, 4, 0, "zigzag"), (False, 128, 8192, 8, 8, 4, "contiguous"), (False, 128, 16384, 8, 2, 0, "zigzag"),
    (True, 128, 8192, 8, 4, 1, "zigzag"), (True, 128, 12288, 8, 4, 0, "zigzag"), (True, 128, 4096, 16, 4, 0, "zigzag"),
    (True, 128, 9216, 8, 8, 4, "contiguous"), (True, 192, 16384, 4, 4, 0, "zigzag"), (True, 64, 8192, 16, 4, 0, "zigzag"),
    (True, 128, 8192, 8, 4, 0, "contiguous"), (False, 128, 8192, 32, 4, 1, "zigzag"), (True, 128, 6144, 32, 4, 3, "zigzag")])  # fmt: skip
def test_share_backward_by_size(in_one, dqk, rows, heads, cp, rank, layout):
    steps = ring_schedule(rank, cp, rows, layout)
    keys = sum(st.kv_rows[1] - st.kv_rows[0] for st in steps)
    assert native.share_backward_in_one(dqk, rows, heads, len(steps), keys, 256) == in_one
